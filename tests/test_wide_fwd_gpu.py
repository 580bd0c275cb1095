"""Forward at H = 256 (bf16) at the edges of tiles and passes, against the oracle: up to 16,384 edges the kernel that shares
a tile over eight waves, beyond them the edge-parallel one."""
import numpy as np
import pytest

from tests.cases import Case, random_csr
from tests.test_f32_split_gpu import _degrees
from tests.test_fused_gpu import check_case, run_fused

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eq", [True, False])
@pytest.mark.parametrize("kind", ["one", "15", "17", "32", "33", "ones", "halves", "long"])
def test_tile_edges(kind, eq):
    """Tiles of 1 to 32 ranks, rows over tiles, a pass with fewer tiles than the block's waves."""
    degs = _degrees(kind) + [0] * 5   # sources besides the row itself
    rowptr, col = random_csr(len(degs), degs, seed=len(degs))
    check_case(Case(rowptr, col, 256, 8, 256, 256, 256, seed=51, eq=eq, mean_agg=eq), "bf16")


@pytest.mark.parametrize("eq,fe", [(True, 0), (True, 24), (True, 32), (True, 56), (False, 8), (False, 32), (False, 40), (False, 64)])
def test_edge_slots(eq, fe):
    """One and two 32-slot slices of edge inputs, permuted edge ids."""
    degs = _degrees("halves")
    rowptr, col = random_csr(len(degs), degs, seed=3)
    perm = np.random.Generator(np.random.PCG64(3)).permutation(len(col))
    check_case(Case(rowptr, col, 64, fe, 256, 256, 256, seed=52, eq=eq, edge_ids=perm), "bf16")


@pytest.mark.parametrize("eq,fe", [(True, 0), (True, 32), (True, 56), (False, 8), (False, 64)])
@pytest.mark.parametrize("kind", ["none", "one", "15", "17", "33", "ones", "halves", "long"])
def test_edge_parallel_tiles(kind, eq, fe):
    """The same tails behind 16,384 edges in rows of 32 (whole tiles, 512 of them: without a tail the tile-sharing kernel's
    last graph), one and two 32-slot slices of edge inputs, permuted edge ids."""
    degs = [32] * 512 + ([] if kind == "none" else _degrees(kind)) + [0] * 5
    rowptr, col = random_csr(len(degs), degs, seed=len(degs))
    perm = np.random.Generator(np.random.PCG64(4)).permutation(len(col))
    check_case(Case(rowptr, col, 32, fe, 256, 256, 256, seed=55, eq=eq, mean_agg=eq, edge_ids=perm), "bf16", backward=False)


def test_many_passes():
    """More tiles than one pass of the grid (512 blocks of four tiles)."""
    degs = np.full(2100, 33)
    rowptr, col = random_csr(len(degs), degs, seed=6)
    check_case(Case(rowptr, col, 16, 16, 256, 256, 256, seed=53, bias=False), "bf16", backward=False)


@pytest.mark.parametrize("eq", [True, False])
def test_infinite_feature(eq):
    """One infinite entry of b1: an infinite message where its weight is positive, SiLU(-inf) = NaN where it is negative,
    as in the oracle (the edge-parallel kernel; rows of 32 edges, so that no row sum multiplies another row's infinity
    by 0)."""
    rowptr, col = random_csr(520, np.full(520, 32), seed=8)
    case = Case(rowptr, col, 32, 8, 256, 256, 256, seed=54, eq=eq)
    case.p["b1"][37] = np.inf
    got = run_fused(case, "bf16", backward=False)["out_msg"]
    up = case.p["w2_msg"][37] > 0
    assert np.isposinf(got[:, up]).all() and np.isnan(got[:, ~up]).all()
