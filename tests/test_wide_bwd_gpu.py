"""Edge-parallel backward at H = 256 (bf16) at the edges of its 16-edge pieces and passes, against the oracle."""
import numpy as np
import pytest

from tests.cases import Case, random_csr
from tests.test_fused_gpu import check_case, run_fused

pytestmark = pytest.mark.gpu


# its range begins at 16,385 edges: 128 whole 128-edge pieces and 1, 16, 17 or 128 edges; 16,384 takes the other kernel
@pytest.mark.parametrize("eq,fe", [(True, 0), (True, 32), (True, 56), (False, 8), (False, 64)])
@pytest.mark.parametrize("E", [16384, 16385, 16400, 16401, 16512])
def test_pass_edges(E, eq, fe):
    """Lanes and whole waves past the last edge, one and two 32-slot slices of edge inputs, permuted edge ids."""
    degs = [40] * (E // 40) + [E % 40, 0]
    rowptr, col = random_csr(len(degs), degs, seed=E)
    perm = np.random.Generator(np.random.PCG64(E)).permutation(E)
    check_case(Case(rowptr, col, 32, fe, 256, 256, 256, seed=61, eq=eq, mean_agg=eq, edge_ids=perm), "bf16")


# 32,769 to 40,960 edges take the other kernel (a second pass for few edges); from there on two passes
@pytest.mark.parametrize("eq", [True, False])
@pytest.mark.parametrize("E", [32768, 32769, 40961])
def test_many_passes(E, eq):
    """More 128-edge pieces than blocks (256): the sums of dw2_mov and dw_d over a block's passes."""
    degs = [33] * (E // 33) + [E % 33]
    rowptr, col = random_csr(len(degs), degs, seed=7)
    check_case(Case(rowptr, col, 16, 16, 256, 256, 256, seed=62, eq=eq), "bf16")


@pytest.mark.parametrize("eq,fe", [(True, 32), (True, 56), (False, 8)])
def test_same_bits_on_both_sides_of_the_rule(eq, fe):
    """A graph of 8,192 edges (the kernels that share a tile) alone and as the first part of one of 17,600 (the
    edge-parallel kernels): its messages and the gradient of its nodes' features are the same to the bit, as every stage
    sums in the same order."""
    part, rest = [32] * 256, [40] * 235 + [8, 0]
    rowptr, col = random_csr(256, part, seed=9)
    more, col2 = random_csr(len(rest), rest, seed=10)
    whole = Case(np.concatenate([rowptr, rowptr[-1] + more[1:]]), np.concatenate([col, 256 + col2]), 64, fe, 256, 256, 256,
                 seed=63, eq=eq, mean_agg=eq)
    alone = Case(rowptr, col, 64, fe, 256, 256, 256, seed=63, eq=eq, mean_agg=eq)
    alone.p = whole.p
    n = alone.N
    alone.h, alone.gm, alone.ef = whole.h[:n], whole.gm[:n], whole.ef[:alone.E]
    if eq:
        alone.coord, alone.gx = whole.coord[:n], whole.gx[:n]
    a, b = run_fused(alone, "bf16"), run_fused(whole, "bf16")
    assert np.array_equal(a["out_msg"], b["out_msg"][:n])
    assert np.array_equal(a["grads"]["h"], b["grads"]["h"][:n])
