"""Edge-parallel backward at H = 256 (bf16) at the edges of its 16-edge pieces and passes, against the oracle."""
import numpy as np
import pytest

from tests.cases import Case, random_csr
from tests.test_fused_gpu import check_case

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
