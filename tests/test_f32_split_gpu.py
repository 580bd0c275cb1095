"""fp32 kernels on split bf16 operands (H = 128) at the edges of their tiles, against the float64 oracle.

Bound: an fp32 product summed over K = 128 terms in any order differs from the exact sum by at most
128 * 2^-24 = 7.6e-6 of the sum of the terms' magnitudes; normwise (largest difference over largest
value) 1e-5 therefore holds for any correct fp32 implementation of the layer, as in test_fused_gpu.
"""
import numpy as np
import pytest
import torch

from oracle import egnn_oracle as orc
from tests.cases import Case, random_csr
from tests.test_fused_gpu import check_case, run_fused

pytestmark = pytest.mark.gpu


def _degrees(kind):
    """Rows that end, begin and go on at every 16-edge half and 32-edge tile boundary."""
    if kind == "one":
        return [1]
    if kind == "15":
        return [15, 0]
    if kind == "16":
        return [16]
    if kind == "17":          # a row over the half boundary, last tile half empty
        return [3, 0, 14]
    if kind == "32":
        return [16, 16]
    if kind == "33":
        return [10, 20, 3]
    if kind == "ones":        # 32 ranks per tile
        return [1] * 70
    if kind == "halves":      # ends exactly at halves and tiles, and just beside them
        return [15, 2, 15, 16, 16, 31, 1, 32, 17, 0, 47, 33, 48, 5]
    return [200, 0, 3, 100, 31, 65, 7]


@pytest.mark.parametrize("eq", [True, False])
@pytest.mark.parametrize("kind", ["one", "15", "16", "17", "32", "33", "ones", "halves", "long"])
def test_tile_edges(kind, eq):
    degs = _degrees(kind) + [0] * 5   # sources besides the row itself (a self edge has no coordinate gradient)
    rowptr, col = random_csr(len(degs), degs, seed=len(degs))
    check_case(Case(rowptr, col, 128, 0, 128, 128, 128, seed=31, eq=eq, mean_agg=eq), "fp32")


@pytest.mark.parametrize("eq,fe", [(True, 8), (True, 24), (True, 32), (True, 40), (False, 8), (False, 32), (False, 64)])
def test_edge_feature_slots(eq, fe):
    """Edge-feature widths around the 32-slot slices (the r^2 slot in the last slice, or alone in one)."""
    degs = _degrees("halves")
    rowptr, col = random_csr(len(degs), degs, seed=3)
    perm = np.random.Generator(np.random.PCG64(3)).permutation(len(col))
    check_case(Case(rowptr, col, 32, fe, 128, 128, 128, seed=32, eq=eq, edge_ids=perm), "fp32")


@pytest.mark.parametrize("eq", [True, False])
def test_not_finite_rows_stay_apart(eq):
    """A node with infinite and NaN features makes its own and its neighbours' rows not finite, no others."""
    degs = np.array([4, 9, 33, 0, 16, 20, 2, 40])
    rowptr, col = random_csr(len(degs), degs, seed=4)
    case = Case(rowptr, col, 128, 0, 128, 128, 128, seed=33, eq=eq)
    ref, _ = case.forward_ref(False)
    case.h[5, 3], case.h[5, 7] = np.inf, np.nan
    rows = np.repeat(np.arange(len(degs)), degs)
    hit = np.unique(np.concatenate([rows[col == 5], rows[rows == 5]]))
    out = run_fused(case, "fp32", backward=False)["out_msg"]
    clean = np.setdiff1d(np.arange(len(degs)), hit)
    assert len(clean) and not np.isfinite(out[hit]).any()
    assert orc.normwise_rel_err(out[clean], ref[clean]) <= 1e-5


def test_extreme_magnitudes():
    """Features from 1e-30 to the largest finite value: the parts of a split value never overflow."""
    degs = np.array([5, 30, 3, 8])
    rowptr, col = random_csr(len(degs), degs, seed=5)
    case = Case(rowptr, col, 16, 0, 128, 128, 128, seed=34, eq=False)
    case.h[0] *= 1e-30
    case.h[1] *= 1e15
    for k in ("w1_msg", "w2_msg"):
        case.p[k] = np.abs(case.p[k])
    case.h = np.abs(case.h).astype(np.float32)
    check_case(case, "fp32", backward=False)
    case.h[2] = np.finfo(np.float32).max
    case.p["w1_msg"] = (case.p["w1_msg"] * 2.0 ** -9).astype(np.float32)
    check_case(case, "fp32", backward=False)
    torch.cuda.synchronize()


def _gemm_case(N, K1, K2, Hn, Fo, res, seed):
    """egnn_node_fwd / bwd in fp32 against float64: pre = [x1 | x2] W1^T + b1, out = SiLU(pre) W2^T + b2 (+ x1)."""
    from pymolecular_amd.node_update import node_update
    g = torch.Generator().manual_seed(seed)
    mk = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    x1, x2 = mk(N, K1), mk(N, K2) if K2 else None
    p = [mk(Hn, K1 + K2) / (K1 + K2) ** 0.5, mk(Hn) * 0.1, mk(Fo, Hn) / Hn ** 0.5, mk(Fo) * 0.1]
    go = mk(N, Fo)

    def run(conv, f):
        a = conv(x1).requires_grad_()
        b = None if x2 is None else conv(x2).requires_grad_()
        lin = [torch.nn.Linear(K1 + K2, Hn), torch.nn.Linear(Hn, Fo)]
        for m, w, v in zip(lin, p[::2], p[1::2]):
            m.weight, m.bias = torch.nn.Parameter(conv(w)), torch.nn.Parameter(conv(v))
        out = f(a, b, *lin)
        wrt = [t for t in (a, b) if t is not None] + [t for m in lin for t in m.parameters()]
        return [out.detach()] + list(torch.autograd.grad(out, wrt, conv(go)))

    def ref(a, b, lin1, lin2):
        y = lin2(torch.nn.functional.silu(lin1(a if b is None else torch.cat([a, b], 1))))
        return y + a if res else y
    got = run(lambda t: t.detach().cuda(), lambda a, b, lin1, lin2: node_update(a, b, lin1, lin2, residual=res))
    want = run(lambda t: t.detach().double(), ref)
    for k, (u, v) in enumerate(zip(got, want)):
        err = ((u.double().cpu() - v).norm() / v.norm().clamp(min=1e-30)).item()
        # sums of up to N products: 2-norm error of a few 2^-24 times sqrt(log-ish growth); 2e-6 is 30 roundings
        assert err <= 2e-6, (k, err)


@pytest.mark.parametrize("N,K1,K2,Hn,Fo,res", [
    (1, 128, 128, 128, 128, True),       # one row
    (31, 128, 0, 128, 128, True),        # below a 32-row tile
    (33, 8, 8, 24, 8, True),             # K of 16 and 24: a slice's tail, columns past N
    (65, 128, 128, 128, 128, False),
    (257, 40, 24, 72, 48, False),        # no multiple of a tile anywhere
    (8200, 128, 128, 128, 128, True),    # 256 tiles and a remainder; 64-row tiles in the weight gradients
    (4099, 136, 120, 256, 136, True),    # concatenation inside a 32-deep slice
])
def test_f32_node_products(N, K1, K2, Hn, Fo, res):
    _gemm_case(N, K1, K2, Hn, Fo, res, N)


@pytest.mark.parametrize("eq", [True, False])
@pytest.mark.parametrize("kind", ["one", "15", "16", "17", "32", "33", "ones", "halves", "long"])
def test_small_width_tile_edges(kind, eq):
    """H = 64, O = M = 32: whole 32-edge tiles per wave in the forward, 16 edges in the backward."""
    degs = _degrees(kind) + [0] * 5
    rowptr, col = random_csr(len(degs), degs, seed=len(degs))
    check_case(Case(rowptr, col, 32, 16, 64, 32, 32, seed=41, eq=eq, mean_agg=eq), "fp32")


@pytest.mark.parametrize("eq,fe", [(True, 0), (True, 8), (True, 24), (True, 32), (False, 0), (False, 8), (False, 24),
                                   (False, 32), (False, 40)])
@pytest.mark.parametrize("linear", [False, True])
def test_small_width_edge_slots(eq, fe, linear):
    """Edge-input slots up to the 32 the small kernels hold and beyond (the general kernels), both weight layouts."""
    degs = _degrees("halves")
    rowptr, col = random_csr(len(degs), degs, seed=3)
    perm = np.random.Generator(np.random.PCG64(3)).permutation(len(col))
    case = Case(rowptr, col, 48, fe, 64, 32, 32, seed=42, eq=eq, edge_ids=perm)
    res, gref = run_fused(case, "fp32", linear=linear), case.backward_ref(False)
    ref = case.forward_ref(False)
    errs = {"msg": orc.normwise_rel_err(res["out_msg"], ref[0])}
    for k, v in gref.items():
        if v is not None and res["grads"].get(k) is not None:
            errs[k] = orc.normwise_rel_err(res["grads"][k].reshape(v.shape), v)
    assert all(e <= 1e-5 for e in errs.values()), errs


def test_small_width_many_tiles_per_wave():
    """More edges than one pass of the grid (512 blocks of 64 edges), so every wave accumulates several times."""
    degs = np.full(3000, 29)
    rowptr, col = random_csr(len(degs), degs, seed=6)
    check_case(Case(rowptr, col, 32, 16, 64, 32, 32, seed=43, bias=False), "fp32")


def test_stack_errors_do_not_add_up():
    """Gradients of the coordinate MLPs of the first two of four layers (512 molecules, 12 seeds) against float64: sums of
    190,000 terms of either sign, in which errors that point the same way for every edge add up.  Bound: their geometric
    mean with the same layer on the fp32 matrix instruction, 6.0e-7 for these inputs (plain float32 torch: 1.9e-6; the
    split products without the alternating signs: 8.8e-7)."""
    from oracle import torch_ref
    from pymolecular_amd import graphs
    from pymolecular_amd.models.EGNN import EGNN
    g = graphs.molecule_batch(512, seed=1001, feat_seed=3)
    edges = [torch.from_numpy(g.rows().astype(np.int64)).cuda(), torch.from_numpy(g.col.astype(np.int64)).cuda()]
    h = torch.from_numpy(g.node_feat).float().cuda()
    logs = []
    for seed in range(12):
        torch.manual_seed(seed)
        exact = torch_ref.EGNNRef(5, 128, 128, 0, n_layers=4).cuda()
        ours = EGNN(5, 128, 128, 0, n_layers=4).cuda()
        ours.load_state_dict({k.replace("layers.", "gcl_"): v for k, v in exact.state_dict().items()})
        x, gx, gh = (1.5 * torch.randn(g.N, 3)).cuda(), torch.randn(g.N, 3).cuda(), torch.randn(g.N, 128).cuda()

        def grads(m, layers, dt):
            out = m(h.to(dt), x.to(dt), edges, None)
            return torch.autograd.grad(out, [p for q in layers for p in q.coord_mlp.parameters()], [gh.to(dt), gx.to(dt)])
        exact = exact.double()
        got, want = grads(ours, [ours.gcl_0, ours.gcl_1], torch.float32), grads(exact, exact.layers[:2], torch.float64)
        logs += [float(((a.double() - b).norm() / b.norm()).log()) for a, b in zip(got, want)]
    err = float(np.exp(np.mean(logs)))
    print("geometric mean of the errors:", err, flush=True)
    assert err <= 6.1e-7


@pytest.mark.parametrize("eq", [True, False])
@pytest.mark.parametrize("dims", [(128, 128, 128), (64, 32, 32)])
def test_infinite_operands(dims, eq):
    """Infinities come out where the float64 oracle has them, in the forward (an infinite bias of the first layer: each
    message feature is infinite or, as SiLU(-inf), NaN) and in the gradients (an infinite message gradient)."""
    H, O, M = dims
    degs = [0] * 20 + _degrees("halves")
    rowptr, col = random_csr(len(degs), degs, seed=8)
    case = Case(rowptr, col, 32, 8, H, O, M, seed=45, eq=eq)
    case.p["b1"][H - 3] = np.inf
    got = run_fused(case, "fp32", backward=False)["out_msg"]
    live = np.diff(rowptr) > 0
    up = case.p["w2_msg"][H - 3] > 0
    assert np.isposinf(got[live][:, up]).all() and np.isnan(got[live][:, ~up]).all() and (got[~live] == 0).all()

    case = Case(rowptr, col, 32, 8, H, O, M, seed=46, eq=eq)
    row, o = int(np.flatnonzero(np.diff(rowptr) == 1)[0]), 5     # a row of one edge: its gradient reaches one source
    case.gm[row, o] = np.inf
    want = case.backward_ref(False)
    res = run_fused(case, "fp32")["grads"]
    assert not np.isfinite(want["b1"]).any() and np.array_equal(np.sign(res["b1"]), np.sign(want["b1"]))
    assert np.isinf(res["b1"]).all()
    w2, ref = res["w2_msg"].reshape(H, O), want["w2_msg"].reshape(H, O)
    assert np.isfinite(np.delete(w2, o, 1)).all() and not np.isfinite(w2[:, o]).any()
    if H == 128:   # at H = 64 the large term and the corrections share an accumulator: NaN
        assert np.array_equal(w2[:, o], ref[:, o])


@pytest.mark.parametrize("N", [5, 4100])
def test_infinite_rows_of_node_products(N):
    from pymolecular_amd.node_update import dense
    torch.manual_seed(N)
    lin = torch.nn.Linear(128, 64).cuda()
    x = torch.randn(N, 128).cuda()
    x[3, 7] = float("inf")
    x.requires_grad_()
    y = dense(x, lin)
    assert torch.equal(y[3], torch.sign(lin.weight[:, 7]) * float("inf")) and torch.isfinite(y).sum() == (N - 1) * 64
