"""The layer's native autograd node against the Python one: the same kernels, so bit for bit the same results."""
import threading

import pytest
import torch

from pymolecular_amd import _capi, graphs, layer_fn
from pymolecular_amd.models.EGNN import E_GCL, MPNN_GCL

pytestmark = pytest.mark.gpu


def _setup(kind, dtype, fe, H=128, residual=True, seed=3):
    g = graphs.molecule_batch(3, seed=seed, feat_seed=seed)
    gen = torch.Generator().manual_seed(seed)
    rows = torch.repeat_interleave(torch.arange(g.N), torch.diff(torch.from_numpy(g.rowptr).long())).cuda()
    edges = [rows, torch.from_numpy(g.col.astype("int64")).cuda()]
    torch.manual_seed(seed)
    net = (E_GCL(H, H, H, edges_in_d=fe, residual=residual) if kind == "egnn" else MPNN_GCL(H, H, H, edges_in_d=fe, residual=residual))
    net = net.to("cuda", dtype)
    h = torch.randn(g.N, H, generator=gen).to("cuda", dtype)
    x = torch.randn(g.N, 3, generator=gen).cuda() if kind == "egnn" else None
    ea = torch.randn(len(g.col), fe, generator=gen).to("cuda", dtype) if fe else None
    return net, h, x, edges, ea


def _run(net, h, x, edges, ea, use=(True, True)):
    h = h.detach().requires_grad_()
    x = None if x is None else x.detach().requires_grad_()
    out = net(h, edges, x, edge_attr=ea)[:2] if x is not None else net(h, edges, ea)[:1]
    gen = torch.Generator(device="cuda").manual_seed(5)
    outs = [o for o, u in zip(out, use) if u]
    gout = [torch.randn(o.shape, generator=gen, device="cuda").to(o.dtype) for o in outs]
    wrt = [h] + ([] if x is None else [x]) + list(net.parameters())
    return [o.detach() for o in out] + list(torch.autograd.grad(outs, wrt, gout, allow_unused=True))


class _Refuse:
    @staticmethod
    def gcl_layer(*a):
        return None


def _python_only(monkeypatch):
    monkeypatch.setattr(layer_fn, "ext", lambda: _Refuse)


def _same(a, b):
    assert len(a) == len(b)
    for u, v in zip(a, b):
        assert (u is None) == (v is None)
        assert u is None or (u.shape == v.shape and u.dtype == v.dtype and torch.equal(u, v))


@pytest.mark.parametrize("kind,dtype,fe,H,residual", [
    ("egnn", torch.float32, 0, 128, True), ("egnn", torch.bfloat16, 16, 128, True), ("egnn", torch.float32, 8, 128, False),
    ("egnn", torch.bfloat16, 32, 256, True), ("mpnn", torch.bfloat16, 16, 128, True), ("mpnn", torch.float32, 0, 128, True)])
def test_matches_python_node(kind, dtype, fe, H, residual, monkeypatch):
    args = _setup(kind, dtype, fe, H, residual)
    uses = [(True, True)] + ([(True, False), (False, True)] if kind == "egnn" else [])
    native = [_run(*args, use=u) for u in uses]
    seen = []
    real = _capi.ext().gcl_layer
    monkeypatch.setattr(layer_fn, "ext", lambda: type("E", (), {"gcl_layer": staticmethod(lambda *a: seen.append(real(*a)) or seen[-1])}))
    _same(native[0], _run(*args))
    assert seen and seen[0] is not None   # these calls take the native node
    _python_only(monkeypatch)
    for u, n in zip(uses, native):
        _same(n, _run(*args, use=u))


@pytest.mark.parametrize("what", ["h strided", "h other dtype", "x double", "x wide", "attr dtype", "frozen", "no grad", "stream",
                                  "hooks", "thread", "retain"])
def test_other_calls(what, monkeypatch):
    """Inputs that need a conversion (the Python node), and the ways a native node is called: same results either way."""
    net, h, x, edges, ea = _setup("egnn", torch.float32, 8)
    if what == "h strided":
        h = torch.cat([h, h], 1)[:, :128]
    elif what == "h other dtype":
        h = h.bfloat16()
        ea = ea.bfloat16()
    elif what == "x double":
        x = x.double()
    elif what == "attr dtype":
        ea = ea.double()
    elif what == "frozen":
        for p in list(net.parameters())[:6]:
            p.requires_grad_(False)

    def call():
        if what == "no grad":
            with torch.no_grad():
                return list(net(h, edges, x, edge_attr=ea)[:2])
        if what == "hooks":
            with torch.autograd.graph.saved_tensors_hooks(lambda t: t.cpu(), lambda t: t.cuda()):
                return _run(net, h, x, edges, ea)
        if what == "stream":
            st = torch.cuda.Stream()
            st.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(st):
                r = _run(net, h, x, edges, ea)
            st.synchronize()
            return r
        if what == "thread":
            r = []
            ts = [threading.Thread(target=lambda: r.append(_run(net, h, x, edges, ea))) for _ in range(2)]
            [t.start() for t in ts]
            [t.join() for t in ts]
            _same(r[0], r[1])
            return r[0]
        if what == "retain":
            hh = h.detach().requires_grad_()
            out = net(hh, edges, x, edge_attr=ea)[0]
            a = torch.autograd.grad(out.sum(), hh, retain_graph=True)[0]
            b = torch.autograd.grad(out.sum(), hh)[0]
            assert torch.equal(a, b)
            return [a]
        if what == "frozen":
            hh = h.detach().requires_grad_()
            ps = [p for p in net.parameters() if p.requires_grad]
            return list(torch.autograd.grad(net(hh, edges, x, edge_attr=ea)[0].sum(), [hh] + ps, allow_unused=True))
        if what == "x wide":
            return list(net(h, edges, torch.cat([x, x], 1)[:, :3], edge_attr=ea)[:2])
        return _run(net, h, x, edges, ea)
    a = call()
    _python_only(monkeypatch)
    _same(a, call())


def test_errors_stay():
    net, h, x, edges, ea = _setup("egnn", torch.float32, 8)
    with pytest.raises(ValueError):   # feature width that does not fit the weights
        net(h, edges, x, edge_attr=torch.cat([ea, ea], 1))
    with pytest.raises(TypeError):
        net(h.half(), edges, x, edge_attr=ea)
    with pytest.raises(RuntimeError):
        net(h.cpu(), edges, x, edge_attr=ea)
    out = net(h.requires_grad_(), edges, x, edge_attr=ea)[0]
    with torch.no_grad():
        net.edge_mlp[0].weight.add_(1.0)
    with pytest.raises(RuntimeError):   # a saved weight changed in place
        out.sum().backward()
