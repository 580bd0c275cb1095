"""The schedule's counting path and the graph builder's key search at their limits, bit for bit."""
import numpy as np
import pytest
import torch

from oracle import graph_oracle as go
from tests.test_schedule import schedule_ref

pytestmark = pytest.mark.gpu


def _check(rowptr, col):
    from pymolecular_amd import fused
    rp, c = torch.from_numpy(rowptr).cuda(), torch.from_numpy(col).cuda()
    print(f"[schedule] N={len(rowptr) - 1} E={len(col)} longest={np.bincount(col).max() if len(col) else 0}", flush=True)
    got = fused.schedule_arrays(fused._build_schedule(rp, c, len(rowptr) - 1))
    ref = schedule_ref(rowptr, col)
    for k, v in ref.items():
        assert np.array_equal(got[k].cpu().numpy(), v), k


@pytest.mark.parametrize("lens", [[1], [0, 2, 0], [63, 64, 65], [128, 129, 3], [256, 257], [511, 512], [513, 4], [2000]])
def test_source_list_lengths(lens):
    """Lists at the register variants' edges (64, 128, 256, 512) and past them (the radix sort)."""
    r = np.random.Generator(np.random.PCG64(len(lens)))
    N = 300
    col = r.permutation(np.concatenate([np.repeat(np.arange(len(lens)) * 7, lens), np.arange(150, 260)])).astype(np.int32)
    deg = np.bincount(r.integers(0, N, size=len(col)), minlength=N)
    _check(np.concatenate([[0], np.cumsum(deg)]).astype(np.int32), col)


@pytest.mark.parametrize("E,hubs,share", [(512, 1, 1.0), (513, 1, 1.0), (40_000, 1, 0.5), (100_000, 5, 1.0), (100_000, 40, 1.0),
                                          (300_000, 1, 0.01), (786_432, 20, 0.9)])
def test_hub_sources(E, hubs, share):
    """Few sources with most of the edges, around the sampled rule that leaves them to the radix sort."""
    r = np.random.Generator(np.random.PCG64(E + hubs))
    N = 5000
    col = np.where(r.random(E) < share, r.integers(0, hubs, size=E) * 97, r.integers(0, N, size=E)).astype(np.int32)
    deg = np.bincount(r.integers(0, N, size=E), minlength=N)
    _check(np.concatenate([[0], np.cumsum(deg)]).astype(np.int32), col)


@pytest.mark.parametrize("N", [1, 2047, 2048, 2049, 65536, 65537, 2048 * 1025 + 3])
def test_scan_block_edges(N):
    """Node counts around one block of the scan, the two row-id launches, and the separate prefix launch."""
    r = np.random.Generator(np.random.PCG64(N))
    E = min(3 * N, 40000)
    deg = np.bincount(r.integers(0, N, size=E), minlength=N)
    col = r.integers(max(0, N - 60000), N, size=E).astype(np.int32)
    _check(np.concatenate([[0], np.cumsum(deg)]).astype(np.int32), col)


@pytest.mark.parametrize("n,k", [(64, 5), (65, 64), (130, 31), (300, 30), (513, 30), (1030, 64)])
@pytest.mark.parametrize("kind", ["grid", "shell"])
def test_ties_in_the_search_key(n, k, kind):
    """Equal fp64 distances (integer grid), and distances that differ in fp64 only (points within 1e-12 of a sphere)."""
    from pymolecular_amd import graph_build
    r = np.random.Generator(np.random.PCG64(n + k))
    if kind == "grid":
        pos = r.integers(-3, 4, size=(n + 9, 3)).astype(np.float64)
    else:
        v = r.standard_normal((n + 9, 3))
        pos = v / np.linalg.norm(v, axis=1, keepdims=True) * (1.0 + 1e-12 * r.standard_normal((n + 9, 1)))
        pos[n // 2] = 0.0   # the centre: all of its candidates share one fp32 key
    seg = [0, n, n + 9]
    p, s = torch.from_numpy(pos).cuda(), torch.tensor(seg, dtype=torch.int32).cuda()
    for got, ref in ((graph_build.knn_graph(p, s, k), go.knn_graph(pos, seg, k)),
                     (graph_build.radius_graph(p, s, 1.0, k), go.radius_graph(pos, seg, 1.0, k))):
        assert np.array_equal(got[0].cpu().numpy(), ref[0]) and np.array_equal(got[1].cpu().numpy(), ref[1])
