"""One-workgroup queries whose fronts hold most of the vertices: sparse uniform
graphs of the largest size that fits, where nearly every vertex is lowered (and
queued) several times and waits in both queues at once, over many sources."""
import numpy as np
import pytest

import gpugraphalgo_amd as gga
import oracle

pytestmark = pytest.mark.gpu
N = 12288


def uniform(n: int, m: int, top: int, seed: int):
    rng = np.random.default_rng(seed)
    u = np.sort(rng.integers(0, n, m))
    row = np.concatenate([[0], np.cumsum(np.bincount(u, minlength=n))]).astype(np.uint32)
    return gga.csr_from_arrays(row, rng.integers(0, n, m).astype(np.uint32), rng.integers(1, top, m).astype(np.uint32))


@pytest.mark.parametrize("n,m,top", [(N, 6 * N, 2), (N, 6 * N, 1000), (N - 1, 5 * N, 30), (4097, 6 * 4097, 100)])
def test_wide_fronts(gpu, n, m, top):
    g = uniform(n, m, top, n + m + top)
    ones = np.ones(g.m, dtype=np.uint32)
    with gga.DeviceGraph(g) as dg:
        dg.split()
        for src in range(0, n, n // 7):
            for bfs in (True, False):
                print(f"[gpu] n={n} m={m} top={top} src={src} bfs={bfs}", flush=True)
                want = oracle.dijkstra(g.row_ptr, g.dst, ones if bfs else g.w, src)
                for _ in range(3):
                    got, st = (dg.bfs if bfs else dg.sssp)(src)
                    assert st["launches"] == 1      # the one-workgroup kernel
                    np.testing.assert_array_equal(got, want)
