"""Waves following their front on mesh-like graphs whose degrees cross the
limits of that path: four edges per vertex and round, 16 followed at most, a
queue that overflows (random graphs spread within a few hops), ids past the
last full group, isolated vertices.  Against the oracle's Dijkstra."""
import numpy as np
import pytest

import gpugraphalgo_amd as gga
import oracle

pytestmark = pytest.mark.gpu


def spread_graph(n: int, degrees, reach: int, seed: int):
    """Vertex v has degrees[v % len] arcs to vertices within `reach` ids (mod n)."""
    rng = np.random.default_rng(seed)
    deg = np.resize(np.asarray(degrees, dtype=np.int64), n)
    u = np.repeat(np.arange(n), deg)
    dst = (u + rng.integers(1, reach + 1, u.size)) % n
    row = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint32)
    return gga.csr_from_arrays(row, dst.astype(np.uint32), rng.integers(1, 1001, u.size))


CASES = [
    ("one_vertex", 1, [1], 1),
    ("ring", 65, [1], 1),
    ("pairs", 1023, [2, 2, 2, 2], 5),
    ("deg4_5", 4099, [4, 5, 3, 4], 40),
    ("deg16_17", 5003, [4, 16, 17, 3, 0, 5, 8, 9], 60),
    ("hubs24", 8191, [3, 4, 24, 5, 4, 3], 30),
    ("random", 20000, [4, 5, 6, 3], 19999),
]


@pytest.mark.parametrize("name,n,degrees,reach", CASES, ids=[c[0] for c in CASES])
@pytest.mark.parametrize("mode", ["worklist", "persistent"])
def test_followed_fronts(gpu, name, n, degrees, reach, mode):
    g = spread_graph(n, degrees, reach, seed=n)
    mean = (g.m + n - 1) // n
    assert g.maxdeg()[0] <= 4 * mean + 8, "the graph has to be mesh-like"
    ones = np.ones(g.m, dtype=np.uint32)
    with gga.DeviceGraph(g) as dg:
        dg.split()
        for src in sorted({0, n // 2, n - 1}):
            hops = oracle.dijkstra(g.row_ptr, g.dst, ones, src)
            dist = oracle.dijkstra(g.row_ptr, g.dst, g.w, src)
            for dense_min in (0, 1, 64, 0xFFFFFFFF):
                print(f"[gpu] {name} {mode} src={src} dense_min={dense_min}", flush=True)
                np.testing.assert_array_equal(dg.bfs(src, mode=mode, dense_min=dense_min)[0], hops)
                for delta in (0, 1000, 0xFFFFFFFF):
                    got, st = dg.sssp(src, mode=mode, dense_min=dense_min, delta=delta)
                    np.testing.assert_array_equal(got, dist)
                    assert st["reached"] == int((dist < gga.INF).sum())


@pytest.mark.parametrize("name,n,degrees,reach", CASES, ids=[c[0] for c in CASES])
@pytest.mark.parametrize("layout", [1, 2], ids=["vertex", "lane"])
def test_followed_fronts_of_engine_lanes(gpu, name, n, degrees, reach, layout):
    g = spread_graph(n, degrees, reach, seed=n + 1)
    ones = np.ones(g.m, dtype=np.uint32)
    rng = np.random.default_rng(n)
    srcs = rng.integers(0, n, 32).astype(np.uint32)
    unit = 0x0F0F00FF                    # BFS lanes
    want = [oracle.dijkstra(g.row_ptr, g.dst, ones if (unit >> i) & 1 else g.w, int(s)) for i, s in enumerate(srcs)]
    with gga.DeviceGraph(g) as dg:
        dg.split()
        for k in (1, 32):
            for dense_min in (0, 1, 0xFFFFFFFF):
                for delta in (0, 1000, 0xFFFFFFFF):
                    print(f"[gpu] {name} layout={layout} k={k} dense_min={dense_min} delta={delta}", flush=True)
                    got, _ = dg.multi_sp(srcs[:k], bfs_lanes=unit & ((1 << k) - 1), ms_layout=layout,
                                         dense_min=dense_min, delta=delta)
                    for i in range(k):
                        np.testing.assert_array_equal(got[i], want[i], err_msg=f"lane {i}")
