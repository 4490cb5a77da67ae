"""Queries that one workgroup runs in LDS: graphs up to the largest that fits
and just past it, thin (few edges a vertex, near-far buckets) and not, against
the oracle's Dijkstra; every way of taking the result; weights and `inf` at the
ends of their range; sources that reach nothing."""
import ctypes

import numpy as np
import pytest

import gpugraphalgo_amd as gga
from gpugraphalgo_amd import _lib
import oracle

pytestmark = pytest.mark.gpu
N = 12288    # vertices that fit


def random_graph(n: int, m: int, top: int, seed: int, spread: int):
    rng = np.random.default_rng(seed)
    u = np.sort(rng.integers(0, n, m))
    v = (u + rng.integers(0, spread, m)) % n          # self-loops and duplicates among them
    row = np.concatenate([[0], np.cumsum(np.bincount(u, minlength=n))]).astype(np.uint32)
    return gga.csr_from_arrays(row, v.astype(np.uint32), rng.integers(0, top, m, dtype=np.uint64).astype(np.uint32))


def star(n: int):
    row = np.full(n + 1, n - 1, dtype=np.uint32)
    row[0] = 0
    return gga.csr_from_arrays(row, np.arange(1, n, dtype=np.uint32), np.arange(1, n, dtype=np.uint32))


GRAPHS = {
    "one": lambda: gga.csr_from_arrays([0, 0], [], []),
    "two": lambda: gga.csr_from_arrays([0, 2, 3], [1, 1, 0], [7, 3, 1]),
    "grid1x33": lambda: gga.gen_grid(1, 33, 0.0, seed=1, wlo=1, whi=1000),
    "grid31x33": lambda: gga.gen_grid(31, 33, 0.0, seed=2, wlo=1, whi=1000),
    "grid96x128": lambda: gga.gen_grid(96, 128, 0.0, seed=3, wlo=1, whi=1000),          # exactly N
    "grid97x128": lambda: gga.gen_grid(97, 128, 0.0, seed=3, wlo=1, whi=1000),          # past it
    "grid16x700cut": lambda: gga.gen_grid(16, 700, 0.005, seed=4, wlo=1, whi=50),
    "wide_weights": lambda: random_graph(3000, 9000, 1 << 32, 5, 40),
    "zero_weights": lambda: random_graph(5000, 15000, 2, 6, 9),
    "sparse": lambda: random_graph(N, 16384, 100, 7, N),
    "dense": lambda: random_graph(200, 16384, 100, 8, 200),
    "rmat10": lambda: gga.gen_rmat(10, 12, seed=9, wlo=1, whi=100),
    "star": lambda: star(N),
}


@pytest.mark.parametrize("name", GRAPHS)
def test_one_workgroup_queries(gpu, name):
    g = GRAPHS[name]()
    ones = np.ones(g.m, dtype=np.uint32)
    hip = ctypes.CDLL("libamdhip64.so")
    buf = ctypes.c_void_p()
    assert hip.hipMalloc(ctypes.byref(buf), ctypes.c_size_t(4 * g.n)) == 0
    host = np.empty(g.n, dtype=np.uint32)
    deg = g.degrees().astype(np.int64)
    try:
        with gga.DeviceGraph(g) as dg:
            for mda in (0, 4):
                dg.split(mda=mda)
                for src in sorted({0, g.n // 2, g.n - 1}):
                    for inf in (gga.INF, gga.REF_INF, 3000):
                        for bfs in (True, False):
                            want = np.minimum(oracle.dijkstra(g.row_ptr, g.dst, ones if bfs else g.w, src, inf=inf), inf)
                            fn = dg.bfs if bfs else dg.sssp
                            for mode in ("auto", "worklist"):
                                print(f"[gpu] {name} mda={mda} src={src} inf={inf} bfs={bfs} {mode}", flush=True)
                                got, st = fn(src, mode=mode, inf=inf)
                                np.testing.assert_array_equal(got, want)
                                assert st["reached"] == int((want < inf).sum())
                                assert st["m_reach"] == int(deg[want < inf].sum())
                            fn(src, inf=inf, keep_on_device=True)
                            np.testing.assert_array_equal(dg.copy_dist(), want)
                            assert dg.verify(src, bfs=bfs, inf=inf)["src_ok"]
                            if not bfs:
                                o, st = gga.graph._opts("auto", inf, False, {}), _lib.Stats()
                                _lib.check(_lib.load().gga_sssp_noalloc(dg._h, src, buf, ctypes.byref(o),
                                                                        ctypes.byref(st)), "gga_sssp_noalloc")
                                assert hip.hipMemcpy(ctypes.c_void_p(host.ctypes.data), buf,
                                                     ctypes.c_size_t(4 * g.n), 2) == 0
                                np.testing.assert_array_equal(host, want)
                                # a scheduled query on the same handle in between
                                np.testing.assert_array_equal(dg.sssp(src, inf=inf, dense_min=1)[0], want)
    finally:
        hip.hipFree(buf)
