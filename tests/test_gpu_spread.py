"""SSSP with its atomics on the permuted copy of the distances (graphs whose
hubs are neighbouring ids): sizes around the copy's least and its powers of
two, every list form, counted and tuned workgroup sizes, re-splits, the
allocation-free query, and results that stay exact from query to query."""
import ctypes

import numpy as np
import pytest

import gpugraphalgo_amd as gga
from gpugraphalgo_amd import _lib
import oracle

pytestmark = pytest.mark.gpu


def hub_graph(n: int, seed: int):
    """Every vertex points to a few of the 40 lowest ids and to random ones; the
    low ids point everywhere.  Heavy ties and repeated improvements."""
    rng = np.random.default_rng(seed)
    lo = min(n, 40)
    u = np.concatenate([np.repeat(np.arange(n), 3), rng.integers(0, lo, 8 * n)])
    v = np.concatenate([rng.integers(0, lo, 2 * n), rng.integers(0, n, n), rng.integers(0, n, 8 * n)])
    order = np.argsort(u, kind="stable")
    row = np.concatenate([[0], np.cumsum(np.bincount(u, minlength=n))]).astype(np.uint32)
    return gga.csr_from_arrays(row, v[order].astype(np.uint32), rng.integers(0, 30, u.size))


def skewed(g):
    share = max(int(g.row_ptr[min(g.n, v + 64)]) - int(g.row_ptr[v]) for v in range(0, g.n, 64))
    mean = (g.m + g.n - 1) // g.n
    return share > g.m // 64 and g.maxdeg()[0] > 4 * mean + 8


@pytest.mark.parametrize("n", [257, 4099, 65535, 65536, 65537, 131072, 131073])
def test_spread_distances(gpu, n):
    g = hub_graph(n, seed=n)
    assert skewed(g)
    hip = ctypes.CDLL("libamdhip64.so")
    buf = ctypes.c_void_p()
    assert hip.hipMalloc(ctypes.byref(buf), ctypes.c_size_t(4 * n)) == 0
    host = np.empty(n, dtype=np.uint32)
    try:
        with gga.DeviceGraph(g) as dg:
            for mda in (16, 0):
                dg.split(mda=mda)
                for src in (0, n // 2, n - 1):
                    for inf in (gga.INF, 40):
                        want = np.minimum(oracle.dijkstra(g.row_ptr, g.dst, g.w, src), inf)
                        for kw in ({}, {"dense_min": 1}, {"dense_min": 0xFFFFFFFF}, {"count": True}, {"block": 128},
                                   {"block": 512, "dense_min": 1}, {"mode": "worklist", "delta": 7}):
                            print(f"[gpu] n={n} mda={mda} src={src} inf={inf} {kw}", flush=True)
                            got, st = dg.sssp(src, inf=inf, **kw)
                            np.testing.assert_array_equal(got, want)
                            assert st["reached"] == int((want < inf).sum())
                        o = gga.graph._opts("worklist", inf, False, {})
                        st = _lib.Stats()
                        _lib.check(_lib.load().gga_sssp_noalloc(dg._h, src, buf, ctypes.byref(o), ctypes.byref(st)),
                                   "gga_sssp_noalloc")
                        assert hip.hipMemcpy(ctypes.c_void_p(host.ctypes.data), buf, ctypes.c_size_t(4 * n), 2) == 0
                        np.testing.assert_array_equal(host, want)
    finally:
        hip.hipFree(buf)
