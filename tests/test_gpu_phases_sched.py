"""The step schedule on graphs that one workgroup would answer by itself, and
on larger ones with no option set: every query here has to be a chain of phase
launches (its `launches` say so), on one vertex, on chains of less and more
than a tile, repeated from sources that need more phases than the last one,
and after queries that ended at the step cap and left stamps behind."""
import numpy as np
import pytest

import gpugraphalgo_amd as gga
import oracle
from test_gpu_phases import chain

pytestmark = pytest.mark.gpu
NEVER = 0xFFFFFFFF
# options that ask for a schedule without changing what a default one does
SCHEDULES = ({"dense_min": NEVER}, {"delta": NEVER}, {"sync_every": 8})


@pytest.mark.parametrize("kw", SCHEDULES)
def test_one_vertex(gpu, kw):
    g = gga.csr_from_arrays([0, 0], [], [])
    with gga.DeviceGraph(g) as dg:
        for fn in (dg.bfs, dg.sssp):
            for _ in range(2):
                got, st = fn(0, mode="worklist", **kw)
                assert got.tolist() == [0] and st["reached"] == 1 and st["m_reach"] == 0
                assert st["launches"] > 1 and st["iterations"] <= 1


@pytest.mark.parametrize("n", [2, 3, 64, 700, 2049, 5000, 13000, 20001])
def test_scheduled_queries(gpu, n):
    g = chain(n, 50)
    deg = g.degrees().astype(np.int64)
    srcs = (n - 1, 0, n // 2)                  # few phases, many, about half
    want = {s: oracle.dijkstra(g.row_ptr, g.dst, g.w, s) for s in srcs}
    hops = {s: oracle.dijkstra(g.row_ptr, g.dst, np.ones(g.m, dtype=np.uint32), s) for s in srcs}
    kws = SCHEDULES if n <= 12288 else SCHEDULES + ({},)

    def check(dg, s, kw):
        print(f"[gpu] n={n} src={s} {kw}", flush=True)
        got, st = dg.sssp(s, mode="worklist", **kw)
        np.testing.assert_array_equal(got, want[s])
        assert st["launches"] > 1
        assert st["reached"] == int((want[s] < gga.INF).sum())
        assert st["m_reach"] == int(deg[want[s] < gga.INF].sum())
        got, st = dg.bfs(s, mode="worklist", **kw)
        np.testing.assert_array_equal(got, hops[s])
        assert st["launches"] > 1

    with gga.DeviceGraph(g) as dg:
        dg.split(mda=16)
        for kw in kws:
            for s in srcs + srcs:
                check(dg, s, kw)
        if n >= 700:                           # far more steps than the cap
            for cap in ({}, {"dense_min": 1}, {"delta": 120}):
                with pytest.raises(gga.graph._lib.GgaError):
                    dg.sssp(0, mode="worklist", max_iters=20, **cap)
                for kw in kws:
                    check(dg, 0, kw)
