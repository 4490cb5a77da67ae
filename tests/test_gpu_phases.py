"""Worklist queries run one phase per launch: the host's batches of launches
(first query, repeated ones, sources that need more phases than the last one,
`sync_every`), the step cap, near-far threshold jumps, and the read-back that
ends a query on graphs of one vertex up to several tiles."""
import numpy as np
import pytest

import gpugraphalgo_amd as gga
import oracle

pytestmark = pytest.mark.gpu


def chain(n: int, weight: int):
    """0 -> 1 -> ... -> n - 1, and a hub at the end that points back to all."""
    dst = np.concatenate([np.arange(1, n), np.arange(n - 1)])
    row = np.concatenate([np.arange(n), [2 * (n - 1)]]).astype(np.uint32)
    return gga.csr_from_arrays(row, dst.astype(np.uint32), np.full(dst.size, weight, dtype=np.uint32))


@pytest.mark.parametrize("n", [2, 3, 64, 700, 2049, 5000])
def test_batches_caps_and_readback(gpu, n):
    g = chain(n, 50)
    want = {s: oracle.dijkstra(g.row_ptr, g.dst, g.w, s) for s in (0, n // 2, n - 1)}
    hops = {s: oracle.dijkstra(g.row_ptr, g.dst, np.ones(g.m, dtype=np.uint32), s) for s in want}
    with gga.DeviceGraph(g) as dg:
        dg.split(mda=16)
        for rep in range(2):
            for s in (n - 1, 0, n // 2):      # few phases, many, about half
                for kw in ({}, {"sync_every": 1}, {"sync_every": 5}, {"dense_min": 1}, {"delta": 1}, {"delta": 120}):
                    print(f"[gpu] n={n} rep={rep} src={s} {kw}", flush=True)
                    got, st = dg.sssp(s, mode="worklist", **kw)
                    np.testing.assert_array_equal(got, want[s])
                    assert st["reached"] == int((want[s] < gga.INF).sum())
                    deg = g.degrees().astype(np.int64)
                    assert st["m_reach"] == int(deg[want[s] < gga.INF].sum())
                    assert st["time_ms"] > 0
                    np.testing.assert_array_equal(dg.bfs(s, mode="worklist", **kw)[0], hops[s])
        if n >= 700:                           # far more steps than the cap
            for kw in ({}, {"dense_min": 1}, {"delta": 120}):
                with pytest.raises(gga.graph._lib.GgaError):
                    dg.sssp(0, mode="worklist", max_iters=20, **kw)
            np.testing.assert_array_equal(dg.sssp(0, mode="worklist")[0], want[0])


def test_one_vertex(gpu):
    g = gga.csr_from_arrays([0, 0], [], [])
    with gga.DeviceGraph(g) as dg:
        for fn in (dg.bfs, dg.sssp):
            got, st = fn(0, mode="worklist")
            assert got.tolist() == [0] and st["reached"] == 1 and st["m_reach"] == 0
