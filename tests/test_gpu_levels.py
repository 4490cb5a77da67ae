"""Level-synchronous BFS (graphs that are not mesh-like, worklist and
persistent modes) where its byte stamps repeat: more than 254 levels, beside a
hub that keeps the graph from being mesh-like.  Every frontier form, against
the oracle's queue BFS."""
import numpy as np
import pytest

import gpugraphalgo_amd as gga
import oracle

pytestmark = pytest.mark.gpu


def long_graph(levels: int, leaves: int, tail: int):
    """A path of `levels` arcs whose vertices also point back to the hub at its
    start; the hub points to `leaves` leaves, and every 10th path vertex to a
    leaf of its own (so that flag steps list more than one vertex)."""
    edges = [(i, i + 1) for i in range(levels)]
    edges += [(i, 0) for i in range(1, levels + 1, 7)]
    first = levels + 1
    edges += [(0, first + k) for k in range(leaves)]
    side = first + leaves
    edges += [(10 * k, side + k) for k in range(levels // 10)]
    n = side + levels // 10 + tail      # `tail` isolated vertices
    e = np.array(sorted(edges), dtype=np.int64)
    row = np.zeros(n + 1, dtype=np.uint32)
    row[1:] = np.cumsum(np.bincount(e[:, 0], minlength=n))
    return gga.csr_from_arrays(row, e[:, 1].astype(np.uint32))


@pytest.mark.parametrize("levels,leaves,tail", [(253, 64, 0), (254, 65, 3), (255, 70, 1), (700, 90, 5), (2600, 300, 2)])
@pytest.mark.parametrize("mode", ["worklist", "persistent"])
def test_levels_past_the_stamp_wrap(gpu, levels, leaves, tail, mode):
    g = long_graph(levels, leaves, tail)
    ones = np.ones(g.m, dtype=np.uint32)
    with gga.DeviceGraph(g) as dg:
        for mda in (0, 16):
            dg.split(mda=mda)
            for src in (0, 3, levels // 2):
                for inf in (gga.INF, gga.REF_INF):
                    want = oracle.dijkstra(g.row_ptr, g.dst, ones, src, inf=inf)
                    for dense_min in (1, 2, 0, 0xFFFFFFFF):
                        print(f"[gpu] levels={levels} {mode} mda={mda} src={src} inf={inf} dense_min={dense_min}",
                              flush=True)
                        got, st = dg.bfs(src, mode=mode, inf=inf, dense_min=dense_min)
                        np.testing.assert_array_equal(got, want)
                        assert st["reached"] == int((want < inf).sum())
                # an `inf` that some levels reach: those vertices stay unreached
                small = levels // 2
                want = np.minimum(oracle.dijkstra(g.row_ptr, g.dst, ones, src), small)
                for dense_min in (1, 0xFFFFFFFF):
                    got, _ = dg.bfs(src, mode=mode, inf=small, dense_min=dense_min)
                    np.testing.assert_array_equal(got, want)
