"""Multi-source engine: 32 lanes meet at one vertex, whose edges are staged 64
at a time -- degrees at the edges of that group, all lanes or half of them
SSSP, both layouts, against the oracle's Dijkstra."""
import numpy as np
import pytest

import gpugraphalgo_amd as gga
import oracle

pytestmark = pytest.mark.gpu
LANES = 32


def funnel(leaves: int):
    """32 sources -> vertex 32 -> `leaves` vertices, each with an edge on to the
    next leaf and every seventh back to the middle."""
    rng = np.random.default_rng(leaves)
    mid, first = LANES, LANES + 1
    n = first + leaves
    edges = [(i, mid, int(rng.integers(1, 50))) for i in range(LANES)]
    edges += [(mid, first + k, int(rng.integers(0, 90))) for k in range(leaves)]
    for k in range(leaves):
        edges.append((first + k, first + (k + 1) % leaves, int(rng.integers(1, 9))))
        if k % 7 == 0:
            edges.append((first + k, mid, 1))
    edges.sort(key=lambda e: e[0])
    u, v, w = (np.array(x, dtype=np.int64) for x in zip(*edges))
    row = np.concatenate([[0], np.cumsum(np.bincount(u, minlength=n))]).astype(np.uint32)
    return gga.csr_from_arrays(row, v.astype(np.uint32), w.astype(np.uint32))


@pytest.mark.parametrize("leaves", [1, 7, 8, 9, 63, 64, 65, 127, 129, 1000])
def test_staged_edges(gpu, leaves):
    g = funnel(leaves)
    ones = np.ones(g.m, dtype=np.uint32)
    with gga.DeviceGraph(g) as dg:
        for mda in (0, 16):
            dg.split(mda=mda)
            for layout in ("vertex", "lane"):
                for inf in (gga.INF, 60):
                    for half, delta, mode in ((0, 0, "worklist"), (16, 0, "worklist"), (0, 20, "worklist"),
                                              (16, 0, "persistent")):
                        print(f"[gpu] leaves={leaves} mda={mda} {layout} inf={inf} bfs lanes={half} "
                              f"delta={delta} {mode}", flush=True)
                        with gga.MultiSourceEngine(dg, inf=inf, layout=layout) as eng:
                            eng.set_delta(delta)
                            eng.start({i: i for i in range(LANES)}, bfs=set(range(half)))
                            assert eng.run(mode=mode) == 0
                            got = eng.fetch(range(LANES))
                        for i in range(LANES):
                            want = oracle.dijkstra(g.row_ptr, g.dst, ones if i < half else g.w, i, inf=inf)
                            np.testing.assert_array_equal(got[i], np.minimum(want, inf))
