"""Near-far engine: graphs whose deferred vertices spread over fewer tiles of 64
than there are waves, just as many, and more, against the oracle's Dijkstra."""
import numpy as np
import pytest

import gpugraphalgo_amd as gga
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(1, 63), (1, 65), (5, 205), (31, 33), (32, 32), (64, 512), (64, 513),
                                       (300, 500), (512, 1025)])
@pytest.mark.parametrize("layout", ["vertex", "lane"])
def test_refill_spread(gpu, rows, cols, layout):
    g = gga.gen_grid(rows, cols, 0.0, seed=rows + cols, wlo=1, whi=100)
    lanes = {0: 0, 7: g.n // 2, 31: g.n - 1}
    ones = np.ones(g.m, dtype=np.uint32)
    with gga.DeviceGraph(g) as dg:
        dg.split(mda=0)
        for delta in (40, 400, 0xFFFFFFF0):
            print(f"[gpu] {rows} x {cols} {layout} delta={delta}", flush=True)
            with gga.MultiSourceEngine(dg, layout=layout) as eng:
                eng.set_delta(delta)
                eng.start(lanes, bfs={7})
                assert eng.run() == 0
                got = eng.fetch(lanes)
            for i, src in lanes.items():
                want = oracle.dijkstra(g.row_ptr, g.dst, ones if i == 7 else g.w, src)
                np.testing.assert_array_equal(got[i], want)
