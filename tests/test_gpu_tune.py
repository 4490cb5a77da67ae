"""gga_tune never leaves a graph slower than it found it: meshes, where the
default schedule runs near-far buckets (and small ones in one workgroup), and
R-MAT, single-source and through the multi-source engine.

The choices that a mistake would record -- plain Bellman-Ford on a mesh, a
switch or grid of another mode -- cost a factor of two and more, repeated calls
differ by a few percent: the line lies at 1.5."""
import time

import numpy as np
import pytest

import gpugraphalgo_amd as gga
import oracle

pytestmark = pytest.mark.gpu

GRAPHS = {
    "grid16x700": lambda: gga.gen_grid(16, 700, 0.0, seed=1, wlo=1, whi=1000),      # one workgroup
    "grid300x300": lambda: gga.gen_grid(300, 300, 0.0, seed=2, wlo=1, whi=1000),
    "grid1024x1024": lambda: gga.gen_grid(1024, 1024, 0.0, seed=3, wlo=1, whi=1000),
    "rmat12": lambda: gga.gen_rmat(12, 4, seed=4, wlo=1, whi=100),                  # one workgroup
    "rmat16": lambda: gga.gen_rmat(16, 16, seed=5, wlo=1, whi=100),
}


def best_of(fn, k=7):
    fn()
    fn()
    t = []
    for _ in range(k):
        t0 = time.perf_counter()
        fn()
        t.append(time.perf_counter() - t0)
    return min(t)


@pytest.mark.parametrize("name", GRAPHS)
def test_tuned_no_slower_than_untuned(gpu, name):
    g = GRAPHS[name]()
    src = int(np.flatnonzero(g.degrees() > 0)[g.n // 3])
    srcs = np.flatnonzero(g.degrees() > 0)[:: max(1, g.n // 40)][:8]
    with gga.DeviceGraph(g) as dg:
        def calls():
            return {"sssp": best_of(lambda: dg.sssp(src, keep_on_device=True)),
                    "persistent": best_of(lambda: dg.sssp(src, mode="persistent", keep_on_device=True)),
                    "engine": best_of(lambda: dg.multi_sp(srcs, keep_on_device=True), 3)}
        dg.split(mda=64)
        before = calls()
        for rep in range(2):
            tr = dg.tune(src)
            after = calls()
            print(f"[gpu] {name} {before} -> {after} {tr}", flush=True)
            for k in before:
                assert after[k] <= 1.5 * before[k], k
        np.testing.assert_array_equal(dg.sssp(src)[0], oracle.dijkstra(g.row_ptr, g.dst, g.w, src))
