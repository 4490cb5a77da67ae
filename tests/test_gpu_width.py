"""Default near-far widths by graph and launch mode, seen in the steps a query
takes, and the results under them."""
import numpy as np
import pytest

import gpugraphalgo_amd as gga
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["auto", "worklist", "persistent"])
def test_paths_take_wide_buckets(gpu, mode):
    """A path of equal weights: a bucket of 32 mean weights is 32 hops, which
    one wave follows within a step (the last bucket may end in a step of its
    own, as may the first)."""
    n = 20000
    g = gga.gen_grid(1, n, 0.0, seed=1, wlo=7, whi=7)
    with gga.DeviceGraph(g) as dg:
        dg.split()
        d, st = dg.sssp(0, mode=mode)
        print(f"[gpu] path {mode}: {st['iterations']} steps", flush=True)
        np.testing.assert_array_equal(d, 7 * np.arange(n, dtype=np.uint32))
        assert st["iterations"] <= n // 32 + 2


def test_persistent_takes_wider_buckets_than_worklist(gpu):
    """A thin grid: the steps of a query by default are those of 16 mean
    weights in the persistent kernel and of 8 in the worklist launches
    (followed fronts race, so steps vary a little: the nearer one counts)."""
    g = gga.gen_grid(4, 3000, 0.0, seed=2, wlo=1, whi=1000)
    mean = -(-int(g.w.astype(np.int64).sum()) // g.m)
    want = oracle.dijkstra(g.row_ptr, g.dst, g.w, 0)
    with gga.DeviceGraph(g) as dg:
        dg.split()
        for mode, near, far in (("persistent", 16, 8), ("worklist", 8, 16)):
            steps = {}
            for k in (0, near, far):
                # (an explicit step period keeps the query out of the one-workgroup kernel)
                d, st = dg.sssp(0, mode=mode, delta=k * mean, sync_every=8)
                np.testing.assert_array_equal(d, want)
                steps[k] = st["iterations"]
            print(f"[gpu] {mode}: {steps}", flush=True)
            assert abs(steps[0] - steps[near]) < abs(steps[0] - steps[far])
