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
