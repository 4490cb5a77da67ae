"""A query's time_ms starts with the initialisation.

The first workgroup lists the source's chunks; where the source is a hub cut
into one chunk an edge, that is the longest part of the query, and it cannot
take less than its bytes at the rate of one CU's stores (64 bytes a clock at
2.4 GHz)."""
import numpy as np
import pytest

import gpugraphalgo_amd as gga

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kw", [{"mode": "auto"}, {"mode": "worklist", "block": 128}, {"mode": "persistent"}])
def test_time_covers_initialisation(gpu, kw):
    n = 1 << 24
    row = np.full(n + 1, n - 1, dtype=np.uint32)
    row[0] = 0
    with gga.DeviceGraph(gga.csr_from_arrays(row, np.arange(1, n, dtype=np.uint32))) as dg:
        dg.split(mda=1)
        for _ in range(3):
            st = dg.bfs(0, keep_on_device=True, **kw)[1]
            assert st["reached"] == n
            print(f"[gpu] {kw} time_ms={st['time_ms']:.4f}", flush=True)
            assert st["time_ms"] >= 4 * (n - 1) / (64 * 2.4e9) * 1e3
