"""Which graphs get the permuted copy of the distances (131 072 words for 100 000
vertices), by the device memory that a graph takes beyond a uniform one of the
same size -- and the distances, either way."""
import numpy as np
import pytest

import gpugraphalgo_amd as gga
import oracle

pytestmark = pytest.mark.gpu
N, M = 100000, 1600000


def graph(out_hubs: bool, in_hubs: bool):
    """Uniform arcs, of which a quarter leave / reach the vertices 640 - 703."""
    rng = np.random.default_rng(5)
    u, v = rng.integers(0, N, M), rng.integers(0, N, M)
    if out_hubs:
        u[: M // 4] = rng.integers(640, 704, M // 4)
    if in_hubs:
        v[M // 8 : M // 8 + M // 4] = rng.integers(640, 704, M // 4)
    order = np.argsort(u, kind="stable")
    row = np.concatenate([[0], np.cumsum(np.bincount(u, minlength=N))]).astype(np.uint32)
    return gga.csr_from_arrays(row, v[order].astype(np.uint32), rng.integers(1, 101, M).astype(np.uint32))


@pytest.mark.parametrize("out_hubs,in_hubs,copy", [(False, False, 0), (True, False, 0), (False, True, 0), (True, True, 1)])
def test_copy_where_hubs_are_destinations_too(gpu, out_hubs, in_hubs, copy):
    with gga.DeviceGraph(graph(False, False)) as plain:
        base = plain.device_bytes
    g = graph(out_hubs, in_hubs)
    with gga.DeviceGraph(g) as dg:
        assert dg.device_bytes - base == copy * 4 * 131072
        dg.split(mda=64)
        for src in (3, 650):
            print(f"[gpu] out_hubs={out_hubs} in_hubs={in_hubs} src={src}", flush=True)
            np.testing.assert_array_equal(dg.sssp(src)[0], oracle.dijkstra(g.row_ptr, g.dst, g.w, src))
