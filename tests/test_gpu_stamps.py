"""Flag steps past 256: a stamp of one step must not list its vertex again in
a later one (byte stamps that lived on would, and a query whose every step is a
flag step would never end).  Long graphs that are not mesh-like, wide enough
that the default list switch takes flag steps throughout."""
import numpy as np
import pytest

import gpugraphalgo_amd as gga
import oracle

pytestmark = pytest.mark.gpu


def wide_ladder(rows: int, cols: int, leaves: int, seed: int):
    """A directed rows x cols grid (right and down arcs), the corner pointing to `leaves` extra vertices."""
    n = rows * cols
    i = np.arange(n)
    right, down = i[i % cols != cols - 1], i[i < n - cols]
    u = np.concatenate([right, down, np.zeros(leaves, dtype=np.int64)])
    v = np.concatenate([right + 1, down + cols, n + np.arange(leaves)])
    order = np.argsort(u * (n + leaves) + v)
    row = np.concatenate([[0], np.cumsum(np.bincount(u, minlength=n + leaves))]).astype(np.uint32)
    w = np.random.default_rng(seed).integers(1, 4, u.size)
    return gga.csr_from_arrays(row, v[order].astype(np.uint32), w)


@pytest.mark.parametrize("rows,cols,leaves", [(1, 700, 40), (3, 600, 40), (700, 900, 60)])
@pytest.mark.parametrize("mode", ["worklist", "persistent"])
def test_no_stamp_outlives_its_step(gpu, rows, cols, leaves, mode):
    g = wide_ladder(rows, cols, leaves, seed=rows)
    want = oracle.dijkstra(g.row_ptr, g.dst, g.w, 0)
    with gga.DeviceGraph(g) as dg:
        dg.split(mda=16)
        for kw in ({}, {"dense_min": 1}, {"dense_min": 1, "count": True}, {"dense_min": 1, "delta": 30}):
            print(f"[gpu] {rows}x{cols} {mode} {kw}", flush=True)
            got, st = dg.sssp(0, mode=mode, **kw)
            np.testing.assert_array_equal(got, want)
            np.testing.assert_array_equal(dg.bfs(0, mode=mode, **kw)[0],
                                          oracle.dijkstra(g.row_ptr, g.dst, np.ones(g.m, dtype=np.uint32), 0))
