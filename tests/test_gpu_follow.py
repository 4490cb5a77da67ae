"""Graphs whose degrees are a mesh's but whose fronts grow with every hop: a
wave must not run ahead along them.

Uniform random graphs, where following every vertex that a wave lowers made a
BFS inspect 2.8 edges for each of the graph's and following next to none 2.2;
2.4 lies between.  Results against the oracle, on trees and random graphs of
several degrees, both queries, both list forms, and engine lanes likewise."""
import numpy as np
import pytest

import gpugraphalgo_amd as gga
import oracle

pytestmark = pytest.mark.gpu


def uniform(n: int, m: int, seed: int):
    rng = np.random.default_rng(seed)
    u = np.sort(rng.integers(0, n, m))
    row = np.concatenate([[0], np.cumsum(np.bincount(u, minlength=n))]).astype(np.uint32)
    return gga.csr_from_arrays(row, rng.integers(0, n, m).astype(np.uint32), rng.integers(1, 101, m).astype(np.uint32))


def tree(n: int):
    """Binary, both arc directions."""
    child = np.arange(1, n)
    u, v = np.concatenate([(child - 1) // 2, child]), np.concatenate([child, (child - 1) // 2])
    order = np.argsort(u, kind="stable")
    row = np.concatenate([[0], np.cumsum(np.bincount(u, minlength=n))]).astype(np.uint32)
    w = np.random.default_rng(n).integers(1, 101, u.size).astype(np.uint32)
    return gga.csr_from_arrays(row, v[order].astype(np.uint32), w)


def test_a_growing_front_is_not_followed(gpu):
    g = uniform(200000, 16 * 200000, 1)
    with gga.DeviceGraph(g) as dg:
        dg.split()
        for src in (0, 66666):
            st = dg.bfs(src, mode="worklist", count=True, keep_on_device=True)[1]
            print(f"[gpu] src={src} edges inspected / m = {st['edges_inspected'] / g.m:.2f}", flush=True)
            assert st["edges_inspected"] <= 2.4 * g.m


@pytest.mark.parametrize("make", [lambda: uniform(20001, 30001, 2), lambda: uniform(50000, 300000, 3),
                                  lambda: uniform(30000, 480000, 4), lambda: tree(65535)])
def test_results(gpu, make):
    g = make()
    ones = np.ones(g.m, dtype=np.uint32)
    deg = g.degrees()
    srcs = [int(s) for s in np.flatnonzero(deg > 0)[[0, 7, -1]]]
    with gga.DeviceGraph(g) as dg:
        dg.split()
        for src in srcs:
            want = {b: oracle.dijkstra(g.row_ptr, g.dst, ones if b else g.w, src) for b in (True, False)}
            for kw in ({}, {"mode": "persistent"}, {"mode": "worklist", "dense_min": 1},
                       {"mode": "worklist", "dense_min": 0xFFFFFFFF}, {"mode": "worklist", "block": 512},
                       {"mode": "worklist", "count": True}):
                print(f"[gpu] n={g.n} m={g.m} src={src} {kw}", flush=True)
                np.testing.assert_array_equal(dg.bfs(src, **kw)[0], want[True])
                np.testing.assert_array_equal(dg.sssp(src, **kw)[0], want[False])


def test_engine_lanes_stop_too(gpu):
    """Eight BFS lanes of one engine: 1.8 edges inspected for each of the
    graph's and lane with a short queue, 2.5 following all; 2.15 lies between."""
    g = uniform(200000, 16 * 200000, 1)
    srcs = [i * g.n // 8 for i in range(8)]
    with gga.DeviceGraph(g) as dg:
        dg.split()
        for layout in (1, 2):
            out, st = dg.multi_sp(srcs, bfs_lanes=0xFF, count=True, ms_layout=layout)
            print(f"[gpu] layout={layout} edges / 8 m = {st['edges_inspected'] / (8 * g.m):.2f}", flush=True)
            assert st["edges_inspected"] <= 2.15 * 8 * g.m
            np.testing.assert_array_equal(out[3], oracle.bfs_queue(g.row_ptr, g.dst, srcs[3]))


@pytest.mark.parametrize("make", [lambda: uniform(20001, 30001, 2), lambda: uniform(30000, 480000, 4),
                                  lambda: tree(65535)])
def test_engine_results(gpu, make):
    g = make()
    ones = np.ones(g.m, dtype=np.uint32)
    srcs = [int(s) for s in np.flatnonzero(g.degrees() > 0)[:: g.n // 20][:9]]
    want = [oracle.dijkstra(g.row_ptr, g.dst, ones if 0x0F >> i & 1 else g.w, s) for i, s in enumerate(srcs)]
    with gga.DeviceGraph(g) as dg:
        dg.split()
        for kw in ({}, {"ms_layout": 1}, {"use_graph": 1}, {"mode": "persistent"}, {"dense_min": 1}):
            print(f"[gpu] n={g.n} m={g.m} {kw}", flush=True)
            out = dg.multi_sp(srcs, bfs_lanes=0x0F, **kw)[0]
            for i in range(len(srcs)):
                np.testing.assert_array_equal(out[i], want[i], err_msg=f"lane {i}")
