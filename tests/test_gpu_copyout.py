"""Results copied to host memory: sizes around the area that a query's last
kernel fills (1 MiB), the units (512 KiB), fills (2 and 4 MiB) and slots (16 MiB)
of the copy and the size where threads start (3 MiB); unaligned and pinned
destinations, rows that are or are not adjacent in the caller's memory, and two
threads copying at once."""
import ctypes

import numpy as np
import pytest

import gpugraphalgo_amd as gga
from gpugraphalgo_amd import _lib

pytestmark = pytest.mark.gpu


def star(n: int):
    """0 points to every other vertex; vertex 1 points to vertex 0."""
    row = np.full(n + 1, n, dtype=np.uint32)
    row[0], row[1] = 0, n - 1
    return gga.csr_from_arrays(row, np.concatenate([np.arange(1, n), [0]]).astype(np.uint32))


SLOT = 1 << 18   # vertices per MiB


@pytest.mark.parametrize("n", [2, 65, SLOT // 2 + 1, SLOT - 1, SLOT, SLOT + 1, 2 * SLOT, 3 * SLOT - 1, 3 * SLOT + 5,
                               8 * SLOT + 1, 16 * SLOT - 1, 16 * SLOT, 16 * SLOT + 1, 37 * SLOT + 77])
def test_distances_and_chunks(gpu, n):
    g = star(n)
    want = {0: np.full(n, 1, dtype=np.uint32), 1: np.full(n, 2, dtype=np.uint32)}
    want[0][0] = 0
    want[1][:2] = 1, 0
    L = _lib.load()
    with gga.DeviceGraph(g) as dg:
        dg.split(mda=1 << 20)
        for src in (0, 1, 0):
            print(f"[gpu] n={n} src={src}", flush=True)
            np.testing.assert_array_equal(dg.bfs(src)[0], want[src])
            np.testing.assert_array_equal(dg.sssp(src, mode="persistent")[0], want[src])
            np.testing.assert_array_equal(dg.copy_dist(), want[src])
            raw = np.zeros(4 * n + 64, dtype=np.uint8)          # 3 bytes off any alignment
            _lib.check(L.gga_graph_copy_dist(dg._h, raw.ctypes.data + 35), "copy_dist")
            np.testing.assert_array_equal(raw[35:35 + 4 * n].view(np.uint8), want[src].view(np.uint8))
            assert not raw[:35].any() and not raw[35 + 4 * n:].any()
        cb, own = dg.chunks()
        assert cb[0] == 0 and cb[-1] == g.m and np.array_equal(np.unique(own), np.arange(n))
        lev, _ = dg.multi_bfs([0, 1, 0])
        np.testing.assert_array_equal(lev, [want[0], want[1], want[0]])


def test_pinned_destination_and_lane_rows(gpu):
    hip = ctypes.CDLL("libamdhip64.so")
    n = 300007
    g = star(n)
    want = np.full(n, 1, dtype=np.uint32)
    want[0] = 0
    L = _lib.load()
    with gga.DeviceGraph(g) as dg:
        dg.split(mda=64)
        dg.bfs(0, keep_on_device=True)
        p = ctypes.c_void_p()
        assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(4 * n), ctypes.c_uint(0)) == 0
        try:
            _lib.check(L.gga_graph_copy_dist(dg._h, p), "copy_dist")
            got = np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_uint32)), shape=(n,)).copy()
        finally:
            hip.hipHostFree(p)
        np.testing.assert_array_equal(got, want)
        got, _ = dg.multi_sp([0] * 32, bfs_lanes=0xFFFFFFFF)     # adjacent rows
        assert (got == want).all()
        with gga.MultiSourceEngine(dg) as eng:                    # rows apart
            eng.start({i: 0 for i in (0, 1, 5, 31)}, bfs={0, 1, 5, 31})
            assert eng.run() == 0
            for row in eng.fetch([0, 1, 5, 31]).values():
                np.testing.assert_array_equal(row, want)


def test_two_threads(gpu):
    import threading
    sizes = [5 * SLOT + 3, 17 * SLOT + 9]
    wrong = []

    def work(n):
        g = star(n)
        with gga.DeviceGraph(g) as dg:
            dg.split(mda=1 << 20)
            for i in range(4):
                d = dg.bfs(i % 2)[0]
                if d[0] != i % 2 or not (d[2:] == 1 + i % 2).all():
                    wrong.append((n, i))

    threads = [threading.Thread(target=work, args=(n,)) for n in sizes]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
