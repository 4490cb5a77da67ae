"""copyout.c against a stand-in for the HIP runtime: host memory copies, counted
allocations, an event that has happened once it is recorded.

How many sets of pinned slots a process makes and keeps over several devices,
sizes and threads, that all are given back, and that bytes arrive whole."""
import ctypes
import os
import subprocess
import threading

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "gpugraphalgo_amd", "csrc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")

STANDIN = r"""
#define _GNU_SOURCE
#include <hip/hip_runtime_api.h>
#include <stdatomic.h>
#include <stdlib.h>
#include <string.h>
#undef hipPointerGetAttributes
atomic_int made, freed, events;
hipError_t hipHostMalloc(void **p, size_t n, unsigned f) { (void)f; *p = malloc(n); atomic_fetch_add(&made, 1); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); atomic_fetch_add(&freed, 1); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned f) { (void)f; *e = (hipEvent_t)malloc(1); atomic_fetch_add(&events, 1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); atomic_fetch_sub(&events, 1); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { (void)e; (void)s; return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { (void)e; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; return hipSuccess; }
hipError_t hipSetDevice(int d) { (void)d; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t t)
{ (void)k; (void)t; memcpy(d, s, n); return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{ (void)p; memset(a, 0, sizeof *a); a->type = hipMemoryTypeUnregistered; return hipSuccess; }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("copyout")
    (d / "standin.c").write_text(STANDIN)
    so = str(d / "copyout.so")
    subprocess.run(["gcc", "-O2", "-std=gnu11", "-fPIC", "-shared", "-pthread", "-D__HIP_PLATFORM_AMD__", "-I",
                    os.path.join(ROCM, "include"), "-Wl,-Bsymbolic", "-o", so, str(d / "standin.c"),
                    os.path.join(CSRC, "host", "copyout.c")], check=True)
    return ctypes.CDLL(so)


def copy(lib, device, words, seed=0):
    src = np.random.default_rng(seed + words).integers(0, 1 << 32, words, dtype=np.uint64).astype(np.uint32)
    dst = np.zeros(words, dtype=np.uint32)
    assert lib.gga_copy_out(device, None, ctypes.c_void_p(dst.ctypes.data), ctypes.c_void_p(src.ctypes.data),
                            ctypes.c_uint64(4 * words)) == 0
    np.testing.assert_array_equal(dst, src)


def counts(lib):
    return [ctypes.c_int.in_dll(lib, k).value for k in ("made", "freed", "events")]


def test_each_device_keeps_its_sets(lib):
    """Copies in turn on eight devices pin one set a device, once."""
    made, freed, _ = counts(lib)
    lib.gga_copy_retain()
    for rep in range(4):
        for device in range(8):
            copy(lib, device, 300000 + device, rep)
    assert counts(lib)[0] - made == 8 and counts(lib)[1] == freed
    lib.gga_copy_release()
    assert counts(lib)[1] - freed == 8 and counts(lib)[2] == 0


def test_sizes_and_threads(lib):
    """Around a unit, a fill, the slots; several threads a device."""
    made, freed, _ = counts(lib)
    lib.gga_copy_retain()
    for words in (1, 131072, 524288, 524289, 786433, 4194303, 4194305, 9000001):
        copy(lib, 0, words)
    failed = []

    def work(i):
        try:
            for k in range(6):
                copy(lib, i % 3, 600001 + 1000 * i, k)
        except Exception as e:   # noqa: BLE001 (reported below)
            failed.append(e)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(9)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failed
    m, f, _ = counts(lib)
    assert (m - made) - (f - freed) <= 2 * 3       # at most two idle sets a device
    lib.gga_copy_release()
    m, f, ev = counts(lib)
    assert m - made == f - freed and ev == 0


def test_a_device_without_sets(lib):
    made = counts(lib)[0]
    lib.gga_copy_retain()
    copy(lib, 1000, 700000)
    lib.gga_copy_release()
    assert counts(lib)[0] == made
