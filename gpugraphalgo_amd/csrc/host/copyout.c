/*
 * copyout.c -- device results into the caller's host memory.
 *
 * A plain hipMemcpy into pageable memory reaches about 18 GB/s into pages that
 * are there, and half that into a fresh allocation whose pages the kernel has
 * to zero first; the link carries 57 GB/s into pinned memory.  A result
 * therefore goes through pinned slots: the link fills them while a few threads
 * empty them into the caller's array (and take its page faults).  A fill costs
 * about 20 us to start, so slots are large: 64 MiB of levels took 4.1 / 3.2 /
 * 2.8 ms through slots of 512 KiB / 1 / 2 MiB, 7.2 ms without (kernel
 * included); three to fourteen threads are within 5% of each other.
 *
 * Pinning memory takes milliseconds, so slot sets are kept for the next copy of
 * any handle: at most KEPT idle sets per device (pinned memory belongs to the
 * device it was made for), given back when the last handle goes.
 * Each copy holds a set of its own, so copies of different threads, handles
 * and streams do not meet.  The threads live for one copy.
 */
#define _GNU_SOURCE
#include <pthread.h>
#include <sched.h>
#include <stdatomic.h>
#include <stdlib.h>
#include <string.h>

#include "../gga_kernels.h"
#include "gga_host.h"

#define SLOT (4u << 20)             /* bytes per slot */
#define SLOTS 4u
#define UNIT (512u << 10)           /* bytes a thread moves at once */
#define FILL_MIN (2u << 20)         /* bytes per fill of results below SLOTS * SLOT */
#define THREADS 4u                  /* at most, beside the calling thread */
#define PARALLEL (3ull << 20)       /* bytes from which threads are worth their start (~0.1 ms) */
#define KEPT 2u                     /* idle sets kept per device */
#define DEVICES 64                  /* devices with sets; copies of further ones go without */

typedef struct slot_set {
    int device;
    uint8_t *pin;
    hipEvent_t ev[SLOTS];           /* a slot's fill has ended */
} slot_set;

static pthread_mutex_t mu = PTHREAD_MUTEX_INITIALIZER;
static slot_set *idle[DEVICES][KEPT];
static uint64_t users;              /* live handles */

static void set_free(slot_set *t)
{
    if (!t) return;
    if (t->pin) hipHostFree(t->pin);
    for (uint32_t i = 0; i < SLOTS; i++)
        if (t->ev[i]) hipEventDestroy(t->ev[i]);
    free(t);
}

void gga_copy_retain(void)
{
    pthread_mutex_lock(&mu);
    users++;
    pthread_mutex_unlock(&mu);
}

void gga_copy_release(void)
{
    slot_set *gone[DEVICES][KEPT];
    pthread_mutex_lock(&mu);
    const int last = --users == 0;
    if (last) {
        memcpy(gone, idle, sizeof gone);
        memset(idle, 0, sizeof idle);
    }
    pthread_mutex_unlock(&mu);
    for (uint32_t i = 0; last && i < DEVICES * KEPT; i++) set_free(gone[i / KEPT][i % KEPT]);
}

/* A set for `device` (current): an idle one, or a new one; NULL: no memory (or no such sets). */
static slot_set *set_take(int device)
{
    slot_set *t = NULL;
    if (device < 0 || device >= DEVICES) return NULL;
    pthread_mutex_lock(&mu);
    for (uint32_t i = 0; i < KEPT && !t; i++) {
        t = idle[device][i];
        idle[device][i] = NULL;
    }
    pthread_mutex_unlock(&mu);
    if (t) return t;
    t = (slot_set *)calloc(1, sizeof *t);
    if (!t) return NULL;
    t->device = device;
    hipError_t e = hipHostMalloc((void **)&t->pin, (uint64_t)SLOTS * SLOT, hipHostMallocDefault);
    if (e != hipSuccess) t->pin = NULL;
    for (uint32_t i = 0; i < SLOTS && e == hipSuccess; i++)
        if ((e = hipEventCreateWithFlags(&t->ev[i], hipEventDisableTiming)) != hipSuccess) t->ev[i] = NULL;
    if (e == hipSuccess) return t;
    (void)hipGetLastError();
    set_free(t);
    return NULL;
}

static void set_give(slot_set *t)
{
    pthread_mutex_lock(&mu);
    for (uint32_t i = 0; i < KEPT && t && users; i++)
        if (!idle[t->device][i]) {
            idle[t->device][i] = t;
            t = NULL;
        }
    pthread_mutex_unlock(&mu);
    set_free(t);
}

typedef struct copy_job {
    slot_set *t;
    uint8_t *dst;
    uint64_t bytes;
    uint32_t fill, fills, units;                  /* bytes per fill; fills; units of all of them */
    atomic_uint filled, next, emptied[SLOTS];     /* fills started, next unit, units moved per slot */
    atomic_int stop;                              /* a call failed */
} copy_job;

static void move_unit(copy_job *j, uint32_t u)
{
    const uint64_t at = (uint64_t)u * UNIT, left = j->bytes - at;
    const uint32_t k = (uint32_t)(at / j->fill), slot = k % SLOTS;
    memcpy(j->dst + at, j->t->pin + (uint64_t)slot * SLOT + at % j->fill, left < UNIT ? left : UNIT);
    atomic_fetch_add(&j->emptied[slot], 1u);
}

/* Moves units as their fills end until none is left. */
static void *drain(void *arg)
{
    copy_job *j = (copy_job *)arg;
    if (hipSetDevice(j->t->device) != hipSuccess) atomic_store(&j->stop, 1);
    for (;;) {
        const uint32_t u = atomic_fetch_add(&j->next, 1u);
        if (u >= j->units) return NULL;
        const uint32_t k = (uint32_t)((uint64_t)u * UNIT / j->fill);
        while (!atomic_load(&j->stop) && atomic_load(&j->filled) <= k) sched_yield();
        if (atomic_load(&j->stop)) return NULL;
        if (hipEventSynchronize(j->t->ev[k % SLOTS]) != hipSuccess) {
            atomic_store(&j->stop, 1);
            return NULL;
        }
        move_unit(j, u);
    }
}

hipError_t gga_copy_out(int device, hipStream_t s, void *dst, const void *src, uint64_t bytes)
{
    if (bytes == 0) return hipSuccess;
    /* memory the runtime knows (pinned by the caller, managed, ...) needs no slots */
    hipPointerAttribute_t pa;
    hipError_t e = hipPointerGetAttributes(&pa, dst);
    const int known = e == hipSuccess && pa.type != hipMemoryTypeUnregistered;
    if (e != hipSuccess) (void)hipGetLastError();
    slot_set *t = known ? NULL : set_take(device);
    if (!t) {
        e = hipMemcpyAsync(dst, src, bytes, known ? hipMemcpyDefault : hipMemcpyDeviceToHost, s);
        return e == hipSuccess ? hipStreamSynchronize(s) : e;
    }
    if (bytes <= FILL_MIN) {   /* one fill: nothing to overlap */
        e = hipMemcpyAsync(t->pin, src, bytes, hipMemcpyDeviceToHost, s);
        const hipError_t es = hipStreamSynchronize(s);
        if (e == hipSuccess) e = es;
        if (e == hipSuccess) memcpy(dst, t->pin, bytes);
        set_give(t);
        return e;
    }
    copy_job j;
    memset(&j, 0, sizeof j);
    j.t = t;
    j.dst = (uint8_t *)dst;
    j.bytes = bytes;
    j.fill = bytes < (uint64_t)SLOTS * SLOT ? FILL_MIN : SLOT;
    j.fills = (uint32_t)((bytes + j.fill - 1) / j.fill);
    j.units = (uint32_t)((bytes + UNIT - 1) / UNIT);
    pthread_t th[THREADS];
    uint32_t nth = 0;
    e = hipSuccess;
    if (bytes >= PARALLEL)
        while (nth < THREADS && pthread_create(&th[nth], NULL, drain, &j) == 0) nth++;
    const uint32_t per = j.fill / UNIT;   /* units of a full slot */
    for (uint32_t k = 0; k < j.fills && e == hipSuccess; k++) {
        const uint32_t i = k % SLOTS;
        /* the slot's last fill has to be moved out first; without threads (or
         * behind them) this thread moves units meanwhile */
        while (atomic_load(&j.emptied[i]) < k / SLOTS * per && !atomic_load(&j.stop)) {
            if (nth) {
                sched_yield();
                continue;
            }
            const uint32_t u = atomic_fetch_add(&j.next, 1u);
            if ((e = hipEventSynchronize(t->ev[u / per % SLOTS])) != hipSuccess) break;
            move_unit(&j, u);
        }
        if (atomic_load(&j.stop) && e == hipSuccess) e = hipErrorUnknown;
        const uint64_t at = (uint64_t)k * j.fill, left = bytes - at;
        if (e == hipSuccess)
            e = hipMemcpyAsync(t->pin + (uint64_t)i * SLOT, (const uint8_t *)src + at, left < j.fill ? left : j.fill,
                               hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipEventRecord(t->ev[i], s);
        if (e == hipSuccess) atomic_store(&j.filled, k + 1u);
    }
    if (e != hipSuccess) atomic_store(&j.stop, 1);
    else drain(&j);
    for (uint32_t i = 0; i < nth; i++) pthread_join(th[i], NULL);
    if (e == hipSuccess && atomic_load(&j.stop)) e = hipErrorUnknown;
    if (e != hipSuccess) hipStreamSynchronize(s);   /* nothing of this copy is left in flight */
    set_give(t);
    return e;
}

hipError_t gga_copy_out2(int device, hipStream_t s, void *dst0, const void *src0, uint64_t bytes0, void *dst1,
                         const void *src1, uint64_t bytes1)
{
    slot_set *t = bytes0 && bytes1 && bytes0 + bytes1 <= FILL_MIN ? set_take(device) : NULL;
    if (!t) {
        const hipError_t e = gga_copy_out(device, s, dst0, src0, bytes0);
        return e == hipSuccess ? gga_copy_out(device, s, dst1, src1, bytes1) : e;
    }
    hipError_t e = hipMemcpyAsync(t->pin, src0, bytes0, hipMemcpyDeviceToHost, s);
    if (e == hipSuccess) e = hipMemcpyAsync(t->pin + bytes0, src1, bytes1, hipMemcpyDeviceToHost, s);
    const hipError_t es = hipStreamSynchronize(s);
    if (e == hipSuccess) e = es;
    if (e == hipSuccess) {
        memcpy(dst0, t->pin, bytes0);
        memcpy(dst1, t->pin + bytes0, bytes1);
    }
    set_give(t);
    return e;
}
