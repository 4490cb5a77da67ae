// relax.hip -- BFS/SSSP edge relaxation over split chunks, for gfx950.
//
// Replaces M_my_drelax (cudaKernels.h:285-344) and its host fixpoint loop
// (bfs_sssp.cu:372-468), my_drelax_no_atomic + my_updateDist
// (cudaKernels.h:129-220) and the dynamic-parallelism child grids
// (my_drelax_dynamicP / dynamicP_relax_coal, cudaKernels.h:347-377,438-521).
//
// Work unit: a wave takes a batch of up to 64 chunk ids (one per lane), reads
// each chunk's bounds and its owner's distance, and walks the concatenation of
// the batch's edge ranges 64 * UNROLL slots per round (wave_owner).  A chunk
// holds at most T edges, so a hub vertex is spread over many chunks and many
// waves; this is the node split.  Chunks of one vertex are adjacent in the
// worklist and in memory, so col[]/w[] loads of a round are contiguous runs.
// Batches are dealt round-robin to the waves of the grid (no shared counter);
// the batch size shrinks with the frontier so that a small frontier still
// spreads over every wave.
//
// Relax (all modes): alt = dist[u] + w (skipped when it would wrap or reach
// inf); a plain read of dist[v] guards the atomicMin (cudaKernels.h:324-325).
// Distances only decrease, so a stale read is never lower than the truth and
// the guard cannot lose an update.  The owner's distance is read when the
// chunk is expanded, so an update made earlier in the same step is used.
//
// Next frontier, chosen per step from the size of the current one:
//   queue step (small frontier): atomicMin with return; a vertex whose
//     distance dropped is queued once per step (step stamp in mark[], taken
//     with an exchange; BFS needs none since a level-synchronous atomicMin
//     succeeds once per vertex).  Queued vertices are staged in wave-private
//     LDS and flushed as chunk ids with one atomicAdd per 64 vertices.
//   flag step (large frontier): fire-and-forget atomicMin and a plain store of
//     a stamp into flag[v] (a byte array: a quarter of mark[]'s lines); then
//     two compaction passes (count per tile, write from the counts before the
//     tile) rebuild the list from flag[] with no shared counter and take each
//     stamp back as its vertex is listed.
// A level-synchronous BFS flag step needs no atomic: the byte is the guard and
// a level is a plain store.  An uninstrumented worklist query is one launch
// per phase (relax, count, write, refill; k_wl_phase), and a small graph's
// whole query one workgroup (k_small).
// Device-scope atomics on MI355X execute past the per-XCD L2 and atomics on
// one address serialize (~16 ns each), so no hot path funnels through a single
// counter: batch assignment is static, work counters are striped, list
// allocation in flag steps is a scan, and the grid barrier is two-level.
//
// Bytes per unit of work (the roofline model): per edge inspected
// col 4 + w 4 (SSSP) + dist[v] 4; per chunk expanded cbeg 4 + cown 4 +
// dist[u] 4 (+ 4 for the worklist id); per relaxation 4 + 4 (queue / stamp).
#include "../gga_kernels.h"
#include "wave.hpp"
#include "sync.hpp"
#include "compact.hpp"

#include <mutex>

using namespace gga;

// Workspace of the allocation-free query (gga_sssp_noalloc): step stamps,
// flag bytes, the two chunk lists, compaction tiles, control words, work
// counters and the near-far arrays, carved by the host out of one static
// array.  Each device that runs the query holds its own copy from module
// load to process end.  Host code never names `scratch` in a kernel
// argument or a copy: it uses the device address ggak_scratch looks up.
static __device__ __align__(256) uint8_t scratch[GGA_SCRATCH_BYTES];

namespace {

constexpr uint32_t BLOCK = 256;
constexpr uint32_t WAVES = BLOCK / GGA_WAVE;
constexpr uint32_t PBUF = 256;          // queued vertices staged per wave before a flush
#ifndef GGA_UNROLL
#define GGA_UNROLL 4
#endif
constexpr uint32_t UNROLL = GGA_UNROLL; // edge slots per lane per round in expand_batch
#ifndef GGA_LVL_UNROLL
#define GGA_LVL_UNROLL 4
#endif
constexpr uint32_t LVL_UNROLL = GGA_LVL_UNROLL;   // the same in expand_level
// Meshes: vertices a wave may follow past its batch within one step (0: off),
// its LDS queue of them, 16-vertex groups expanded per round, and the largest
// degree followed.  SSSP on a pure 1024^2 grid / the 4096^2 grid with 0.5%
// shortcuts, ms: queue of 256, one group 6.43 / 6.94, two 6.14 / 7.18; queue
// of 512, one 6.45 / 6.40, two 6.23 / 6.33, four 6.34 / 6.34 (a short queue
// overflows into the list); following 256 / 512 / 1024 / 2048 (queue of 512,
// four groups): 6.94 / 6.38 / 6.34 / 6.80 and 6.55 / 6.42 / 6.34 / 6.92.
#ifndef GGA_CONT
#define GGA_CONT 1024
#endif
#ifndef GGA_CQ
#define GGA_CQ 512
#endif
#ifndef GGA_CONT_GROUPS
#define GGA_CONT_GROUPS 2
#endif
constexpr uint32_t CQ = GGA_CQ;
constexpr uint32_t CONT_DEG = 16;
// A wave stops following once more than CONT_FRONT vertices, plus a quarter of
// those it followed, wait in its queue.  A mesh front that one wave follows
// stays thin (its perimeter: some 45 of 256 followed on a grid); on a graph as
// even in its degrees but without locality -- uniform random edges, a tree --
// every round queues more than it follows, and the wave runs ahead of the
// others into vertices that they reach on shorter ways.  Uniform graphs, all
// 1024 followed -> stopped (and as it was with a queue of 128): BFS on 200 k
// vertices of degree 16 880 -> 281 us (750), 4 M of degree 4 1767 -> 833
// (1590), SSSP on 100 k of degree 6 989 -> 769 (900), on a binary tree of 1 M
// 597 -> 485 (560); grids within 2%.  64 + a quarter: 4096^2 grid with
// shortcuts BFS 5% slower than following nothing beyond its queue of 128; 384:
// uniform BFS 444, 4 M 954-1406.
constexpr uint32_t CONT_FRONT = 128;
// Only steps whose list is at most this many chunks follow: a thin wavefront
// leaves most of the chip idle and each step is a chain of dependent loads;
// a wide one (a mesh with shortcuts, past its first levels) already fills the
// chip, and following would only expand the same vertices twice (4096^2 grid
// + 0.5% shortcuts, BFS: 5.1 ms without, 8.4 ms following in every step).
constexpr uint32_t CONT_LIST = 65536;

enum { OUT_CHANGED = 0, OUT_QUEUE = 1, OUT_FLAG = 2 };

// Work counters of one wave: wave-uniform values, kept in scalar registers
// (32 bits: one wave's share of one step), added to the striped 64-bit
// counters once per wave at the end.
struct Counters {
    uint32_t edges = 0, chunks = 0, relax = 0;
};

// Whether waves follow their front (follow_front): not; without or with a
// guard read before the atomic; or as w.guard says (kernels that are not built
// once for each: the read's branch costs a mesh's SSSP 1%).
enum { FOLLOW_NONE, FOLLOW, FOLLOW_GUARD, FOLLOW_EITHER };

// A lane's chunk in a batch: its edge range [eb, ee) and owner.
struct ChunkDesc {
    uint32_t eb = 0, ee = 0, own = 0;
    bool valid = false;
};

// Edge arrays, lists and chunk descriptors are read with plain loads: a chunk's
// run and its neighbours' share lines, and a thin mesh front comes back to the
// same edges.  Against non-temporal loads: SSSP on R-MAT s22 2204 -> 2118 us,
// on 2^17 vertices 442 -> 412, 32 engine lanes on R-MAT s20 5634 -> 5500, on
// the 4096^2 grid 256 -> 246 ms.  The exception is a mesh batch's own edges,
// which the wide steps of a large mesh stream once (4096^2 grid + 0.5%
// shortcuts, SSSP: 6.86 ms non-temporal, 7.01 plain).
template <bool STREAM>
__device__ __forceinline__ uint32_t edge_load(const uint32_t *p) {
    return STREAM ? stream_load(p) : *p;
}

template <bool CONT, bool OWN = true>
__device__ __forceinline__ ChunkDesc load_chunk(const gga_dev_graph &g, uint32_t c, bool valid) {
    ChunkDesc d;
    d.valid = valid;
    if (valid) {
        d.eb = edge_load<CONT>(&g.cbeg[c]);
        d.ee = edge_load<CONT>(&g.cbeg[c + 1]);
        if (OWN) d.own = edge_load<CONT>(&g.cown[c]);
    }
    return d;
}

// Lists x for the next step where `want`: the step's flag byte, or (queue
// steps) the step stamp taken by exchange and a push.  PLAIN: every vertex
// comes once, no stamp needed.  Whole-wave call.
template <bool PLAIN, int OUT>
__device__ __forceinline__ void list_vertex(const gga_dev_graph &g, const gga_dev_work &w, bool want, uint32_t x,
                                            uint32_t it, uint32_t *pbuf, uint32_t &pcount, uint32_t *qout,
                                            uint32_t *tail) {
    if (OUT == OUT_FLAG) {
        if (want) w.flag[x] = 1;
    } else if (OUT == OUT_QUEUE) {
        if (!PLAIN && want) want = (w.mark[x] != it) && (atomic_xchg_u32(&w.mark[x], it) != it);
        const uint64_t mask = __ballot(want);
        if (mask) {
            const uint32_t nw = (uint32_t)__popcll(mask);
            if (pcount + nw > PBUF) {
                flush_pushes(g, pbuf, pcount, qout, tail, w.qcap, w.ctl);
                pcount = 0;
            }
            if (want)
                pbuf[pcount + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                                        __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u))] = x;
            pcount += nw;
            __builtin_amdgcn_wave_barrier();
        }
    }
}

// Queues (x, the distance this wave wrote there, its edge range) where `near`,
// as far as the queue [qh, qt) has room; true on the lanes queued.  Whole-wave
// call.
__device__ __forceinline__ bool queue_near(bool near, uint32_t x, uint32_t d, uint32_t r0, uint32_t r1, uint4 *cq,
                                           uint32_t qh, uint32_t &qt) {
    const uint64_t qm = __ballot(near);
    if (!qm) return false;
    const uint32_t rank = __builtin_amdgcn_mbcnt_hi((uint32_t)(qm >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)qm, 0u));
    const uint32_t room = CQ - (qt - qh), nnear = (uint32_t)__popcll(qm);
    const bool queued = near && rank < room;
    if (queued) cq[(qt + rank) % CQ] = make_uint4(x, d, r0, r1);
    qt += nnear < room ? nnear : room;
    return queued;
}

// Meshes: a wave follows its own front within the step.  Each round expands
// up to 64 vertices of the wave's queue -- vertices it lowered below the
// threshold, each from the distance it wrote there, all edges -- until the
// queue empties or GGA_CONT vertices were followed; what is then left, what
// found the queue full and what has more than CONT_DEG edges is listed for
// the next step.  So every improvement is either expanded at the distance
// written or listed, as in a plain step, and distances converge to the same
// fixed point.  A followed vertex records the distance it was expanded at
// (near-far), as a listed one does when the next step expands it.
//
// What bounds it: the chain of dependent accesses of a round.  A queue entry
// holds the vertex's edge range, fetched beside the atomic that lowered it,
// and four neighbouring lanes take a vertex's edges (four at a time), so a
// round needs no chunk lookup, scan or owner search; and with no guard read
// before the atomic it is two accesses, edge and atomic (it was chunk start,
// chunk bounds, edge, dist[v], atomic, behind a 6-shuffle search).  A thin
// front leaves the atomic units idle: without the guard SSSP on a pure 1024^2
// grid went from 4.70 to 4.08 ms, on a 100 x 77 grid from 0.47 to 0.40.  Where
// many arcs lead to a few neighbouring vertices it is read (w.guard: in_hubs()
// in host/graph.c has the sizes).  With the queue of 512, SSSP: pure 1024^2 grid 8.9 -> 6.2
// ms, a 100 x 77 grid 0.80 -> 0.60, 4096^2 with shortcuts 6.8 -> 6.3; BFS on
// the pure 1024^2 / 4096^2 grid 4.1-4.6 -> 2.9-3.2 / 19-25 -> 13-18 ms.
template <bool BFS, bool COUNT, int OUT, bool GUARD>
__device__ __forceinline__ void follow_front(const gga_dev_graph &g, const gga_dev_work &w, uint32_t it,
                                             uint32_t *pbuf, uint32_t &pcount, uint32_t *qout, uint32_t *tail,
                                             Counters &cnt, uint32_t thr, uint4 *cq, uint32_t qt) {
    constexpr uint32_t PER = GGA_WAVE / 4u, G = GGA_CONT_GROUPS;   // vertices per group, groups per round
    const uint32_t l = lane_id(), sub = l & 3u;
    uint32_t *__restrict__ dist = w.dist;
    const uint32_t inf = w.inf;
    uint32_t qh = 0, budget = (uint32_t)GGA_CONT;
    while (qh != qt) {
        __builtin_amdgcn_wave_barrier();
        const uint32_t avail = qt - qh;
        // (avail > CONT_FRONT + followed / 4: a growing front)
        if (4u * avail + budget > 4u * CONT_FRONT + (uint32_t)GGA_CONT) budget = 0u;
        // budget spent, or too little room for what a round may queue: the
        // oldest entries are listed
        const bool drain = budget == 0u || CQ - avail < GGA_WAVE * G;
        uint32_t take = drain ? GGA_WAVE : PER * G;
        take = take < avail ? take : avail;
        take = drain || take < budget ? take : budget;
        {
            const uint4 q = cq[(qh + l) % CQ];
            const bool mine = l < take, hub = q.w - q.z > CONT_DEG;
            list_vertex<false, OUT>(g, w, mine && (drain || hub), q.x, it, pbuf, pcount, qout, tail);
            if (w.last && mine && !drain && !hub) w.last[q.x] = q.y;
            if (COUNT && !drain) {
                cnt.edges += wave_last(wave_incl_scan(mine && !hub ? q.w - q.z : 0u));
                cnt.chunks += __builtin_amdgcn_readfirstlane((uint32_t)__popcll(__ballot(mine && !hub && q.w != q.z)));
            }
        }
        const uint32_t head = qh;
        qh += take;
        if (drain) continue;
        budget -= take;
        uint32_t eb[G], n[G], du[G], most = 0;
#pragma unroll
        for (uint32_t u = 0; u < G; u++) {
            const uint32_t i = u * PER + (l >> 2);
            const uint4 q = cq[(head + i) % CQ];
            du[u] = q.y;
            eb[u] = q.z;
            n[u] = i < take && q.w - q.z <= CONT_DEG ? q.w - q.z : 0u;
            most = n[u] > most ? n[u] : most;
        }
        __builtin_amdgcn_wave_barrier();   // the entries are read before the pushes below write the queue
        for (uint32_t j = sub;; j += 4u) {
            uint32_t v[G], alt[G], cur[G], r0[G], r1[G];
            bool act[G];
#pragma unroll
            for (uint32_t u = 0; u < G; u++) {
                if (u * PER >= take) break;
                act[u] = j < n[u];
                const uint32_t e = act[u] ? eb[u] + j : 0u;   // (the graph has an edge: slot 0 is in bounds)
                v[u] = g.col[e];
                alt[u] = du[u] + (BFS ? 1u : g.w[e]);
            }
            if (GUARD) {
                uint32_t d[G];
#pragma unroll
                for (uint32_t u = 0; u < G; u++) d[u] = u * PER < take ? dist[v[u]] : 0u;
#pragma unroll
                for (uint32_t u = 0; u < G; u++) act[u] = act[u] && alt[u] < d[u];
            }
#pragma unroll
            for (uint32_t u = 0; u < G; u++) {
                if (u * PER >= take) break;
                act[u] = act[u] && alt[u] >= du[u] && alt[u] < inf;
                if (act[u]) {
                    cur[u] = atomic_min_u32(&dist[v[u]], alt[u]);
                    r0[u] = g.row[v[u]];
                    r1[u] = g.row[v[u] + 1u];
                }
            }
#pragma unroll
            for (uint32_t u = 0; u < G; u++) {
                if (u * PER >= take) break;
                const bool imp = act[u] && alt[u] < cur[u];
                if (COUNT) cnt.relax += __builtin_amdgcn_readfirstlane((uint32_t)__popcll(__ballot(imp)));
                const bool queued = queue_near(imp && alt[u] < thr, v[u], alt[u], r0[u], r1[u], cq, qh, qt);
                (void)queued;
            }
            if (__ballot(j + 4u < most) == 0ull) break;
            // a vertex of more than four edges: room for the next four
            while (CQ - (qt - qh) < GGA_WAVE * G) {
                __builtin_amdgcn_wave_barrier();
                const uint32_t x = cq[(qh + l) % CQ].x;
                list_vertex<false, OUT>(g, w, l < qt - qh, x, it, pbuf, pcount, qout, tail);
                qh += qt - qh < GGA_WAVE ? qt - qh : GGA_WAVE;
            }
        }
    }
}

// Expand one batch of chunks (this lane's chunk d when d.valid).
// thr (near-far): a destination whose new distance is >= thr is lowered but
// not listed -- it is deferred until the threshold passes it, and w.last
// (when set) records the distance each owner was expanded at, so that a
// deferred vertex is recognised by dist < last.  thr = 0xFFFFFFFF: plain
// worklist (every improvement is listed).
//
// CONT (meshes), cq given (a short list), list steps: the vertices that the
// batch lowers below the threshold go to the wave's queue instead of the list,
// and follow_front expands them within the step.  (BFS then takes the step
// stamp too: levels reached out of order can drop twice.)
//
// SPREAD (SSSP on graphs whose hubs are neighbours, w.sdist set): atomics run at
// 26 G/s over distinct memory channels on MI355X, but at 3.8 (2^17 vertices)
// to 7 G/s (2^22) where they fall as R-MAT destinations do, because the hubs'
// words share a few 256-byte granules.  They go to a permuted copy of the
// distances instead, sdist, which decides; dist, in vertex order, whose
// gathers profit from the same neighbourhood, stays the guard.  Whoever lowers
// sdist (the atomic's result says so, in flag steps too) stores its distance
// to dist; racing stores may leave dist above sdist, never below, and each of
// them lists its vertex, whose next expansion starts from sdist and brings
// dist up to date.  So when no list is left, dist equals sdist.  SSSP, three
// sources each, without / with: R-MAT 2^16 320 / 280 / 274 -> 268 / 224 / 232
// us, 2^17 (T = 992) 396 / 349 / 433 -> 347 / 307 / 381, 2^20 781 / 950 / 740
// -> 667 / 787 / 626, 2^21 1098 / 1204 / 1494 -> 1070 / 1144 / 1414; 2^22 2090
// -> 2186 (the copy falls out of the caches there: see skewed() for the rule).
// Stores and stamps by everyone who passes the guard, no result awaited, left
// dist loose enough to expand a quarter more edges (2^22: 2650 us).
template <bool BFS, bool COUNT, int OUT, int CONT = FOLLOW_NONE, bool SPREAD = false>
__device__ __forceinline__ void expand_batch(const gga_dev_graph &g, const gga_dev_work &w,
                                             const ChunkDesc &d, uint32_t it, uint32_t *pbuf,
                                             uint32_t &pcount, uint32_t *qout, uint32_t *tail,
                                             bool &improved, Counters &cnt, uint2 *tab, uint32_t nown,
                                             uint32_t thr = 0xFFFFFFFFu, uint4 *cq = nullptr) {
    const uint32_t l = lane_id();
    uint32_t *__restrict__ dist = w.dist;
    const uint32_t inf = w.inf;
    uint32_t eb = 0, n = 0, du = inf;
    if (d.valid) {
        eb = d.eb;
        const uint32_t ee = d.ee;
        const uint32_t own = d.own;
        du = SPREAD ? w.sdist[gga_spread(own, w.smask)] : dist[own];
        // SSSP: an owner already lowered and listed again during this step is
        // expanded in the next one with its newer distance, which relaxes
        // every edge at least as far -- expanding it now would only repeat
        // that work, so its chunks are left to the next step.
        bool again = false;
        if (!BFS && OUT == OUT_FLAG) again = w.flag[own] != 0;
        if (!BFS && OUT == OUT_QUEUE) again = w.mark[own] == it;
        // Near-far: only an owner below the threshold is expanded (every
        // vertex listed by a stamp or a refill is).  Expanding a deferred one
        // could go wrong: a concurrent improvement of it would be >= thr,
        // deferred rather than stamped, and found later only through dist <
        // last -- but with several chunks reading different distances, the
        // chunk that saw the newer one may write last[] after the others,
        // leaving dist == last while edges expanded with the older distance
        // are never relaxed again.
        const bool go = du < inf && !again && du < thr;
        n = go ? ee - eb : 0u;
        if (!SPREAD && w.last && go) w.last[own] = du;
        if (SPREAD && go) dist[own] = du;
    }
    constexpr bool cont = CONT != FOLLOW_NONE && OUT != OUT_CHANGED;
    uint32_t qt = 0;   // vertices queued (wave-uniform)
    const uint32_t incl = wave_incl_scan(n);
    const uint32_t total = wave_last(incl);
    if (COUNT) {
        cnt.edges += __builtin_amdgcn_readfirstlane(total);
        cnt.chunks += __builtin_amdgcn_readfirstlane((uint32_t)__popcll(__ballot(n > 0)));
    }
    const uint32_t excl = incl - n;
    // the wave's owner table (LDS): slot k of owner j reads edge
    // (eb_j - excl_j) + k from distance du_j -- one LDS load per slot
    // instead of two more shuffles
    tab[l] = make_uint2(eb - excl, du);
    __builtin_amdgcn_wave_barrier();
    // owners are lanes 0 .. nown - 1: the search starts at half the next
    // power of two of them (wave-uniform)
    const uint32_t half = nown <= 1u ? 0u : 1u << (31 - __builtin_clz(nown - 1u));
    // UNROLL groups of 64 slots per round.  Within a group, slots past the end
    // are clamped to the last slot, so every load below has an in-bounds
    // address and all gathers of a lane are issued before the first result is
    // used; a group wholly past the end is skipped (total and left are
    // scalars, so the skips are scalar branches) -- a small batch, e.g. one
    // chunk of a dozen edges, runs one group, not UNROLL.
    for (uint32_t base = 0; base < total; base += GGA_WAVE * UNROLL) {
        uint32_t e[UNROLL], ds[UNROLL], v[UNROLL], wt[UNROLL], cur[UNROLL], kk[UNROLL], own[UNROLL];
        uint32_t r0[UNROLL] = {}, r1[UNROLL] = {};
        bool act[UNROLL];
        const uint32_t left = total - base;   // > 0
#pragma unroll
        for (uint32_t u = 0; u < UNROLL; u++) {
            const uint32_t k = base + u * GGA_WAVE + l;
            act[u] = k < total;
            kk[u] = act[u] ? k : total - 1;
            own[u] = 0;
        }
        // slot k's owner: the first lane whose inclusive prefix exceeds k
        // (binary search, one shuffle per halving; the groups' shuffles are
        // independent and issued together, skipped groups included)
        for (uint32_t step = half; step != 0; step >>= 1) {
#pragma unroll
            for (uint32_t u = 0; u < UNROLL; u++) {
                const uint32_t y = __shfl(incl, (int)(own[u] + step - 1), GGA_WAVE);
                own[u] += y <= kk[u] ? step : 0u;
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < UNROLL; u++) {
            if (u * GGA_WAVE >= left) break;
            const uint2 t = tab[own[u]];
            e[u] = t.x + kk[u];
            ds[u] = t.y;
        }
#pragma unroll
        for (uint32_t u = 0; u < UNROLL; u++) {
            if (u * GGA_WAVE >= left) break;
            v[u] = edge_load<CONT != FOLLOW_NONE>(&g.col[e[u]]);
            wt[u] = BFS ? 1u : edge_load<CONT != FOLLOW_NONE>(&g.w[e[u]]);
        }
#pragma unroll
        for (uint32_t u = 0; u < UNROLL; u++) {
            if (u * GGA_WAVE >= left) break;
            cur[u] = dist[v[u]];
        }
#pragma unroll
        for (uint32_t u = 0; u < UNROLL; u++) {
            if (u * GGA_WAVE >= left) break;
            bool imp = false;
            const uint32_t alt = ds[u] + wt[u];
            if (act[u] && alt >= ds[u] && alt < inf && alt < cur[u]) {
                if (cont && cq) {   // the queue's row offsets, on their way beside the atomic
                    r0[u] = g.row[v[u]];
                    r1[u] = g.row[v[u] + 1u];
                }
                uint32_t *const at = SPREAD ? &w.sdist[gga_spread(v[u], w.smask)] : &dist[v[u]];
                if (OUT == OUT_FLAG && !SPREAD) {
                    (void)atomic_min_u32(at, alt);  // result unused: no-return atomic
                    imp = true;
                } else {
                    const uint32_t old = atomic_min_u32(at, alt);
                    imp = alt < old;
                }
                if (SPREAD && imp) dist[v[u]] = alt;
            }
            if (COUNT) cnt.relax += __builtin_amdgcn_readfirstlane((uint32_t)__popcll(__ballot(imp)));
            if (OUT == OUT_CHANGED) {
                improved |= imp;
                continue;
            }
            const bool near = imp && alt < thr;
            bool queued = false;
            if (cont && cq) queued = queue_near(near, v[u], alt, r0[u], r1[u], cq, 0u, qt);
            list_vertex<BFS && !cont, OUT>(g, w, near && !queued, v[u], it, pbuf, pcount, qout, tail);
        }
    }
    if (cont && cq && qt != 0u) {
        if (CONT == FOLLOW_GUARD || (CONT == FOLLOW_EITHER && w.guard))
            follow_front<BFS, COUNT, OUT, true>(g, w, it, pbuf, pcount, qout, tail, cnt, thr, cq, qt);
        else
            follow_front<BFS, COUNT, OUT, false>(g, w, it, pbuf, pcount, qout, tail, cnt, thr, cq, qt);
    }
}

// Expand one batch of a level-synchronous BFS step (w.lvl): every listed
// chunk's owner was reached in the step before, so its distance is the step's
// level and is not read, and whatever a step reaches gets the same value,
// `alt`.  The guard is therefore the byte flag[v] (0: not reached) instead of
// dist[v] -- n bytes, which an XCD's 4 MB L2 holds where 4 n are gathered past
// it -- and a flag step needs no atomic: racing (or stale) guards store the
// same byte, and the compaction gives the stamped vertices their distance.  A
// queue step takes the vertex with atomicMin's result, which is inf for
// exactly one of the racers, and stamps it for later guards.
//
// What bounds it: the gathers, at the rate the L1s take misses (R-MAT s22,
// the widest level: 45 M edges in 0.34 ms).  Against guarding with dist[v] and
// a device-scope atomicMin per improvement: BFS on R-MAT s22 (T = 128) 878 ->
// 727 us a query, on a 1.5 M-vertex R-MAT graph, ef 8, 450 -> 380 us on the
// device.  A bitmap of the reached vertices in front of the bytes (hot words
// in L1) gained 15% in the widest level and lost more in the one before,
// where half the edges find an unset bit and read the byte as well.
template <bool COUNT, int OUT>
__device__ __forceinline__ void expand_level(const gga_dev_graph &g, const gga_dev_work &w, const ChunkDesc &d,
                                             uint32_t alt, uint8_t stamp, uint32_t *pbuf, uint32_t &pcount,
                                             uint32_t *qout, uint32_t *tail, Counters &cnt, uint32_t *tab,
                                             uint32_t nown) {
    const uint32_t l = lane_id();
    uint8_t *__restrict__ flag = w.flag;
    const uint32_t n = d.valid ? d.ee - d.eb : 0u;
    const uint32_t incl = wave_incl_scan(n);
    const uint32_t total = wave_last(incl);
    if (COUNT) {
        cnt.edges += __builtin_amdgcn_readfirstlane(total);
        cnt.chunks += __builtin_amdgcn_readfirstlane((uint32_t)__popcll(__ballot(n > 0)));
    }
    tab[l] = d.eb - (incl - n);   // slot k of owner j is edge tab[j] + k (see expand_batch)
    __builtin_amdgcn_wave_barrier();
    const uint32_t half = nown <= 1u ? 0u : 1u << (31 - __builtin_clz(nown - 1u));
    for (uint32_t base = 0; base < total; base += GGA_WAVE * LVL_UNROLL) {
        uint32_t v[LVL_UNROLL], kk[LVL_UNROLL], own[LVL_UNROLL], seen[LVL_UNROLL];
        const uint32_t left = total - base;
#pragma unroll
        for (uint32_t u = 0; u < LVL_UNROLL; u++) {
            const uint32_t k = base + u * GGA_WAVE + l;
            kk[u] = k < total ? k : total - 1u;
            own[u] = 0;
        }
        for (uint32_t step = half; step != 0; step >>= 1) {
#pragma unroll
            for (uint32_t u = 0; u < LVL_UNROLL; u++) {
                const uint32_t y = __shfl(incl, (int)(own[u] + step - 1), GGA_WAVE);
                own[u] += y <= kk[u] ? step : 0u;
            }
        }
#pragma unroll
        for (uint32_t u = 0; u < LVL_UNROLL; u++) {
            if (u * GGA_WAVE >= left) break;
            v[u] = g.col[tab[own[u]] + kk[u]];
        }
#pragma unroll
        for (uint32_t u = 0; u < LVL_UNROLL; u++) {
            if (u * GGA_WAVE >= left) break;
            seen[u] = flag[v[u]];
        }
#pragma unroll
        for (uint32_t u = 0; u < LVL_UNROLL; u++) {
            if (u * GGA_WAVE >= left) break;
            bool imp = base + u * GGA_WAVE + l < total && seen[u] == 0u && alt < w.inf;
            if (OUT == OUT_FLAG) {
                if (imp) flag[v[u]] = stamp;
            } else {
                if (imp) imp = alt < atomic_min_u32(&w.dist[v[u]], alt);
                if (imp) flag[v[u]] = stamp;
                const uint64_t mask = __ballot(imp);
                if (mask) {
                    const uint32_t nw = (uint32_t)__popcll(mask);
                    if (pcount + nw > PBUF) {
                        flush_pushes(g, pbuf, pcount, qout, tail, w.qcap, w.ctl);
                        pcount = 0;
                    }
                    if (imp)
                        pbuf[pcount + __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                                                __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u))] = v[u];
                    pcount += nw;
                    __builtin_amdgcn_wave_barrier();
                }
            }
            if (COUNT) cnt.relax += __builtin_amdgcn_readfirstlane((uint32_t)__popcll(__ballot(imp)));
        }
    }
    __builtin_amdgcn_wave_barrier();   // the table is read before the next batch writes it
}

// Work counters: lane 0 of each wave adds to one of GGA_CNT_SLOTS striped slots.
template <bool COUNT>
__device__ __forceinline__ void publish_counters(const gga_dev_work &w, const Counters &c) {
    if (COUNT && lane_id() == 0) {
        const uint32_t slot = (blockIdx.x * (blockDim.x / GGA_WAVE) + threadIdx.x / GGA_WAVE) % GGA_CNT_SLOTS;
        uint64_t *s = w.cnt + 4u * slot;
        if (c.edges) atomic_add_u64(&s[0], c.edges);
        if (c.chunks) atomic_add_u64(&s[1], c.chunks);
        if (c.relax) atomic_add_u64(&s[2], c.relax);
    }
}

// ---------------------------------------------------------------- init
__global__ __launch_bounds__(BLOCK) void k_fill(uint32_t *p, uint32_t value, uint64_t count) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < count;
         i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = value;
}

// dist = inf except dist[src] = 0 (bfs_sssp.cu:302-318, with the source as an
// argument instead of the hard-coded parent 0); worklist = chunks of src;
// ring slot 0 = {len, step epoch}; counters and barrier zeroed.
__global__ __launch_bounds__(BLOCK) void k_query_init(gga_dev_graph g, gga_dev_work w, uint32_t src,
                                                      uint32_t epoch) {
    const uint64_t t0 = wall_clock64();   // the query's start, before the fills
    const uint64_t tid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    const uint64_t nth = (uint64_t)gridDim.x * blockDim.x;
    for (uint64_t v = tid; v < g.n; v += nth) w.dist[v] = (v == src) ? 0u : w.inf;
    for (uint64_t v = tid; v < g.n; v += nth)
        w.flag[v] = w.lvl && v == src ? 255u : 0u;
    if (w.last)
        for (uint64_t v = tid; v < g.n; v += nth) w.last[v] = w.inf;
    if (w.sdist)
        for (uint64_t i = tid; i <= w.smask; i += nth) w.sdist[i] = i == gga_spread(src, w.smask) ? 0u : w.inf;
    for (uint64_t i = tid; i < 4ull * GGA_CNT_SLOTS; i += nth) w.cnt[i] = 0;
    if (blockIdx.x == 0) {
        const uint32_t cs = g.cstart[src], nch = g.cstart[src + 1] - cs;
        for (uint32_t i = threadIdx.x; i < nch; i += blockDim.x) w.q0[i] = cs + i;
        if (threadIdx.x < 3) {
            w.ctl[GGA_CTL_TAIL(threadIdx.x)] = threadIdx.x == 0 ? nch : 0u;
            w.ctl[GGA_CTL_ITER(threadIdx.x)] = epoch;
            // near-far: the first bucket is [0, delta); plain worklist: no bound
            w.ctl[GGA_CTL_THR(threadIdx.x)] = w.last ? (w.delta < w.inf ? w.delta : w.inf) : 0xFFFFFFFFu;
        }
        if (threadIdx.x == 0) {
            w.ctl[GGA_CTL_FAR] = 0;
            for (uint32_t i = 0; i < 3; i++) {
                w.ctl[GGA_CTL_PHASE(i)] = GGA_PH_START;
                w.ctl[GGA_CTL_PSTEP(i)] = 0;
                w.ctl[GGA_CTL_PLEN(i)] = 0;
                w.ctl[GGA_CTL_LISTED(i)] = 0;
            }
            w.ctl[GGA_CTL_PHASES] = 0;
            *reinterpret_cast<uint64_t *>(w.ctl + GGA_CTL_T0) = t0;
            w.ctl[GGA_CTL_RSTEP] = epoch - 1u;   // no refill yet (step numbers start at epoch)
        }
        if (threadIdx.x < GGA_BAR_GROUPS) w.ctl[GGA_CTL_BARG(threadIdx.x)] = 0;
        if (threadIdx.x == 0) {
            w.ctl[GGA_CTL_CHANGED] = 0;
            w.ctl[GGA_CTL_STEPS] = 0;
            w.ctl[GGA_CTL_ERR] = 0;
            w.ctl[GGA_CTL_BAR] = 0;
        }
        if (threadIdx.x < 6) w.ctl[GGA_CTL_CNT + threadIdx.x] = 0;
        if (threadIdx.x < 8) w.ctl[GGA_CTL_RED + threadIdx.x] = 0;
    }
}

// ------------------------------------------------------ topology step
// Every chunk, every step: the reference's M_my_drelax schedule with chunks in
// place of split nodes (chunks of unreached owners contribute no edges).
template <bool BFS, bool COUNT>
__global__ __launch_bounds__(BLOCK) void k_topo_step(gga_dev_graph g, gga_dev_work w) {
    const uint32_t lb = xcd_block(blockIdx.x, gridDim.x);
    const uint64_t c = ((uint64_t)lb * WAVES + threadIdx.x / GGA_WAVE) * GGA_WAVE + lane_id();
    const bool valid = c < g.C;
    bool improved = false;
    uint32_t pcount = 0;
    Counters cnt;
    __shared__ uint2 s_tab[WAVES][GGA_WAVE];
    expand_batch<BFS, COUNT, OUT_CHANGED>(g, w, load_chunk<false>(g, valid ? (uint32_t)c : 0u, valid), 0u, nullptr,
                                          pcount, nullptr, nullptr, improved, cnt,
                                          s_tab[__builtin_amdgcn_readfirstlane(threadIdx.x / GGA_WAVE)], GGA_WAVE);
    if (__ballot(improved) && lane_id() == 0) w.ctl[GGA_CTL_CHANGED] = 1u;  // *changed = true
    publish_counters<COUNT>(w, cnt);
}

// ------------------------------------------------------ worklist step
// Level-synchronous BFS (w.lvl): the byte that marks a vertex reached at
// `level` >= 1; never 0 (not reached), repeating every 254 levels (255: the source).
__device__ __forceinline__ uint8_t level_stamp(uint32_t level) { return (uint8_t)(1u + (level - 1u) % 254u); }

__device__ __forceinline__ bool flag_step(const gga_dev_work &w, uint32_t nq) {
    return nq >= w.dense_min;
}

// One step = expand the list of ring slot (step % 3), fill slot (step + 1) % 3.
template <bool BFS, bool COUNT, int CONT, bool SPREAD = false>
__device__ __forceinline__ void worklist_step(const gga_dev_graph &g, const gga_dev_work &w,
                                              uint32_t step, uint32_t nq, uint32_t it,
                                              uint32_t *pbuf, uint4 *cq, uint2 *tab, Counters &cnt) {
    const uint32_t sout = (step + 1u) % 3u;
    const uint32_t *qin = (step & 1u) ? w.q1 : w.q0;
    uint32_t *qout = (step & 1u) ? w.q0 : w.q1;
    uint32_t *tail = &w.ctl[GGA_CTL_TAIL(sout)];
    // batches of bsz chunks dealt round-robin, at most 64 chunks each.
    // Ragged chunks (bmin 1): ~16 batches per wave when the list is long
    // enough, for balance; small batches also expand more chunks late in the
    // step, when more of their owners have been re-listed and can be left to
    // the next step (R-MAT s22 SSSP, batches per wave 4 / 8 / 16 / 32: 2.33 /
    // 2.17 / 2.14 / 2.26 ms).  Uniform small chunks (meshes, bmin > 1): few
    // large batches -- every batch is a chain of dependent loads -- with one
    // batch per 1/1024 of the list, but at least bmin chunks (2: each wave
    // then follows its own wavefront, see expand_batch).
    // Level-synchronous BFS has nothing to leave to the next step and takes 8
    // batches per wave (R-MAT s22, 4 / 8 / 16 / 32: 773 / 739 / 755 / 802 us)
    constexpr bool LVL = BFS && !CONT;
    const uint32_t wpb = blockDim.x / GGA_WAVE;   // waves per workgroup (128, 256 or 512 threads)
    const uint32_t waves = gridDim.x * wpb;
    uint32_t bsz = w.bmin > 1u ? nq >> 10 : nq / ((LVL ? 8u : 16u) * waves);
    bsz = bsz < w.bmin ? w.bmin : bsz;
    bsz = bsz < 1u ? 1u : (bsz > GGA_WAVE ? GGA_WAVE : bsz);
    const uint32_t nbatch = (nq + bsz - 1) / bsz;
    const uint32_t wid = blockIdx.x * wpb + __builtin_amdgcn_readfirstlane(threadIdx.x / GGA_WAVE);
    const bool flags = flag_step(w, nq);
    const uint32_t l = lane_id();
    const uint32_t thr = w.ctl[GGA_CTL_THR(step % 3u)];
    uint32_t pcount = 0;
    bool dummy = false;
    const uint32_t alt = it - w.epoch + 1u;   // LVL: the level this step reaches
    const uint8_t stamp = level_stamp(alt);
    uint4 *const follow = (CONT && nq <= CONT_LIST) ? cq : nullptr;   // the continuation's queue
    // Software pipeline over the wave's batches b, b + waves, b + 2 waves...:
    // while a batch is expanded, the next batch's chunk descriptors and the
    // list entries of the one after it are already in flight, so a batch
    // starts at its owners' distances instead of two dependent loads
    // earlier.  The list and the chunk table do not change during a step.
    auto entry = [&](uint64_t bb, bool &ok) -> uint32_t {
        const uint64_t idx = bb * bsz + l;
        ok = bb < nbatch && l < bsz && idx < nq;
        return ok ? edge_load<CONT != FOLLOW_NONE>(&qin[idx]) : 0u;
    };
    bool ok_next;
    uint32_t c_next;
    ChunkDesc cur;
    {
        bool ok0;
        const uint32_t c0 = entry(wid, ok0);
        c_next = entry((uint64_t)wid + waves, ok_next);
        cur = load_chunk<CONT != FOLLOW_NONE, !LVL>(g, c0, ok0);
    }
    for (uint64_t b = wid; b < nbatch; b += waves) {
        bool ok_after;
        const uint32_t c_after = entry(b + 2ull * waves, ok_after);
        const ChunkDesc nxt = load_chunk<CONT != FOLLOW_NONE, !LVL>(g, c_next, ok_next);
        if (LVL && flags)
            expand_level<COUNT, OUT_FLAG>(g, w, cur, alt, stamp, pbuf, pcount, qout, tail, cnt,
                                          reinterpret_cast<uint32_t *>(tab), bsz);
        else if (LVL)
            expand_level<COUNT, OUT_QUEUE>(g, w, cur, alt, stamp, pbuf, pcount, qout, tail, cnt,
                                           reinterpret_cast<uint32_t *>(tab), bsz);
        else if (flags)
            expand_batch<BFS, COUNT, OUT_FLAG, CONT, SPREAD>(g, w, cur, it, pbuf, pcount, qout, tail, dummy, cnt, tab, bsz,
                                                     thr, follow);
        else
            expand_batch<BFS, COUNT, OUT_QUEUE, CONT, SPREAD>(g, w, cur, it, pbuf, pcount, qout, tail, dummy, cnt, tab, bsz,
                                                      thr, follow);
        cur = nxt;
        c_next = c_after;
        ok_next = ok_after;
    }
    if (pcount) flush_pushes(g, pbuf, pcount, qout, tail, w.qcap, w.ctl);
}

// A vertex belongs to the next list when the current (flag) step stamped it
// (a non-zero byte).  One byte per vertex, so the two passes over the stamps
// read n bytes, not 4n; the write pass (CLEAR) takes the stamps back, each
// cleared by the thread that lists its vertex, so that no later step meets
// them.
template <bool CLEAR>
struct StampMarked {
    uint8_t *flag;
    static constexpr bool vec8 = true;
    __device__ __forceinline__ bool operator()(uint32_t v) const {
        const bool m = flag[v] != 0;
        if (CLEAR && m) flag[v] = 0;
        return m;
    }
    // bit i: vertex v + i is stamped (v a multiple of 8)
    __device__ __forceinline__ uint32_t mark8(uint64_t v) const {
        const uint2 x = *reinterpret_cast<const uint2 *>(flag + v);
        uint32_t m = 0;
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) {
            m |= ((x.x >> (8u * i)) & 0xFFu) != 0u ? 1u << i : 0u;
            m |= ((x.y >> (8u * i)) & 0xFFu) != 0u ? 1u << (4u + i) : 0u;
        }
        if (CLEAR && m) *reinterpret_cast<uint2 *>(flag + v) = make_uint2(0u, 0u);
        return m;
    }
};

// Level-synchronous BFS: the vertices a flag step stamped get their distance
// here (write pass), each written by the thread that lists it.  From the
// level on at which stamps repeat, a stamped vertex is new only while its
// distance is still inf (the count pass sees it so too: it writes nothing).
template <bool WRITE>
struct LevelMarked {
    const uint8_t *flag;
    uint32_t *dist;
    uint32_t level, inf;
    uint8_t stamp;
    static constexpr bool vec8 = true;
    __device__ __forceinline__ bool operator()(uint32_t v) const {
        if (flag[v] != stamp || (level > 254u && dist[v] != inf)) return false;
        if (WRITE) dist[v] = level;
        return true;
    }
    __device__ __forceinline__ uint32_t mark8(uint64_t v) const {
        const uint2 x = *reinterpret_cast<const uint2 *>(flag + v);
        uint32_t m = 0;
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) {
            m |= ((x.x >> (8u * i)) & 0xFFu) == stamp ? 1u << i : 0u;
            m |= ((x.y >> (8u * i)) & 0xFFu) == stamp ? 1u << (4u + i) : 0u;
        }
        if (level > 254u) {
#pragma unroll
            for (uint32_t i = 0; i < 8; i++)
                if (((m >> i) & 1u) && dist[v + i] != inf) m &= ~(1u << i);
        }
        if (WRITE) {
#pragma unroll
            for (uint32_t i = 0; i < 8; i++)
                if ((m >> i) & 1u) dist[v + i] = level;
        }
        return m;
    }
};
template <bool WRITE>
__device__ __forceinline__ LevelMarked<WRITE> level_marked(const gga_dev_work &w, uint32_t it) {
    const uint32_t level = it - w.epoch + 1u;
    return LevelMarked<WRITE>{w.flag, w.dist, level, w.inf, level_stamp(level)};
}

// The single list of the plain layout for step `step`.
__device__ __forceinline__ ListOut list_out(const gga_dev_graph &g, const gga_dev_work &w, uint32_t step) {
    ListOut o;
    o.cstart = g.C == g.n ? nullptr : g.cstart;   // every vertex has a chunk
    o.q = (step & 1u) ? w.q0 : w.q1;
    o.qcap = w.qcap;
    o.tiles = w.tiles;
    o.tail = &w.ctl[GGA_CTL_TAIL((step + 1u) % 3u)];
    o.ctl = w.ctl;
    return o;
}

// Per-step bookkeeping done by one thread: next slot's step number, clear the
// slot consumed one step ago (it becomes the output slot of the next step).
__device__ __forceinline__ void step_bookkeeping(uint32_t *ctl, uint32_t step, uint32_t it,
                                                 uint32_t nq) {
    const uint32_t sout = (step + 1u) % 3u, sclr = (step + 2u) % 3u;
    ctl[GGA_CTL_ITER(sout)] = it + 1u;
    ctl[GGA_CTL_THR(sout)] = ctl[GGA_CTL_THR(step % 3u)];
    ctl[GGA_CTL_TAIL(sclr)] = 0u;
    ctl[GGA_CTL_LISTED(sout)] = 0u;
    if (nq) ctl[GGA_CTL_STEPS] += 1u;
}

__device__ __forceinline__ uint32_t step_len(const gga_dev_work &w, uint32_t step) {
    const uint32_t t = w.ctl[GGA_CTL_TAIL(step % 3u)];
    return t < w.qcap ? t : w.qcap;  // > qcap only with QFULL set
}

// Placement of the running wave: XCC id << 8 | SE / SH / CU bits of HW_ID.
__device__ __forceinline__ uint32_t hw_place() {
    uint32_t hw, xcc;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_HW_ID)" : "=s"(hw));
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(xcc));
    return ((xcc & 0xFu) << 8) | ((hw >> 8) & 0xFFu);
}

// TL: instrumented variant (the reference's my_drelax_metric, cudaKernels.h:2-70,
// which stores each block's clock64 span): each workgroup writes its start,
// duration and placement to tl[blockIdx.x].  Every variant keeps eight waves
// per SIMD (at most 64 VGPRs; the counting variants would otherwise take 62-65
// and drop to seven): the relax is bound by the latency of its gathers.  (The
// mesh variants' queues, 8 KB of LDS per wave, leave room for four.)
// BS: workgroup size, 128, 256 or 512 threads (the tuner times all three).
template <bool BFS, bool COUNT, bool TL, uint32_t BS, bool CONT, bool SPREAD>
__global__ __launch_bounds__(BS) __attribute__((amdgpu_waves_per_eu(CONT ? 4 : 8, 8)))
void k_wl_step(gga_dev_graph g, gga_dev_work w, uint32_t step, gga_wg_record *tl) {
    __shared__ uint32_t s_pbuf[BS / GGA_WAVE][PBUF];
    __shared__ uint4 s_cq[CONT ? BS / GGA_WAVE : 1][CONT ? CQ : 1];
    __shared__ uint2 s_tab[BS / GGA_WAVE][GGA_WAVE];
    uint64_t t0 = 0;
    if (TL && threadIdx.x == 0) t0 = wall_clock64();
    const uint32_t nq = step_len(w, step);
    const uint32_t it = w.ctl[GGA_CTL_ITER(step % 3u)];
    if (blockIdx.x == 0 && threadIdx.x == 0) step_bookkeeping(w.ctl, step, it, nq);
    if (nq != 0) {
        Counters cnt;
        const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x / GGA_WAVE);
        worklist_step<BFS, COUNT, CONT ? FOLLOW_EITHER : FOLLOW_NONE, SPREAD>(g, w, step, nq, it, s_pbuf[wv], s_cq[CONT ? wv : 0], s_tab[wv], cnt);
        publish_counters<COUNT>(w, cnt);
    }
    if (TL) {
        __syncthreads();
        if (threadIdx.x == 0) {
            gga_wg_record r;
            r.start = t0;
            r.ticks = (uint32_t)(wall_clock64() - t0);
            r.place = hw_place();
            tl[blockIdx.x] = r;
        }
    }
}

// The compaction passes run after k_wl_step(step): count, then write (which
// also sums the counts before each tile, and with near-far buckets starts
// the refill when the list came out empty, below); both are no-ops after a
// queue step.  A count workgroup that finds stamped vertices marks the slot
// LISTED (plain stores of the same value), so that the write pass knows
// whether the list is empty without summing every count.
template <bool LVL>
__global__ __launch_bounds__(BLOCK) void k_compact_count(gga_dev_graph g, gga_dev_work w, uint32_t step) {
    __shared__ uint32_t s_wave[WAVES];
    const uint32_t nq = step_len(w, step);
    if (nq == 0 || !flag_step(w, nq)) return;
    const ListOut o = list_out(g, w, step);
    const uint32_t it = w.ctl[GGA_CTL_ITER(step % 3u)];
    uint32_t any = 0;
    for (uint32_t t = blockIdx.x; t < GGA_TILES(g.n); t += gridDim.x)
        any |= LVL ? compact_count_tile(o, g.n, t, level_marked<false>(w, it), s_wave)
                   : compact_count_tile(o, g.n, t, StampMarked<false>{w.flag}, s_wave);
    if (any && threadIdx.x == 0) w.ctl[GGA_CTL_LISTED((step + 1u) % 3u)] = 1u;
}

// ---- near-far refill: after a step whose next list came out empty, list
// the deferred vertices (dist < last) under the next threshold.
// The count pass stamps what it counts (flag[], all clear when a list is
// empty), so that the write pass reads n bytes instead of dist and last again.
__device__ __forceinline__ uint32_t stamps4(uint32_t bits) {   // byte i = bit i
    return (bits & 1u) | (bits & 2u) << 7 | (bits & 4u) << 14 | (bits & 8u) << 21;
}
struct DeferredUnder {
    const uint32_t *dist, *last;
    uint32_t t;
    uint32_t *mn;    // the smallest deferred distance seen (under t or not)
    uint8_t *flag;   // gets the stamps
    static constexpr bool vec8 = true;
    __device__ __forceinline__ bool operator()(uint32_t v) const {
        const uint32_t d = dist[v];
        const bool deferred = d < last[v];
        if (deferred && d < *mn) *mn = d;
        if (deferred && d < t) flag[v] = 1;
        return deferred && d < t;
    }
    // bit i: vertex v + i is deferred under t (v a multiple of 8); dist may
    // be a caller's buffer (the allocation-free query), so 16-byte loads
    // only when it is 16-byte aligned (last always is)
    __device__ __forceinline__ uint32_t mark8(uint64_t v) const {
        uint32_t m = 0;
        if ((reinterpret_cast<uintptr_t>(dist) & 15u) == 0) {
            const uint4 d0 = *reinterpret_cast<const uint4 *>(dist + v);
            const uint4 d1 = *reinterpret_cast<const uint4 *>(dist + v + 4);
            const uint4 l0 = *reinterpret_cast<const uint4 *>(last + v);
            const uint4 l1 = *reinterpret_cast<const uint4 *>(last + v + 4);
            const uint32_t d[8] = {d0.x, d0.y, d0.z, d0.w, d1.x, d1.y, d1.z, d1.w};
            const uint32_t s[8] = {l0.x, l0.y, l0.z, l0.w, l1.x, l1.y, l1.z, l1.w};
            uint32_t lo = 0xFFFFFFFFu;
#pragma unroll
            for (uint32_t i = 0; i < 8; i++) {
                m |= (d[i] < s[i] && d[i] < t) ? 1u << i : 0u;
                lo = d[i] < s[i] && d[i] < lo ? d[i] : lo;
            }
            if (lo < *mn) *mn = lo;
            if (m) *reinterpret_cast<uint2 *>(flag + v) = make_uint2(stamps4(m), stamps4(m >> 4));
        } else {
#pragma unroll
            for (uint32_t i = 0; i < 8; i++) m |= (*this)((uint32_t)(v + i)) ? 1u << i : 0u;
        }
        return m;
    }
};

__device__ __forceinline__ uint32_t sat_add(uint32_t a, uint32_t b) {
    const uint32_t s = a + b;
    return s < a ? 0xFFFFFFFFu : s;
}

// count: chunk ids per tile under thr + delta, and the tile's smallest deferred distance
__device__ __forceinline__ void refill_count_body(const gga_dev_graph &g, const gga_dev_work &w, uint32_t step,
                                                  uint32_t *s_wave, uint32_t *s_min) {
    const ListOut o = list_out(g, w, step);
    uint32_t m = 0xFFFFFFFFu;   // the thread's smallest deferred distance, gathered by the count
    const DeferredUnder pred{w.dist, w.last, sat_add(w.ctl[GGA_CTL_THR((step + 1u) % 3u)], w.delta), &m, w.flag};
    for (uint32_t t = blockIdx.x; t < GGA_TILES(g.n); t += gridDim.x) {
        m = 0xFFFFFFFFu;
        compact_count_tile(o, g.n, t, pred, s_wave);
#pragma unroll
        for (uint32_t off = 32; off >= 1; off >>= 1) {
            const uint32_t y = __shfl_xor(m, (int)off, GGA_WAVE);
            m = y < m ? y : m;
        }
        if (lane_id() == 0) s_min[threadIdx.x / GGA_WAVE] = m;
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t x = s_min[0];
            for (uint32_t i = 1; i < WAVES; i++) x = s_min[i] < x ? s_min[i] : x;
            w.tmin[t] = x;
        }
        __syncthreads();
    }
}

// scan (one workgroup): offsets and list length; the threshold of the new
// list; when nothing lies under it but deferred vertices remain, the
// threshold jumps to the smallest deferred distance and FAR asks for another
// refill.
__device__ __forceinline__ void refill_scan_body(const gga_dev_graph &g, const gga_dev_work &w, uint32_t step,
                                                 uint32_t *s_wave, uint32_t *s_min) {
    const uint32_t sout = (step + 1u) % 3u;
    const uint32_t t1 = sat_add(w.ctl[GGA_CTL_THR(sout)], w.delta);
    const ListOut o = list_out(g, w, step);
    compact_scan(o, g.n, s_wave);
    uint32_t m = 0xFFFFFFFFu;
    for (uint32_t i = threadIdx.x; i < GGA_TILES(g.n); i += blockDim.x) m = w.tmin[i] < m ? w.tmin[i] : m;
#pragma unroll
    for (uint32_t off = 32; off >= 1; off >>= 1) {
        const uint32_t y = __shfl_xor(m, (int)off, GGA_WAVE);
        m = y < m ? y : m;
    }
    if (lane_id() == 0) s_min[threadIdx.x / GGA_WAVE] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        uint32_t gmin = s_min[0];
        for (uint32_t i = 1; i < WAVES; i++) gmin = s_min[i] < gmin ? s_min[i] : gmin;
        const uint32_t total = *o.tail;
        w.ctl[GGA_CTL_RTHR] = t1;
        if (total) {
            w.ctl[GGA_CTL_THR(sout)] = t1;
            w.ctl[GGA_CTL_FAR] = 0u;
            w.ctl[GGA_CTL_RSTEP] = w.ctl[GGA_CTL_ITER(step % 3u)];
        } else if (gmin != 0xFFFFFFFFu) {
            w.ctl[GGA_CTL_THR(sout)] = gmin;   // the next refill lists [gmin, gmin + delta)
            w.ctl[GGA_CTL_FAR] = 1u;
        } else {
            w.ctl[GGA_CTL_FAR] = 0u;           // nothing deferred: converged
        }
    }
    __syncthreads();
}

__device__ __forceinline__ void refill_write_body(const gga_dev_graph &g, const gga_dev_work &w, uint32_t step,
                                                  uint32_t *s_wave, uint32_t *stage) {
    const ListOut o = list_out(g, w, step);
    for (uint32_t t = blockIdx.x; t < GGA_TILES(g.n); t += gridDim.x)
        compact_write_tile(o, g.n, t, StampMarked<true>{w.flag}, s_wave, stage);
}

// The standalone refill is two launches: its count runs in the compaction's
// write launch (k_compact_write, whose first thread also records the
// threshold the refill lists under, RTHR, and that this step refills, RSTEP
// = its step number), then k_refill_write, which sums the counts before each
// tile itself (compact_write_tiles); its first workgroup folds the total and
// the tiles' minima into the next threshold as the scan body above does.
// That write reads only RTHR / RSTEP, which no workgroup of it changes, so
// the list length it stores midway does not change its course.
//
// In the compaction's write launch: after a flag
// step the list is empty exactly when no count workgroup marked it LISTED,
// after a queue step when no push reached it (its length, final since the
// relax ended); either way every workgroup reads the same words, which no
// workgroup of this launch changes.  (The refill's counts reuse tiles[],
// which the compaction reads only when the list is not empty.)  Its first
// thread records the threshold the refill lists under (RTHR) and that this
// step refills (RSTEP = its step number).
template <bool LVL>
__global__ __launch_bounds__(BLOCK) void k_compact_write(gga_dev_graph g, gga_dev_work w, uint32_t step) {
    __shared__ uint32_t s_wave[WAVES], s_min[WAVES], s_stage[CSTAGE];
    const uint32_t nq = step_len(w, step), sout = (step + 1u) % 3u;
    const bool flags = nq != 0 && flag_step(w, nq);
    if (flags) {
        if (!w.last || w.ctl[GGA_CTL_LISTED(sout)] != 0u) {
            const uint32_t it = w.ctl[GGA_CTL_ITER(step % 3u)];
            if (LVL) compact_write_tiles(list_out(g, w, step), g.n, level_marked<true>(w, it), s_wave, s_stage);
            else compact_write_tiles(list_out(g, w, step), g.n, StampMarked<true>{w.flag}, s_wave, s_stage);
            return;
        }
    } else if (!w.last || w.ctl[GGA_CTL_TAIL(sout)] != 0u) {
        return;
    }
    if (LVL) return;   // (BFS has no buckets)
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        w.ctl[GGA_CTL_RTHR] = sat_add(w.ctl[GGA_CTL_THR(sout)], w.delta);
        w.ctl[GGA_CTL_RSTEP] = w.ctl[GGA_CTL_ITER(step % 3u)];
    }
    refill_count_body(g, w, step, s_wave, s_min);
}

// (every workgroup of the grid calls this; s_min: one entry per wave)
__device__ __forceinline__ void refill_list_body(const gga_dev_graph &g, const gga_dev_work &w, uint32_t step,
                                                 uint32_t *s_wave, uint32_t *s_min, uint32_t *stage) {
    const uint32_t sout = (step + 1u) % 3u, t1 = w.ctl[GGA_CTL_RTHR];
    const ListOut o = list_out(g, w, step);
    if (blockIdx.x == 0) {
        // the new threshold: t1 when the refill lists anything, else a jump
        // to the smallest deferred distance (FAR: refill again), else done
        const uint32_t ntiles = GGA_TILES(g.n);
        uint32_t sum = 0, m = 0xFFFFFFFFu, ex;
        for (uint32_t i = threadIdx.x; i < ntiles; i += blockDim.x) {
            sum += o.tiles[i];
            m = w.tmin[i] < m ? w.tmin[i] : m;
        }
        const uint32_t total = block_excl_scan(sum, ex, s_wave);
#pragma unroll
        for (uint32_t off = 32; off >= 1; off >>= 1) {
            const uint32_t y = __shfl_xor(m, (int)off, GGA_WAVE);
            m = y < m ? y : m;
        }
        if (lane_id() == 0) s_min[threadIdx.x / GGA_WAVE] = m;
        __syncthreads();
        if (threadIdx.x == 0) {
            uint32_t gmin = s_min[0];
            for (uint32_t i = 1; i < WAVES; i++) gmin = s_min[i] < gmin ? s_min[i] : gmin;
            if (total) {
                w.ctl[GGA_CTL_THR(sout)] = t1;
                w.ctl[GGA_CTL_FAR] = 0u;
            } else if (gmin != 0xFFFFFFFFu) {
                w.ctl[GGA_CTL_THR(sout)] = gmin;   // the next refill lists [gmin, gmin + delta)
                w.ctl[GGA_CTL_FAR] = 1u;
            } else {
                w.ctl[GGA_CTL_FAR] = 0u;           // nothing deferred: converged
            }
        }
        __syncthreads();
    }
    compact_write_tiles(o, g.n, StampMarked<true>{w.flag}, s_wave, stage);
}

__global__ __launch_bounds__(BLOCK) void k_refill_write(gga_dev_graph g, gga_dev_work w, uint32_t step) {
    __shared__ uint32_t s_wave[WAVES], s_min[WAVES], s_stage[CSTAGE];
    if (!w.last) return;
    if (w.ctl[GGA_CTL_RSTEP] != w.ctl[GGA_CTL_ITER(step % 3u)]) return;  // no refill after this step
    refill_list_body(g, w, step, s_wave, s_min, s_stage);
}

// ------------------------------------------------------ one launch per phase
// A query's steps as a chain of launches of this kernel, each running the next
// phase (gga_next_phase).  The launches of a step as kernels of their own --
// relax, count, write, refill -- cost a kernel boundary (~4.5 us) and a host
// enqueue each whether the step needs them or not: a queue step needs one of
// the four.
template <bool BFS, int CONT, bool SPREAD>
__global__ __launch_bounds__(BLOCK) __attribute__((amdgpu_waves_per_eu(CONT ? 4 : 8, 8)))
void k_wl_phase(gga_dev_graph g, gga_dev_work w, uint32_t launch) {
    __shared__ uint32_t s_pbuf[WAVES][PBUF];
    __shared__ uint4 s_cq[CONT ? WAVES : 1][CONT ? CQ : 1];
    __shared__ uint2 s_tab[WAVES][GGA_WAVE];
    __shared__ uint32_t s_wave[WAVES], s_min[WAVES];
    constexpr bool LVL = BFS && !CONT;
    uint32_t *const stage = &s_pbuf[0][0];   // (the push buffers are free outside the relax phase)
    static_assert(CSTAGE <= WAVES * PBUF, "staging fits the push buffers");
    uint32_t step;
    const uint32_t phase = gga_next_phase(w.ctl, launch, w.dense_min, !BFS && w.last != nullptr, w.cap, &step);
    if (phase == GGA_PH_DONE || phase == GGA_PH_CAPPED) {
        if (blockIdx.x == 0 && threadIdx.x == 0) w.ctl[GGA_CTL_PHASE(launch)] = phase;
        return;
    }
    const uint32_t it = w.ctl[GGA_CTL_ITER(step % 3u)], sout = (step + 1u) % 3u;
    const uint32_t nq = phase == GGA_PH_RELAX ? step_len(w, step) : 0u;
    if (blockIdx.x == 0 && threadIdx.x == 0) {
        w.ctl[GGA_CTL_PHASE(launch)] = phase;
        w.ctl[GGA_CTL_PSTEP(launch)] = step;
        w.ctl[GGA_CTL_PLEN(launch)] = nq;
        w.ctl[GGA_CTL_PHASES] += 1u;
        if (phase == GGA_PH_RELAX) step_bookkeeping(w.ctl, step, it, nq);
        if (phase == GGA_PH_RCOUNT) w.ctl[GGA_CTL_RTHR] = sat_add(w.ctl[GGA_CTL_THR(sout)], w.delta);
    }
    if (phase == GGA_PH_RELAX) {
        Counters cnt;
        const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x / GGA_WAVE);
        worklist_step<BFS, false, CONT, SPREAD>(g, w, step, nq, it, s_pbuf[wv], s_cq[CONT ? wv : 0], s_tab[wv], cnt);
    } else if (phase == GGA_PH_COUNT) {
        const ListOut o = list_out(g, w, step);
        uint32_t any = 0;
        for (uint32_t t = blockIdx.x; t < GGA_TILES(g.n); t += gridDim.x)
            any |= LVL ? compact_count_tile(o, g.n, t, level_marked<false>(w, it), s_wave)
                       : compact_count_tile(o, g.n, t, StampMarked<false>{w.flag}, s_wave);
        if (any && threadIdx.x == 0) w.ctl[GGA_CTL_LISTED(sout)] = 1u;
    } else if (phase == GGA_PH_WRITE) {
        const ListOut o = list_out(g, w, step);
        if (LVL) compact_write_tiles(o, g.n, level_marked<true>(w, it), s_wave, stage);
        else compact_write_tiles(o, g.n, StampMarked<true>{w.flag}, s_wave, stage);
    } else if (!BFS && phase == GGA_PH_RCOUNT) {
        refill_count_body(g, w, step, s_wave, s_min);
    } else if (!BFS) {
        refill_list_body(g, w, step, s_wave, s_min, stage);
    }
}

// ------------------------------------------------------ persistent kernel
template <bool BFS, bool COUNT, bool CONT>
__global__ __launch_bounds__(BLOCK) void k_persistent(gga_dev_graph g, gga_dev_work w,
                                                      uint32_t max_steps, uint64_t spin_ticks) {
    __shared__ uint32_t s_pbuf[WAVES][PBUF];
    __shared__ uint4 s_cq[CONT ? WAVES : 1][CONT ? CQ : 1];
    __shared__ uint2 s_tab[WAVES][GGA_WAVE];
    __shared__ uint32_t s_state[2];
    __shared__ uint32_t s_wave[WAVES], s_min[WAVES];
    uint32_t gen = 0;
    if (threadIdx.x == 0)
        gen = __hip_atomic_load(&w.ctl[GGA_CTL_BARGEN], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    Counters cnt;
    for (uint32_t step = 0; step < max_steps; step++) {
        const uint32_t sin = step % 3u;
        if (threadIdx.x == 0) {
            s_state[0] = __hip_atomic_load(&w.ctl[GGA_CTL_TAIL(sin)], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            s_state[1] = __hip_atomic_load(&w.ctl[GGA_CTL_ERR], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        const uint32_t nq = s_state[0] < w.qcap ? s_state[0] : w.qcap, err = s_state[1];
        __syncthreads();
        if (nq == 0 || err) break;
        const uint32_t it = w.ctl[GGA_CTL_ITER(sin)];
        if (blockIdx.x == 0 && threadIdx.x == 0) step_bookkeeping(w.ctl, step, it, nq);
        const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x / GGA_WAVE);
        worklist_step<BFS, COUNT, CONT ? FOLLOW_EITHER : FOLLOW_NONE>(g, w, step, nq, it, s_pbuf[wv], s_cq[CONT ? wv : 0], s_tab[wv], cnt);
        if (flag_step(w, nq)) {
            const ListOut o = list_out(g, w, step);
            grid_barrier(w.ctl, gridDim.x, gen, spin_ticks);
            for (uint32_t t = blockIdx.x; t < GGA_TILES(g.n); t += gridDim.x) {
                if (BFS && !CONT) compact_count_tile(o, g.n, t, level_marked<false>(w, it), s_wave);
                else compact_count_tile(o, g.n, t, StampMarked<false>{w.flag}, s_wave);
            }
            grid_barrier(w.ctl, gridDim.x, gen, spin_ticks);
            // each workgroup sums the tile counts before its own tiles: no
            // serial scan between two more grid barriers
            if (BFS && !CONT) compact_write_tiles(o, g.n, level_marked<true>(w, it), s_wave, &s_pbuf[0][0]);
            else compact_write_tiles(o, g.n, StampMarked<true>{w.flag}, s_wave, &s_pbuf[0][0]);
        }
        grid_barrier(w.ctl, gridDim.x, gen, spin_ticks);
        // near-far: an empty next list is refilled from the deferred vertices,
        // as often as the threshold has to jump over empty buckets
        while (w.last) {
            if (threadIdx.x == 0) {
                s_state[0] = __hip_atomic_load(&w.ctl[GGA_CTL_TAIL((step + 1u) % 3u)], __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
                s_state[1] = __hip_atomic_load(&w.ctl[GGA_CTL_ERR], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            __syncthreads();
            const uint32_t tail = s_state[0], rerr = s_state[1];
            __syncthreads();
            if (tail || rerr) break;
            refill_count_body(g, w, step, s_wave, s_min);
            grid_barrier(w.ctl, gridDim.x, gen, spin_ticks);
            if (blockIdx.x == 0) refill_scan_body(g, w, step, s_wave, s_min);
            grid_barrier(w.ctl, gridDim.x, gen, spin_ticks);
            if (threadIdx.x == 0) {
                s_state[0] = __hip_atomic_load(&w.ctl[GGA_CTL_TAIL((step + 1u) % 3u)], __ATOMIC_RELAXED,
                                               __HIP_MEMORY_SCOPE_AGENT);
                s_state[1] = __hip_atomic_load(&w.ctl[GGA_CTL_FAR], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
            __syncthreads();
            const uint32_t listed = s_state[0], far = s_state[1];
            __syncthreads();
            if (listed) {
                refill_write_body(g, w, step, s_wave, &s_pbuf[0][0]);
                grid_barrier(w.ctl, gridDim.x, gen, spin_ticks);
                break;
            }
            if (!far) break;   // converged: the next step finds an empty list
        }
    }
    publish_counters<COUNT>(w, cnt);
}

// ------------------------------------------------------ reductions
// Block-wide sum of one uint64 per thread (all threads get the total).
__device__ __forceinline__ uint64_t block_sum64(uint64_t x, uint64_t *s_red) {
    x = wave_sum64(x);
    if (lane_id() == 0) s_red[threadIdx.x / GGA_WAVE] = x;
    __syncthreads();
    uint64_t t = 0;
    for (uint32_t i = 0; i < WAVES; i++) t += s_red[i];
    __syncthreads();
    return t;
}

// Pass 1 (REACH_BLOCKS workgroups): per-workgroup reached / m_reach partials
// into cnt slots [0, REACH_BLOCKS) word 3 and [REACH_BLOCKS, 2 REACH_BLOCKS)
// word 3 -- plain stores, no shared counter.
constexpr uint32_t REACH_BLOCKS = GGA_CNT_SLOTS / 2;
// A thread's reached vertices and their out-degree sum.
__device__ __forceinline__ void reach_sum(const gga_dev_graph &g, const gga_dev_work &w, uint64_t &reached,
                                          uint64_t &mr) {
    reached = mr = 0;
    const uint64_t S = (uint64_t)gridDim.x * blockDim.x;
    uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    // four vertices S apart per round, every load issued before the first
    // is used (a latency-bound loop otherwise: 20 us on 4.2 M vertices)
    for (; v + 3u * S < g.n; v += 4u * S) {
        uint32_t d[4], r0[4], r1[4];
#pragma unroll
        for (uint32_t k = 0; k < 4; k++) {
            d[k] = w.dist[v + k * S];
            r0[k] = g.row[v + k * S];
            r1[k] = g.row[v + k * S + 1u];
        }
#pragma unroll
        for (uint32_t k = 0; k < 4; k++)
            if (d[k] < w.inf) {
                reached += 1;
                mr += r1[k] - r0[k];
            }
    }
    for (; v < g.n; v += S) {
        if (w.dist[v] < w.inf) {
            reached += 1;
            mr += g.row[v + 1] - g.row[v];
        }
    }
}

__global__ __launch_bounds__(BLOCK) void k_reach(gga_dev_graph g, gga_dev_work w) {
    __shared__ uint64_t s_red[WAVES];
    uint64_t reached, mr;
    reach_sum(g, w, reached, mr);
    reached = block_sum64(reached, s_red);
    mr = block_sum64(mr, s_red);
    if (threadIdx.x == 0) {
        w.cnt[4u * blockIdx.x + 3u] = reached;
        w.cnt[4u * (REACH_BLOCKS + blockIdx.x) + 3u] = mr;
    }
}

// Pass 2 (one workgroup): fold the partials into ctl[RED] and the striped work
// counters into ctl[CNT].
__global__ __launch_bounds__(BLOCK) void k_reach_fold(gga_dev_work w) {
    __shared__ uint64_t s_red[WAVES];
    uint64_t s[5] = {0, 0, 0, 0, 0};
    for (uint32_t i = threadIdx.x; i < GGA_CNT_SLOTS; i += blockDim.x) {
        for (uint32_t k = 0; k < 3; k++) s[k] += w.cnt[4u * i + k];
        s[i < REACH_BLOCKS ? 3 : 4] += w.cnt[4u * i + 3u];
    }
    uint64_t *cnt = reinterpret_cast<uint64_t *>(w.ctl + GGA_CTL_CNT);
    uint64_t *red = reinterpret_cast<uint64_t *>(w.ctl + GGA_CTL_RED);
    for (uint32_t k = 0; k < 5; k++) {
        const uint64_t t = block_sum64(s[k], s_red);
        if (threadIdx.x == 0) {
            if (k < 3) cnt[k] = t;
            else red[k - 3] = t;
        }
    }
}

// The ending of a phase-launched query: reach partials and the control words
// (lines 0 to 8) straight to the pinned read-back area, one launch where the
// reach pass, its fold and a copy were three; stage: the distances of a small
// graph go to pinned memory with it.
__global__ __launch_bounds__(BLOCK) void k_finish(gga_dev_graph g, gga_dev_work w, uint32_t *host, uint32_t *stage) {
    __shared__ uint64_t s_red[WAVES];
    uint64_t *part = reinterpret_cast<uint64_t *>(host + GGA_FIN_PART);
    if (blockIdx.x == 0) {
        if (threadIdx.x == 0) {
            uint64_t *clock = reinterpret_cast<uint64_t *>(host + GGA_FIN_CLOCK);
            clock[1] = wall_clock64();
            clock[0] = *reinterpret_cast<uint64_t *>(w.ctl + GGA_CTL_T0);
        }
        for (uint32_t i = threadIdx.x; i < 9u * GGA_CTL_LINE; i += blockDim.x) host[i] = w.ctl[i];
    }
    if (stage)
        for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < g.n; v += (uint64_t)gridDim.x * blockDim.x)
            stage[v] = w.dist[v];
    uint64_t reached, mr;
    reach_sum(g, w, reached, mr);
    reached = block_sum64(reached, s_red);
    mr = block_sum64(mr, s_red);
    if (threadIdx.x == 0) {
        part[2u * blockIdx.x] = reached;
        part[2u * blockIdx.x + 1u] = mr;
    }
}

// ------------------------------------------------------ small graphs
// A whole query in one launch of one workgroup: distances, row offsets and both
// frontier queues in LDS (12 bytes a vertex), col and w read from L2.  On a
// graph this small every step is a chain of dependent accesses whatever the
// grid, and the launches around it cost more than the step: here a step is an
// LDS read, one edge load, an LDS atomic and a workgroup barrier (0.7 us:
// BFS on a 100 x 77 grid, 176 levels in 121 us).  What bounds it: that chain on meshes, one CU's rate of
// edges elsewhere (plan_query in host/graph.c has the sizes).
// 1024 / 512 / 256 threads: 100 x 77 grid 164 / 199 / 271 us, 110 x 111 246 /
// 302 / 427, R-MAT of 15 k edges 79 / 107 / 148.
//
// A vertex waits in the next queue at most once (bit in `mark`).  Taking it
// from the queue clears the bit before its distance is read, so an
// improvement either comes before that read or queues the vertex again.
//
// MESH: few edges a vertex; SSSP then lists only distances under a threshold
// (near-far, buckets of w.delta): the others set the vertex's bit in `far`, and
// an empty queue is refilled from those under the next threshold.
constexpr uint32_t SMALL_BLOCK = 1024, SMALL_WAVES = SMALL_BLOCK / GGA_WAVE;
template <bool BFS, bool MESH>
__global__ __launch_bounds__(SMALL_BLOCK) void k_small(gga_dev_graph g, gga_dev_work w, uint32_t src, uint32_t *host,
                                                       uint32_t *stage) {
    extern __shared__ __align__(16) uint32_t lds[];
    constexpr bool NEAR = MESH && !BFS;
    __shared__ uint2 s_tab[MESH ? 1 : SMALL_WAVES][GGA_WAVE];
    __shared__ uint64_t s_red[2][SMALL_WAVES];
    __shared__ uint32_t s_len[3], s_low;
    const uint32_t n = g.n, inf = w.inf, l = lane_id();
    const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x / GGA_WAVE);
    uint32_t *const dist = lds, *const row = dist + n, *const mark = row + n + 1u;
    uint32_t *const far = mark + (n + 31u) / 32u;   // (near-far only)
    uint16_t *const q0 = reinterpret_cast<uint16_t *>(NEAR ? far + (n + 31u) / 32u : far), *const q1 = q0 + n;
    uint2 *const tab = s_tab[MESH ? 0 : wv];
    uint32_t thr = NEAR ? w.delta : 0xFFFFFFFFu;
    uint64_t t0 = 0;
    if (threadIdx.x == 0) t0 = wall_clock64();
    for (uint32_t v = threadIdx.x; v < n; v += SMALL_BLOCK) {
        dist[v] = v == src ? 0u : inf;
        row[v] = g.row[v];
    }
    for (uint32_t i = threadIdx.x; i < (n + 31u) / 32u; i += SMALL_BLOCK) {
        mark[i] = 0u;
        if (NEAR) far[i] = 0u;
    }
    if (threadIdx.x == 0) {
        row[n] = g.m;
        q0[0] = (uint16_t)src;
        s_len[0] = 1u;
        s_len[1] = s_len[2] = 0u;
    }
    __syncthreads();
    uint32_t step = 0, cur = 0, nf;
    for (;; step++) {
        nf = s_len[cur];
        if (NEAR && nf == 0u) {
            // the deferred vertices under the next threshold, which starts at
            // the smallest of them when the bucket after this one is empty
            if (threadIdx.x == 0) s_low = 0xFFFFFFFFu;
            __syncthreads();
            uint32_t low = 0xFFFFFFFFu;
            for (uint32_t v = threadIdx.x; v < n; v += SMALL_BLOCK)
                if ((far[v >> 5] >> (v & 31u)) & 1u) low = dist[v] < low ? dist[v] : low;
            if (low != 0xFFFFFFFFu) atomicMin(&s_low, low);
            __syncthreads();
            low = s_low;
            if (low == 0xFFFFFFFFu) break;
            thr = sat_add(low > thr ? low : thr, w.delta);
            uint16_t *const qin = (step & 1u) ? q1 : q0;
            for (uint32_t v = threadIdx.x; v < n; v += SMALL_BLOCK)
                if (((far[v >> 5] >> (v & 31u)) & 1u) && dist[v] < thr) {
                    atomicOr(&mark[v >> 5], 1u << (v & 31u));
                    qin[atomicAdd(&s_len[cur], 1u)] = (uint16_t)v;
                }
            __syncthreads();
            nf = s_len[cur];
        }
        if (nf == 0u || step >= w.cap) break;   // (the same for every thread)
        const uint32_t nxt = cur == 2u ? 0u : cur + 1u;
        // the slot after the next: read last in the step before, filled in the next one
        if (threadIdx.x == 0) s_len[nxt == 2u ? 0u : nxt + 1u] = 0u;
        const uint16_t *const qin = (step & 1u) ? q1 : q0;
        uint16_t *const qout = (step & 1u) ? q0 : q1;
        // lowers dist[v] to alt where `on` and queues v; whole-wave call
        auto relax = [&](bool on, uint32_t v, uint32_t alt) {
            bool push = false;
            if (on && alt < __hip_atomic_fetch_min(&dist[v], alt, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) {
                const uint32_t bit = 1u << (v & 31u);
                if (NEAR && alt >= thr) atomicOr(&far[v >> 5], bit);
                else
                    push = !(__hip_atomic_fetch_or(&mark[v >> 5], bit, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP) &
                             bit);
            }
            const uint64_t pm = __ballot(push);
            if (pm) {
                uint32_t at = 0;
                if (l == 0) at = atomicAdd(&s_len[nxt], (uint32_t)__popcll(pm));
                at = wave_bcast(at, 0) + __builtin_amdgcn_mbcnt_hi((uint32_t)(pm >> 32),
                                                                  __builtin_amdgcn_mbcnt_lo((uint32_t)pm, 0u));
                if (push) qout[at] = (uint16_t)v;   // (a vertex once: at < n)
            }
        };
        // out of the queue: its distance from now on.  (Its distance is under
        // the threshold, so no deferral of it can follow.)  By one lane a
        // vertex: a second clear of the bit could come after another wave has
        // set it and queued x again, and x would be queued twice, past n.
        // (Cleared by all four lanes of a group SSSP took 10% longer.)
        auto clear = [&](uint32_t x) {
            if (NEAR) atomicAnd(&far[x >> 5], ~(1u << (x & 31u)));
            __hip_atomic_fetch_and(&mark[x >> 5], ~(1u << (x & 31u)), __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_WORKGROUP);
        };
        auto distance = [&](uint32_t x) {
            return __hip_atomic_load(&dist[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        };
        if (MESH) {
            // four neighbouring lanes a vertex, four edges at a time: no scan,
            // no owner search (as in follow_front)
            for (uint32_t b = wv * 16u; b < nf; b += SMALL_WAVES * 16u) {
                const uint32_t i = b + (l >> 2);
                uint32_t x = 0, eb = 0, ne = 0, du = inf;
                if (i < nf) {
                    x = qin[i];
                    eb = row[x];
                    ne = row[x + 1u] - eb;
                    if ((l & 3u) == 0u) clear(x);
                }
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");   // the clears before the reads
                __builtin_amdgcn_wave_barrier();
                if (i < nf) du = distance(x);
                for (uint32_t j = l & 3u; __ballot(j < ne) != 0ull; j += 4u) {
                    const bool on = j < ne;
                    const uint32_t e = on ? eb + j : 0u;   // (some lane has an edge: slot 0 is in bounds)
                    const uint32_t v = g.col[e], alt = du + (BFS ? 1u : g.w[e]);
                    relax(on && alt >= du && alt < inf, v, alt);
                }
            }
            cur = nxt;
            __syncthreads();
            continue;
        }
        uint32_t bsz = (nf + SMALL_WAVES - 1u) / SMALL_WAVES;
        bsz = bsz < GGA_WAVE ? bsz : GGA_WAVE;
        const uint32_t half = bsz <= 1u ? 0u : 1u << (31 - __builtin_clz(bsz - 1u));
        for (uint32_t b = wv * bsz; b < nf; b += SMALL_WAVES * bsz) {
            uint32_t eb = 0, ne = 0, du = inf;
            if (l < bsz && b + l < nf) {
                const uint32_t x = qin[b + l];
                clear(x);
                du = distance(x);
                eb = row[x];
                ne = row[x + 1u] - eb;
            }
            const uint32_t incl = wave_incl_scan(ne);
            const uint32_t total = wave_last(incl);
            tab[l] = make_uint2(eb - (incl - ne), du);   // (as in expand_batch)
            __builtin_amdgcn_wave_barrier();
            for (uint32_t base = 0; base < total; base += GGA_WAVE * UNROLL) {
                uint32_t v[UNROLL], alt[UNROLL], ds[UNROLL], kk[UNROLL], own[UNROLL];
                const uint32_t left = total - base;
#pragma unroll
                for (uint32_t u = 0; u < UNROLL; u++) {
                    const uint32_t k = base + u * GGA_WAVE + l;
                    kk[u] = k < total ? k : total - 1u;
                    own[u] = 0;
                }
                for (uint32_t s = half; s != 0; s >>= 1) {
#pragma unroll
                    for (uint32_t u = 0; u < UNROLL; u++) {
                        const uint32_t y = __shfl(incl, (int)(own[u] + s - 1), GGA_WAVE);
                        own[u] += y <= kk[u] ? s : 0u;
                    }
                }
#pragma unroll
                for (uint32_t u = 0; u < UNROLL; u++) {
                    if (u * GGA_WAVE >= left) break;
                    const uint2 t = tab[own[u]];
                    ds[u] = t.y;
                    v[u] = g.col[t.x + kk[u]];
                    alt[u] = t.y + (BFS ? 1u : g.w[t.x + kk[u]]);
                }
#pragma unroll
                for (uint32_t u = 0; u < UNROLL; u++) {
                    if (u * GGA_WAVE >= left) break;
                    relax(base + u * GGA_WAVE + l < total && alt[u] >= ds[u] && alt[u] < inf && alt[u] < dist[v[u]],
                          v[u], alt[u]);
                }
            }
            __builtin_amdgcn_wave_barrier();
        }
        cur = nxt;
        __syncthreads();
    }
    uint64_t reached = 0, mr = 0;
    for (uint32_t v = threadIdx.x; v < n; v += SMALL_BLOCK) {
        const uint32_t d = dist[v];
        w.dist[v] = d;
        if (stage) stage[v] = d;
        if (d < inf) {
            reached += 1u;
            mr += row[v + 1u] - row[v];
        }
    }
    reached = wave_sum64(reached);
    mr = wave_sum64(mr);
    if (l == 0) {
        s_red[0][wv] = reached;
        s_red[1][wv] = mr;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        uint64_t *part = reinterpret_cast<uint64_t *>(host + GGA_FIN_PART);
        uint64_t *clock = reinterpret_cast<uint64_t *>(host + GGA_FIN_CLOCK);
        reached = mr = 0;
        for (uint32_t i = 0; i < SMALL_WAVES; i++) {
            reached += s_red[0][i];
            mr += s_red[1][i];
        }
        part[0] = reached;
        part[1] = mr;
        clock[0] = t0;
        clock[1] = wall_clock64();
        for (uint32_t i = 0; i < 3; i++) host[GGA_CTL_ITER(i)] = w.epoch;   // (no stamps taken)
        host[GGA_CTL_STEPS] = step;
        host[GGA_CTL_ERR] = 0u;
        host[GGA_CTL_TAIL(0)] = nf;   // not 0: the step cap
    }
}

// Fingerprint of dist: sum over v of mix64(v << 32 | dist[v]) (the host's
// gga_checksum); partials in word 3 of cnt slots [0, REACH_BLOCKS), folded
// into ctl[RED + 4] (uint64).
__device__ __forceinline__ uint64_t mix64(uint64_t x) {
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    return x ^ (x >> 31);
}

__global__ __launch_bounds__(BLOCK) void k_checksum(gga_dev_graph g, gga_dev_work w) {
    __shared__ uint64_t s_red[WAVES];
    uint64_t h = 0;
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < g.n;
         v += (uint64_t)gridDim.x * blockDim.x)
        h += mix64((v << 32) | w.dist[v]);
    h = block_sum64(h, s_red);
    if (threadIdx.x == 0) w.cnt[4u * blockIdx.x + 3u] = h;
}

__global__ __launch_bounds__(BLOCK) void k_checksum_fold(gga_dev_work w) {
    __shared__ uint64_t s_red[WAVES];
    uint64_t h = 0;
    for (uint32_t i = threadIdx.x; i < REACH_BLOCKS; i += blockDim.x) h += w.cnt[4u * i + 3u];
    h = block_sum64(h, s_red);
    if (threadIdx.x == 0) reinterpret_cast<uint64_t *>(w.ctl + GGA_CTL_RED)[2] = h;
}

// verifysolution (myutils.h:1-18) plus tightness, over chunks.
template <bool BFS>
__global__ __launch_bounds__(BLOCK) void k_verify_edges(gga_dev_graph g, gga_dev_work w,
                                                        uint8_t *tight) {
    const uint32_t l = lane_id();
    const uint64_t c = ((uint64_t)blockIdx.x * WAVES + threadIdx.x / GGA_WAVE) * GGA_WAVE + l;
    uint32_t eb = 0, n = 0, du = w.inf;
    if (c < g.C) {
        eb = g.cbeg[c];
        du = w.dist[g.cown[c]];
        n = du < w.inf ? g.cbeg[c + 1] - eb : 0u;
    }
    const uint32_t incl = wave_incl_scan(n);
    const uint32_t total = wave_last(incl);
    const uint32_t excl = incl - n;
    uint64_t nerr = 0;
    for (uint32_t base = 0; base < total; base += GGA_WAVE) {
        const uint32_t k = base + l;
        const uint32_t kk = k < total ? k : total - 1;
        const uint32_t j = wave_owner(incl, kk);
        const uint32_t e = wave_bcast(eb, j) + (kk - wave_bcast(excl, j));
        const uint32_t ds = wave_bcast(du, j);
        if (k < total) {
            const uint32_t v = g.col[e];
            const uint32_t wt = BFS ? 1u : g.w[e];
            const uint32_t alt = ds + wt;
            if (alt >= ds) {
                const uint32_t dv = w.dist[v];
                if (wt > 0 && alt < w.inf && alt < dv) nerr++;
                if (alt == dv) tight[v] = 1;
            }
        }
    }
    nerr = wave_sum64(nerr);
    if (l == 0 && nerr) atomic_add_u64(reinterpret_cast<uint64_t *>(w.ctl + GGA_CTL_RED), nerr);
}

__global__ __launch_bounds__(BLOCK) void k_verify_vertices(gga_dev_graph g, gga_dev_work w,
                                                           uint32_t src, const uint8_t *tight) {
    uint64_t bad = 0;
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < g.n;
         v += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t d = w.dist[v];
        if (v == src) bad += d != 0u;
        else if (d < w.inf && !tight[v]) bad++;
    }
    bad = wave_sum64(bad);
    if (lane_id() == 0 && bad) atomic_add_u64(reinterpret_cast<uint64_t *>(w.ctl + GGA_CTL_RED) + 1, bad);
}

inline int launch_status() { return (int)hipGetLastError(); }

inline uint32_t grid_for(uint64_t items, uint32_t cap) {
    uint64_t gsz = (items + BLOCK - 1) / BLOCK;
    if (gsz == 0) gsz = 1;
    return (uint32_t)(gsz < cap ? gsz : cap);
}

}  // namespace

namespace {
constexpr int SCRATCH_DEVICES = 64;
std::mutex scratch_mu;
void *scratch_addr[SCRATCH_DEVICES];   // device address of `scratch`, per device
}  // namespace

extern "C" int ggak_scratch(int device, void **ptr) {
    *ptr = nullptr;
    if (device < 0 || device >= SCRATCH_DEVICES) return (int)hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lock(scratch_mu);
    if (!scratch_addr[device]) {
        // once per device, with that device current
        int cur = -1;
        hipError_t e = hipGetDevice(&cur);
        if (e != hipSuccess) return (int)e;
        if (cur != device && (e = hipSetDevice(device)) != hipSuccess) return (int)e;
        void *p = nullptr;
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (cur != device) (void)hipSetDevice(cur);
        if (e != hipSuccess) return (int)e;
        if (!p) return (int)hipErrorInvalidSymbol;
        scratch_addr[device] = p;
    }
    *ptr = scratch_addr[device];
    return 0;
}

extern "C" int ggak_fill_u32(uint32_t *p, uint32_t value, uint64_t count, hipStream_t s) {
    if (count == 0) return 0;
    k_fill<<<grid_for(count, 8192), BLOCK, 0, s>>>(p, value, count);
    return launch_status();
}

extern "C" int ggak_query_init(gga_dev_graph g, gga_dev_work w, uint32_t src, uint32_t epoch,
                               hipStream_t s) {
    k_query_init<<<grid_for(g.n, 8192), BLOCK, 0, s>>>(g, w, src, epoch);
    return launch_status();
}

extern "C" int ggak_topo_step(gga_dev_graph g, gga_dev_work w, int bfs, int count, hipStream_t s) {
    const uint64_t waves = ((uint64_t)g.C + GGA_WAVE - 1) / GGA_WAVE;
    const uint32_t grid = (uint32_t)((waves + WAVES - 1) / WAVES);
    if (grid == 0) return 0;
    if (bfs) {
        if (count) k_topo_step<true, true><<<grid, BLOCK, 0, s>>>(g, w);
        else k_topo_step<true, false><<<grid, BLOCK, 0, s>>>(g, w);
    } else {
        if (count) k_topo_step<false, true><<<grid, BLOCK, 0, s>>>(g, w);
        else k_topo_step<false, false><<<grid, BLOCK, 0, s>>>(g, w);
    }
    return launch_status();
}

// Kernel variants by (bfs, count, instrumented, mesh continuation) and
// workgroup size.  The continuation has kernels of its own, so that the
// registers of the others stay as they were.
template <bool BFS, bool COUNT, bool TL, bool CONT, bool SPREAD>
static const void *wl_fn_c(uint32_t block) {
    switch (block) {
    case 128: return reinterpret_cast<const void *>(&k_wl_step<BFS, COUNT, TL, 128, CONT, SPREAD>);
    case 512: return reinterpret_cast<const void *>(&k_wl_step<BFS, COUNT, TL, 512, CONT, SPREAD>);
    default: return reinterpret_cast<const void *>(&k_wl_step<BFS, COUNT, TL, 256, CONT, SPREAD>);
    }
}
// (spread: SSSP on graphs that are not meshes, see expand_batch)
template <bool BFS, bool COUNT, bool TL>
static const void *wl_fn(uint32_t block, int cont, int spread) {
    if constexpr (!BFS)
        if (spread) return wl_fn_c<BFS, COUNT, TL, false, true>(block);
    return cont ? wl_fn_c<BFS, COUNT, TL, true, false>(block) : wl_fn_c<BFS, COUNT, TL, false, false>(block);
}
template <bool BFS, bool COUNT>
static const void *persistent_fn(int cont) {
    return cont ? reinterpret_cast<const void *>(&k_persistent<BFS, COUNT, true>)
                : reinterpret_cast<const void *>(&k_persistent<BFS, COUNT, false>);
}
// cont: the graph is a mesh (bmin > 1) and the continuation is compiled in
static int use_cont(const gga_dev_work &w) { return GGA_CONT > 0 && w.bmin > 1u; }
// Level-synchronous BFS: worklist and persistent queries without the
// continuation (which reaches levels out of order).
extern "C" int ggak_level_sync(gga_dev_work w, int bfs) { return bfs && !use_cont(w); }
static const void *pick_kernel(int persistent, int bfs, int count, uint32_t block, int cont, int spread) {
    if (persistent) {
        if (bfs) return count ? persistent_fn<true, true>(cont) : persistent_fn<true, false>(cont);
        return count ? persistent_fn<false, true>(cont) : persistent_fn<false, false>(cont);
    }
    if (bfs) return count ? wl_fn<true, true, false>(block, cont, 0) : wl_fn<true, false, false>(block, cont, 0);
    return count ? wl_fn<false, true, false>(block, cont, spread) : wl_fn<false, false, false>(block, cont, spread);
}

extern "C" int ggak_wl_step(gga_dev_graph g, gga_dev_work w, uint32_t step, int bfs, int count,
                            uint32_t grid, uint32_t block, gga_wg_record *tl, hipStream_t s) {
    if (grid == 0 || (block != 128 && block != 256 && block != 512)) return (int)hipErrorInvalidValue;
    void *args[] = {&g, &w, &step, &tl};
    // the instrumented variant always counts (its timeline goes with the work counters)
    const int cont = use_cont(w), spread = w.sdist != nullptr;
    const void *fn = tl ? (bfs ? wl_fn<true, true, true>(block, cont, 0) : wl_fn<false, true, true>(block, cont, spread))
                        : pick_kernel(0, bfs, count, block, cont, spread);
    return (int)hipLaunchKernel(fn, dim3(grid), dim3(block), args, 0, s);
}

// Convergence of one step against the final distances (printConv_rtime,
// convergence.h:100-140): diff = vertices whose distance differs; sq = sum of
// (final - cur)^2 evaluated in uint32 arithmetic as the reference does with
// its unsigned foru values (so an unreached vertex contributes
// (final - inf)^2 mod 2^32).  rows[0] += diff, rows[1] += sq.
__global__ __launch_bounds__(BLOCK) void k_conv(const uint32_t *dist, const uint32_t *fin, uint32_t n,
                                                uint64_t *rows) {
    __shared__ uint64_t s_red[WAVES];
    uint64_t diff = 0, sq = 0;
    for (uint64_t v = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n; v += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t fs = fin[v], fi = dist[v];
        const uint32_t d = fs - fi;
        diff += fs != fi;
        sq += (uint32_t)(d * d);
    }
    diff = block_sum64(diff, s_red);
    sq = block_sum64(sq, s_red);
    if (threadIdx.x == 0) {
        if (diff) atomic_add_u64(&rows[0], diff);
        if (sq) atomic_add_u64(&rows[1], sq);
    }
}

extern "C" int ggak_conv(const uint32_t *dist, const uint32_t *fin, uint32_t n, uint64_t *rows, hipStream_t s) {
    k_conv<<<grid_for(n, 1024), BLOCK, 0, s>>>(dist, fin, n, rows);
    return launch_status();
}

extern "C" int ggak_wl_phase(gga_dev_graph g, gga_dev_work w, uint32_t launch, int bfs, uint32_t grid, hipStream_t s) {
    if (grid == 0) return (int)hipErrorInvalidValue;
    if (bfs) {
        if (use_cont(w) && w.guard) k_wl_phase<true, FOLLOW_GUARD, false><<<grid, BLOCK, 0, s>>>(g, w, launch % 3u);
        else if (use_cont(w)) k_wl_phase<true, FOLLOW, false><<<grid, BLOCK, 0, s>>>(g, w, launch % 3u);
        else k_wl_phase<true, FOLLOW_NONE, false><<<grid, BLOCK, 0, s>>>(g, w, launch % 3u);
    } else {
        if (use_cont(w) && w.guard) k_wl_phase<false, FOLLOW_GUARD, false><<<grid, BLOCK, 0, s>>>(g, w, launch % 3u);
        else if (use_cont(w)) k_wl_phase<false, FOLLOW, false><<<grid, BLOCK, 0, s>>>(g, w, launch % 3u);
        else if (w.sdist) k_wl_phase<false, FOLLOW_NONE, true><<<grid, BLOCK, 0, s>>>(g, w, launch % 3u);
        else k_wl_phase<false, FOLLOW_NONE, false><<<grid, BLOCK, 0, s>>>(g, w, launch % 3u);
    }
    return launch_status();
}

extern "C" int ggak_finish(gga_dev_graph g, gga_dev_work w, uint32_t *host, uint32_t *stage, uint32_t *blocks,
                           hipStream_t s) {
    *blocks = grid_for(g.n, GGA_FIN_BLOCKS);
    k_finish<<<*blocks, BLOCK, 0, s>>>(g, w, host, stage);
    return launch_status();
}

static uint32_t small_bytes(uint32_t n) { return 4u * n + 4u * (n + 1u) + 8u * ((n + 31u) / 32u) + 4u * n; }

extern "C" int ggak_small(gga_dev_graph g, gga_dev_work w, uint32_t src, int bfs, int thin, uint32_t *host, uint32_t *stage,
                          hipStream_t s) {
    if (g.n == 0 || g.n > GGA_SMALL_N || src >= g.n || (thin && !bfs && w.delta == 0u)) return (int)hipErrorInvalidValue;
    const uint32_t bytes = small_bytes(g.n);
    const void *fn = bfs ? (thin ? reinterpret_cast<const void *>(&k_small<true, true>)
                                 : reinterpret_cast<const void *>(&k_small<true, false>))
                         : (thin ? reinterpret_cast<const void *>(&k_small<false, true>)
                                 : reinterpret_cast<const void *>(&k_small<false, false>));
    hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)small_bytes(GGA_SMALL_N));
    if (e != hipSuccess) return (int)e;
    void *args[] = {&g, &w, &src, &host, &stage};
    return (int)hipLaunchKernel(fn, dim3(1), dim3(SMALL_BLOCK), args, bytes, s);
}

extern "C" int ggak_refill(gga_dev_graph g, gga_dev_work w, uint32_t step, hipStream_t s) {
    if (!w.last) return 0;
    const uint32_t ntiles = GGA_TILES(g.n);
    const uint32_t grid = ntiles < 2048u ? (ntiles ? ntiles : 1u) : 2048u;
    k_refill_write<<<grid, BLOCK, 0, s>>>(g, w, step);   // (its count ran in k_compact_write)
    return launch_status();
}

extern "C" int ggak_compact(gga_dev_graph g, gga_dev_work w, uint32_t step, hipStream_t s) {
    const uint32_t ntiles = GGA_TILES(g.n);
    const uint32_t grid = ntiles < 2048u ? (ntiles ? ntiles : 1u) : 2048u;
    if (w.lvl) {
        k_compact_count<true><<<grid, BLOCK, 0, s>>>(g, w, step);
        k_compact_write<true><<<grid, BLOCK, 0, s>>>(g, w, step);
    } else {
        k_compact_count<false><<<grid, BLOCK, 0, s>>>(g, w, step);
        k_compact_write<false><<<grid, BLOCK, 0, s>>>(g, w, step);
    }
    return launch_status();
}

extern "C" uint32_t ggak_wl_grid(int device, int persistent, int bfs, int count, uint32_t block) {
    int cus = 0, per = 0;
    if (persistent) block = BLOCK;
    if (block != 128 && block != 256 && block != 512) return 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) return 0;
    // (asked of the variants without followed fronts, 8 of 256 threads per CU.
    // The mesh variants hold a queue of 8 KB a wave and four fit: their grid is
    // twice what is resident, and steps are too short for that to show -- the
    // tuner's grids of a half and a quarter are within 2% on 300^2 and 1024^2.
    // Persistent grids take one per CU either way.)
    const void *fn = pick_kernel(persistent, bfs, count, block, 0, 0);
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per, fn, (int)block, 0) != hipSuccess) return 0;
    if (per <= 0) return 0;
    // A grid barrier needs every workgroup resident at once.  On gfx950 the
    // occupancy query (7-8 per CU for these kernels) overstates what the
    // hardware co-schedules (6 per CU measured for the persistent kernel), and
    // the cooperative launch does not reject the excess.  Barrier cost grows
    // with the number of workgroups (8 us at 256, 25 us at 1024 measured), so
    // the persistent grid is one workgroup per CU.
    if (persistent && per > 1) per = 1;
    return (uint32_t)cus * (uint32_t)per;
}

extern "C" int ggak_persistent(gga_dev_graph g, gga_dev_work w, int bfs, int count, uint32_t grid,
                               uint32_t max_steps, uint32_t spin_limit_ms, hipStream_t s) {
    if (grid == 0) return (int)hipErrorInvalidValue;
    int dev = 0, khz = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev) != hipSuccess || khz <= 0)
        khz = 100000;  // 100 MHz
    uint64_t spin_ticks = (uint64_t)spin_limit_ms * (uint64_t)khz;
    void *args[] = {&g, &w, &max_steps, &spin_ticks};
    hipError_t e = hipLaunchCooperativeKernel(pick_kernel(1, bfs, count, BLOCK, use_cont(w), 0), dim3(grid),
                                              dim3(BLOCK), args, 0, s);
    if (e != hipSuccess) return (int)e;
    return launch_status();
}

extern "C" int ggak_reach(gga_dev_graph g, gga_dev_work w, hipStream_t s) {
    // REACH_BLOCKS partial slots are always all written (idle workgroups store 0)
    k_reach<<<REACH_BLOCKS, BLOCK, 0, s>>>(g, w);
    k_reach_fold<<<1, BLOCK, 0, s>>>(w);
    return launch_status();
}

extern "C" int ggak_checksum(gga_dev_graph g, gga_dev_work w, hipStream_t s) {
    k_checksum<<<REACH_BLOCKS, BLOCK, 0, s>>>(g, w);
    k_checksum_fold<<<1, BLOCK, 0, s>>>(w);
    return launch_status();
}

extern "C" int ggak_verify(gga_dev_graph g, gga_dev_work w, uint32_t src, int bfs, uint8_t *d_tight,
                           hipStream_t s) {
    const uint64_t waves = ((uint64_t)g.C + GGA_WAVE - 1) / GGA_WAVE;
    const uint32_t grid = (uint32_t)((waves + WAVES - 1) / WAVES);
    if (grid) {
        if (bfs) k_verify_edges<true><<<grid, BLOCK, 0, s>>>(g, w, d_tight);
        else k_verify_edges<false><<<grid, BLOCK, 0, s>>>(g, w, d_tight);
    }
    k_verify_vertices<<<grid_for(g.n, 4096), BLOCK, 0, s>>>(g, w, src, d_tight);
    return launch_status();
}
