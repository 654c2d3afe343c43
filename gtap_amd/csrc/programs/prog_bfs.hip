// prog_bfs.hip -- asynchronous (label-correcting) BFS as a thread-executed task program,
// with EPAQ routing of vertex tasks by out-degree bucket.
//
// Source program (shape of the reference's examples/asynchronous_bfs/asynchronous_bfs_thread.cu:19-55
// and evaluation/2-comparison/bfs/gtap_thread_bfs.cu:21-54):
//
//   #pragma gtap function
//   __device__ void bfs(int v, int s, int e, int d) {
//       if (depth[v] < d) return;                      // a shorter path already re-expanded v
//       if (e - s > SPLIT) {                           // split a long adjacency range into
//           int k = min(8, ceil((e - s) / SPLIT));     // k near-equal pieces
//           for (int i = 0; i < k; ++i) {
//               int ps = s + (e - s) * i / k, pe = s + (e - s) * (i + 1) / k;
//               #pragma gtap task queue(bucket(pe - ps))
//               bfs(v, ps, pe, d);
//           }
//           return;
//       }
//       for (int i = s; i < e; ++i) {
//           int u = col[i];
//           if (atomicMin(&depth[u], d + 1) > d + 1) {
//               #pragma gtap task queue(bucket(row[u + 1] - row[u]))
//               bfs(u, row[u], row[u + 1], d + 1);   // (the flat scan: not for a u without out-edges)
//           }
//       }
//   }
//
// bucket(deg) = 0 for deg < 8, 1 for < 64, 2 for < 512, 3 otherwise (4 EPAQ queues); with one
// queue every task goes to queue 0. No task waits for its children (detached spawns); the
// launch ends by quiescence. Distances are the BFS hop counts whatever the schedule.
//
// With 4 queues, queue 3 (ranges of 512 edges and more) is a wave queue: its task runs on a
// whole wavefront, which scans the range 512 edges at a time as a round's lane tasks are
// (expand, below). A range above kWaveSplitEdges (or an eighth of the deque
// capacity, if smaller) is first cut into up to 64 near-equal pieces, one spawned per lane.
// A hub's adjacency list is thus scanned by a few wave rounds instead of a tree of 64-edge
// lane tasks and their split tasks. One queue keeps the lane program for every range. (The
// reference cuts a long list into 32-edge tasks all spawned by one task,
// asynchronous_bfs_thread.cu:25-33; a bounded fan-out keeps one lane's spawn loop short.)
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "../device/gtap_abi.hpp"
#include "../device/gtap_block.hpp"
#include "../host/gtap_launch.hpp"

namespace gtap {
namespace bfs {

enum : uint32_t { F_BFS = 1 };
struct BfsArg {
    int32_t v;
    int32_t s;
    int32_t e;
    int32_t d;
};
struct BfsArgs {
    const int32_t* row;
    const int32_t* col;
    int32_t* depth;
    int32_t nv;
    int32_t split;
    int64_t ne;  // column entries: a vertex's offsets must satisfy 0 <= row[u] <= row[u+1] <= ne
    int32_t hub;   // a wave scans its rounds flat once it has met a range longer than this (-1: at once)
};

__host__ __device__ __forceinline__ uint32_t degree_bucket(int32_t deg) {
    return deg < 8 ? 0u : (deg < 64 ? 1u : (deg < 512 ? 2u : 3u));
}

// Set in the depth of a piece of a hub's range (depths are at most 0x3f3f3f3f), so that the wave that
// takes the piece knows too.
constexpr int32_t kHubPiece = 1 << 30;
constexpr int32_t kSplitFanout = 8;         // pieces per split of a lane task's range
constexpr int32_t kWaveSplitEdges = 2048;  // a wave task scans at most this many edges (and cap / 8)
constexpr int kWindows = 8;                 // edges per lane per step of an expansion
constexpr int32_t kMaxExpand = 1 << 20;     // edges of one range in one scan: 64 of them stay within an int32
constexpr int kHits = 192;                  // improved vertices held before their tasks are spawned

struct Segment {   // one task's edges in the flat sequence of a round's edges
    int32_t shift; // flat edge f is column entry f + shift
    int32_t nd;    // depth its neighbours get
};
// With 4 queues a workgroup takes 50784 bytes of LDS in all; three fit a CU up to 53760 (R-MAT 22
// with 53856 bytes, two a CU: 1343 us, with three 1161 us).
struct ExpandShared {
    uint32_t starts[2 * kWindows];  // per window of 64 flat edges, which of them start a segment
    Segment seg[kWave];
    uint32_t task[kWave];           // per segment, its task's id, for error reports
    int32_t hit[kHits];             // improved vertices
    uint8_t from[kHits];            // the segment that improved them
};

// kFlat: the ranges of a round are scanned as one sequence by the whole wave (expand), from the
// start or once the wave has met a hub; else, and until then, one range per lane (lane_scan).
template <int NQ, bool kFlat = true>
struct Program {
    static constexpr int kQueues = NQ;
    static constexpr int kWaveQueue = NQ == 4 ? 3 : -1;
    static constexpr bool kNoTaskwait = true;  // detached spawns only
    static constexpr uint32_t kIdleProbes = 2;
    static constexpr int kWavesPerSimd = 3;    // 3072 wavefront workers with 4 queues too (4 per SIMD measured slower)
    static constexpr int kFrameWords = 4;
    static constexpr uint32_t kMaxFunc = F_BFS;
    static constexpr uint32_t kFrameBytes = 16;
    using Args = BfsArgs;
    using WaveShared = std::conditional_t<kFlat, ExpandShared, int32_t>;
    static constexpr bool kCoop = kFlat;  // the edges of a round are scanned by run_coop
    // With one queue a wave holds few tasks while the search spreads, and batches of 32 tasks of up
    // to 64 edges spread it sooner: R-MAT 18, 64 / 32 / 16 a batch: 297 / 258 / 286 us. Ranges cut
    // smaller than that make a batch of 32 too little work for its round (R-MAT 22 in ranges of 32
    // edges, 32 / 64 a batch: 1212 / 995 us), so a batch holds 2048 edges' worth of tasks. With four
    // queues, each queue's batch is smaller anyway: R-MAT 22, 64 / 32: 1116 / 1196 us.
    __device__ __forceinline__ static uint32_t batch_cap(const Args& g) {
        if constexpr (NQ != 1) return (uint32_t)kWave;
        const uint32_t n = g.split > 0 ? (uint32_t)(2048 / g.split) : (uint32_t)kWave;
        return n < 32u ? 32u : (n > (uint32_t)kWave ? (uint32_t)kWave : n);
    }
    // A wave that has not met a hub takes full batches: with 32 a search of a large graph without
    // hubs goes deeper first and expands more vertices twice (4M vertices of 4 edges, 32 / 64 a
    // batch: 16.9 / 10.7 M tasks, 2350 / 1550 us).
    static constexpr bool kRoundCap = kFlat;
    template <class L>
    __device__ __forceinline__ static uint32_t round_cap(L& lane) {
        const bool met = ballot(lane.coop_arg) != 0ull;
        lane.coop_arg = met;  // on every lane: the next round may leave the lane that met it without a task
        return met ? batch_cap(*lane.args) : (uint32_t)kWave;
    }
    template <class L>
    __device__ __forceinline__ static void run(L& lane);
    template <class L>
    __device__ __forceinline__ static void run_coop(L& lane, uint64_t mask, WaveShared* sh);
    template <class W>
    __device__ __forceinline__ static void run_wave(W& wt);
};

template <int NQ>
__device__ __forceinline__ uint32_t route(int32_t deg) {
    if constexpr (NQ == 1) {
        return 0u;
    } else {
        return degree_bucket(deg);
    }
}

template <class P>
__device__ __forceinline__ void spawn_one(Lane<P>& t, uint32_t f, uint32_t q, const BfsArg& a) {
    __gtap_spawn_task_detached(t, f, q, a);
}
template <class P>
__device__ __forceinline__ void spawn_one(WaveTask<P>& t, uint32_t f, uint32_t q, const BfsArg& a) {
    t.spawn_detached_lane(f, q, a);
}

// Spawns the tasks of the `count` improved vertices in sh->hit, one per lane and turn. A vertex
// without out-edges needs none.
template <int NQ, class T>
__device__ __forceinline__ void spawn_hits(T& t, const BfsArgs& g, ExpandShared* sh, int32_t count) {
    const int32_t l = lane_id();
    wave_sync();
    for (int32_t b = 0; b < count; b += kWave) {
        if (b + l < count) {
            const int32_t u = lds(sh->hit)[b + l];
            const uint32_t sg = lds(sh->from)[b + l];
            const int32_t us = g.row[u], ue = g.row[u + 1];
            if (us < 0 || ue < us || (int64_t)ue > g.ne)  // malformed offsets: never read past col
                GTAP_DEVICE_ERROR(*t.dev, GTAP_ERROR_INVALID_ARGUMENT, lds(sh->task)[sg], -1, u, g.nv);
            else if (ue > us)
                spawn_one(t, F_BFS, route<NQ>(ue - us), BfsArg{u, us, ue, lds(sh->seg)[sg].nd});
        }
    }
    wave_sync();
}

// Scans a round's edges on all 64 lanes: each lane brings a range of `length` columns from
// `begin` (none: 0), whose vertices get depth nd. The ranges form one flat sequence of edges and
// lane l takes edges b + 64 j + l of it, so every lane has work until the last edges, a round
// lasts as long as its edges and not as its longest range, and loads are contiguous. (With one
// range per lane, 16 edges at a time, a round of R-MAT 22 took 22.6 us for some 700 edges, up to
// four chains of dependent loads for the longest range; now 17.3 us for 610. R-MAT 18 with one
// queue: 367 us then, 249 us now.)
//
// kWindows column loads per lane are in flight together, then their probes, then their atomics.
// A plain load of depth[u] filters the atomics: depths only decrease, so a stale cached value is
// never below the true one and can only cost an unneeded atomic.
template <int NQ, class T>
__device__ __forceinline__ void expand(T& t, const BfsArgs& g, ExpandShared* sh, int32_t begin, int32_t length,
                                       int32_t nd_own) {
    const int32_t l = lane_id();
    int32_t end = length;  // inclusive prefix sum
#pragma unroll
    for (int d = 1; d < kWave; d <<= 1) {
        const int32_t o = (int32_t)__shfl_up(end, (unsigned)d, kWave);
        if (l >= d) end += o;
    }
    const int32_t start = end - length;
    const int32_t total = shfl(end, kWave - 1);
    const bool has = length > 0;
    const uint64_t hm = ballot(has);
    if (has) {
        lds(sh->seg)[rank_in(hm)].shift = begin - start;
        lds(sh->seg)[rank_in(hm)].nd = nd_own;
        lds(sh->task)[rank_in(hm)] = t.tid;
    }
    int32_t hits = 0;
    for (int32_t b = 0; b < total; b += kWindows * kWave) {
        wave_sync();
        if (l < 2 * kWindows) lds(sh->starts)[l] = 0u;
        wave_sync();
        if (has && start >= b && start - b < kWindows * kWave)
            atomicOr(&sh->starts[(start - b) >> 5], 1u << ((start - b) & 31));
        wave_sync();
        int32_t before = popc(ballot(has && start < b));  // segments that start before the window
        int32_t u[kWindows], nd[kWindows];
        uint32_t from[kWindows / 4] = {};  // each edge's segment, 8 bits
#pragma unroll
        for (int j = 0; j < kWindows; ++j) {
            const uint64_t m = uniform((uint64_t)lds(sh->starts)[2 * j] | ((uint64_t)lds(sh->starts)[2 * j + 1] << 32));
            const int32_t r = before + rank_in(m) + (int32_t)((m >> l) & 1ull) - 1;
            before += popc(m);
            const int32_t f = b + j * kWave + l;
            const bool in = f < total;
            const uint32_t sg = in ? (uint32_t)r : 0u;
            const int32_t shift = lds(sh->seg)[sg].shift;
            nd[j] = lds(sh->seg)[sg].nd;
            from[j / 4] |= sg << (8 * (j % 4));
            u[j] = in ? g.col[f + shift] : -1;
        }
        bool bad = false;
        uint32_t bad_from = 0;
#pragma unroll
        for (int j = 0; j < kWindows; ++j) {
            if (u[j] >= g.nv || u[j] < -1) {
                bad = true;
                bad_from = from[j / 4] >> (8 * (j % 4)) & 255u;
            }
        }
        if (ballot(bad)) {
            if (bad) GTAP_DEVICE_ERROR(*t.dev, GTAP_ERROR_INVALID_ARGUMENT, lds(sh->task)[bad_from], -1, -1, g.nv);
            break;
        }
        int32_t old[kWindows];
#pragma unroll
        for (int j = 0; j < kWindows; ++j) old[j] = u[j] >= 0 ? g.depth[u[j]] : 0;
#pragma unroll
        for (int j = 0; j < kWindows; ++j) {
            if (old[j] > nd[j])
                old[j] = __hip_atomic_fetch_min(g.depth + u[j], nd[j], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
#pragma unroll
        for (int j = 0; j < kWindows; ++j) {
            const bool hit = old[j] > nd[j];
            const uint64_t m = ballot(hit);
            if (m == 0) continue;
            if (hits + popc(m) > kHits) {
                spawn_hits<NQ>(t, g, sh, hits);
                hits = 0;
            }
            if (hit) {
                lds(sh->hit)[hits + rank_in(m)] = u[j];
                lds(sh->from)[hits + rank_in(m)] = (uint8_t)(from[j / 4] >> (8 * (j % 4)));
            }
            hits += popc(m);
        }
    }
    if (hits) spawn_hits<NQ>(t, g, sh, hits);
}

// One range of up to kLaneEdges edges per lane: the column loads, the depth probes and the atomics
// of a range are issued back to back, and its improved vertices spawned one a turn. Where it is
// the better form:
// - splits of up to kShortSplit edges with one queue. The flat scan's fixed work per round (prefix
//   sum, window masks, hit list) does not pay for so few edges. Flat / per lane (us): R-MAT 22,
//   split 8: 1590 / 1370, 16: 1245 / 1106, 24: 1080 / 1070, 32: 995 / 1013; R-MAT 20, 16: 415 / 408,
//   24: 415 / 420; R-MAT 18, 8: 283 / 268, 16: 263 / 254, 24: 249 / 259;
// - large graphs without hubs, where the flat scan's rounds of equal ranges gain nothing and its
//   search expands more vertices twice. Uniform random graphs of 4M vertices and 4 / 8 / 16 edges a
//   vertex, flat with batches of 32 / per lane (us): one queue 2350 / 1455, 3180 / 1910, 3610 / 2440;
//   four queues (batches of 64) 1548 / 1438, 2200 / 1830, 3600 / 2430; 1M vertices of 16 edges 484 /
//   473 and 648 / 487. A graph is large here above 3 * 2^18 vertices with one queue (700K vertices
//   with 6 or 16 edges a vertex, their ends drawn at random: 342 / 375 and 419 / 433 us; 1M with
//   4: 409 / 397), above 2^19 with four (700K, 16: 530 / 483 us; 524K, 16: the same) and there of at
//   least 8 edges a vertex (1M, 4: 546 / 700 us). R-MAT graphs have hubs: their waves turn to the flat
//   scan within a round or two and keep its gain.
constexpr int32_t kShortSplit = 16;
template <int NQ>
constexpr int32_t kLaneEdges = NQ == 4 ? 8 : kShortSplit;  // with four queues 16 spill 20 registers, 8 spill 7
static_assert(kLaneEdges<1> >= kShortSplit, "a short range is scanned at once");
template <int NQ, class L>
__device__ __forceinline__ void lane_scan(L& lane, const BfsArgs& g, int32_t s, int32_t e, int32_t nd) {
    constexpr int32_t kC = kLaneEdges<NQ>;
    int32_t u[kC], old[kC];
#pragma unroll
    for (int j = 0; j < kC; ++j) u[j] = s + j < e ? g.col[s + j] : -1;
    bool bad = false;
#pragma unroll
    for (int j = 0; j < kC; ++j) bad |= u[j] >= g.nv || u[j] < -1;
    if (bad) {
        GTAP_DEVICE_ERROR(*lane.dev, GTAP_ERROR_INVALID_ARGUMENT, lane.tid, -1, -1, g.nv);
        return;
    }
#pragma unroll
    for (int j = 0; j < kC; ++j) old[j] = u[j] >= 0 ? g.depth[u[j]] : 0;
    uint32_t hits = 0;
#pragma unroll
    for (int j = 0; j < kC; ++j) {
        if (old[j] > nd)
            old[j] = __hip_atomic_fetch_min(g.depth + u[j], nd, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
#pragma unroll
    for (int j = 0; j < kC; ++j) hits |= (old[j] > nd ? 1u : 0u) << j;
    while (hits) {
        const int j = __builtin_ctz(hits);
        hits &= hits - 1u;
        int32_t v = u[0];
#pragma unroll
        for (int k = 1; k < kC; ++k) v = j == k ? u[k] : v;
        const int32_t us = g.row[v], ue = g.row[v + 1];
        if (us < 0 || ue < us || (int64_t)ue > g.ne)  // malformed offsets: never read past col
            GTAP_DEVICE_ERROR(*lane.dev, GTAP_ERROR_INVALID_ARGUMENT, lane.tid, -1, v, g.nv);
        else
            spawn_one(lane, F_BFS, route<NQ>(ue - us), BfsArg{v, us, ue, nd});
    }
}

template <int NQ, bool kFlat>
template <class L>
__device__ __forceinline__ void Program<NQ, kFlat>::run(L& lane) {
    const BfsArgs& g = *lane.args;
    const int32_t v = lane.template arg<int32_t>(0);
    const int32_t s = lane.template arg<int32_t>(4);
    const int32_t e = lane.template arg<int32_t>(8);
    const int32_t piece = lane.template arg<int32_t>(12) & kHubPiece;
    const int32_t d = lane.template arg<int32_t>(12) & ~kHubPiece;
    // else v was reached by a shorter path meanwhile
    if (ld32(reinterpret_cast<const int32_t*>(g.depth) + v) >= d) {
        if constexpr (kFlat) lane.coop_arg |= piece != 0 || e - s > g.hub ? 1u : 0u;
        const bool flat = kFlat && ballot(lane.coop_arg) != 0ull;
        if (e - s > g.split) {
            // up to kSplitFanout near-equal pieces, each routed by its own length
            const int64_t len = (int64_t)e - s;
            int32_t k = (int32_t)((len + g.split - 1) / g.split);
            if (k > kSplitFanout) k = kSplitFanout;
            const int32_t pd = d | (kFlat && (piece != 0 || e - s > g.hub) ? kHubPiece : 0);
            for (int32_t i = 0; i < k; ++i) {
                const int32_t ps = s + (int32_t)(len * i / k);
                const int32_t pe = s + (int32_t)(len * (i + 1) / k);
                __gtap_spawn_task_detached(lane, F_BFS, route<NQ>(pe - ps), BfsArg{v, ps, pe, pd});
            }
        } else if constexpr (kFlat) {
            if (flat) {
                lane.coop = true;  // its edges: run_coop
            } else {
                constexpr int32_t kC = kLaneEdges<NQ>;
                for (int32_t at = s; at < e; at += kC) lane_scan<NQ>(lane, g, at, e - at < kC ? e : at + kC, d + 1);
            }
        } else {
            lane_scan<NQ>(lane, g, s, e, d + 1);
        }
    }
    __gtap_finish_task(lane);
}

template <int NQ, bool kFlat>
template <class L>
__device__ __forceinline__ void Program<NQ, kFlat>::run_coop(L& lane, uint64_t mask, WaveShared* sh) {
    (void)mask;
    const int32_t s = (int32_t)lane.frame[1], nd = ((int32_t)lane.frame[3] & ~kHubPiece) + 1;
    int32_t left = lane.coop ? (int32_t)lane.frame[2] - s : 0, at = s;
    do {
        const int32_t n = left < kMaxExpand ? left : kMaxExpand;
        expand<NQ>(lane, *lane.args, sh, at, n, nd);
        at += n;
        left -= n;
    } while (NQ == 1 && ballot(left > 0));  // again with splits above kMaxExpand only
}

// The wave form of the same task (queue 3 with 4 queues): all 64 lanes enter with one (v, s, e, d).
template <int NQ, bool kFlat>
template <class W>
__device__ __forceinline__ void Program<NQ, kFlat>::run_wave(W& wt) {
    const BfsArgs& g = *wt.args;
    const int32_t v = wt.template arg<int32_t>(0);
    const int32_t s = wt.template arg<int32_t>(4);
    const int32_t e = wt.template arg<int32_t>(8);
    const int32_t d = wt.template arg<int32_t>(12) & ~kHubPiece;
    if (wt.func != F_BFS) {
        if (wt.lane == 0) GTAP_DEVICE_ERROR(*wt.dev, GTAP_ERROR_INVALID_FUNCTION, wt.tid, wt.queue, wt.func, F_BFS);
        wt.finish();
        return;
    }
    if ((int32_t)uniform((uint32_t)ld32(reinterpret_cast<const int32_t*>(g.depth) + v)) < d) {  // stale
        wt.finish();
        return;
    }
    // a scan spawns at most one task per edge in one round: an eighth of the deque capacity
    // stays within what a round may append (the deque keeps up to half its capacity published
    // and a margin free)
    const int32_t wsplit = kWaveSplitEdges < (int32_t)(wt.dev->cap / 8) ? kWaveSplitEdges : (int32_t)(wt.dev->cap / 8);
    if (e - s > wsplit) {
        // up to 64 near-equal pieces, lane i spawning piece i
        const int64_t len = (int64_t)e - s;
        int32_t k = (int32_t)((len + wsplit - 1) / wsplit);
        if (k > kWave) k = kWave;
        if (wt.lane < k) {
            const int32_t ps = s + (int32_t)(len * wt.lane / k);
            const int32_t pe = s + (int32_t)(len * (wt.lane + 1) / k);
            wt.spawn_detached_lane(F_BFS, route<NQ>(pe - ps), BfsArg{v, ps, pe, d | kHubPiece});
        }
        wt.finish();
        return;
    }
    expand<NQ>(wt, g, wt.sh, s, wt.lane == 0 ? e - s : 0, d + 1);
    wt.finish();
}

}  // namespace bfs
}  // namespace gtap

namespace gtap {
namespace bfs {

// Block-mode form (examples/asynchronous_bfs/asynchronous_bfs_block.cu:17-32): one vertex task
// runs on a whole 256-thread workgroup, thread t taking edge s + t of the vertex's range; each
// thread that lowers a neighbour's depth spawns that neighbour's task. A range longer than
// kBlockEdges is split in halves first (a workgroup invocation spawns at most kBlockMaxSpawn
// tasks; the reference walks the whole list with a stride instead).
constexpr int32_t kBlockEdges = 128;

struct BlockProgram {
    static constexpr int kFrameWords = 4;
    static constexpr uint32_t kMaxFunc = F_BFS;
    static constexpr uint32_t kFrameBytes = 16;
    using Args = BfsArgs;
    struct Shared {
        int32_t unused;
    };
    template <class B>
    __device__ __forceinline__ static void run(B& blk) {
        const BfsArgs& g = *blk.args;
        const int32_t v = blk.template arg<int32_t>(0);
        const int32_t s = blk.template arg<int32_t>(4);
        const int32_t e = blk.template arg<int32_t>(8);
        const int32_t d = blk.template arg<int32_t>(12);
        const uint32_t t = threadIdx.x;
        const bool stale = ld32(reinterpret_cast<const int32_t*>(g.depth) + v) < d;
        if (!stale) {
            if (e - s > kBlockEdges) {
                if (t == 0) {
                    const int32_t m = s + (e - s) / 2;
                    blk.spawn_detached(F_BFS, BfsArg{v, s, m, d});
                    blk.spawn_detached(F_BFS, BfsArg{v, m, e, d});
                }
            } else if ((int32_t)t < e - s) {
                const int32_t u = g.col[s + (int32_t)t];
                if (u < 0 || u >= g.nv) {
                    GTAP_DEVICE_ERROR(*blk.dev, GTAP_ERROR_INVALID_ARGUMENT, blk.tid, -1, u, g.nv);
                } else if (g.depth[u] > d + 1 &&
                           __hip_atomic_fetch_min(g.depth + u, d + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) > d + 1) {
                    const int32_t us = g.row[u], ue = g.row[u + 1];
                    if (us < 0 || ue < us || (int64_t)ue > g.ne)
                        GTAP_DEVICE_ERROR(*blk.dev, GTAP_ERROR_INVALID_ARGUMENT, blk.tid, -1, u, g.nv);
                    else
                        blk.spawn_detached(F_BFS, BfsArg{u, us, ue, d + 1});
                }
            }
        }
        blk.finish();
    }
};
static_assert(kBlockEdges <= (int32_t)kBlockMaxSpawn, "one invocation spawns at most kBlockMaxSpawn tasks");

}  // namespace bfs
}  // namespace gtap

using Bfs1 = gtap::bfs::Program<1>;
using Bfs1Short = gtap::bfs::Program<1, false>;
using Bfs4 = gtap::bfs::Program<4>;

namespace {

__global__ void bfs_init_depth(int32_t* depth, int32_t nv, int32_t source) {
    const int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t v = i; v < nv; v += stride) depth[v] = (v == source) ? 0 : 0x3f3f3f3f;
}

}  // namespace

// BFS from `source` over a CSR graph already in device memory (row: nv+1 int32 offsets,
// col: ne int32 columns). depth (nv int32, device) receives the hop counts, 0x3f3f3f3f for
// unreached vertices. num_queues = 1 (no EPAQ) or 4 (EPAQ by out-degree bucket).
// Replaces the program of examples/asynchronous_bfs/asynchronous_bfs_thread.cu:51-141.
extern "C" int gtap_bfs(const int32_t* row, const int32_t* col, int32_t nv, int64_t ne, int32_t source,
                        int32_t* depth, int32_t num_queues, int32_t split, gtap_run_stats* stats) {
    using namespace gtap;
    if (!row || !col || !depth || nv <= 0 || source < 0 || source >= nv || ne < 0)
        return host::invalid_argument("gtap_bfs: bad graph arguments");
    if (num_queues != 1 && num_queues != 4) return host::invalid_argument("gtap_bfs: num_queues must be 1 or 4");
    if (split <= 0) split = 64;
    host::Runtime& R = host::rt();
    if (!R.initialized) {
        int st = gtap_initialize();
        if (st) return st;
    }
    hipLaunchKernelGGL(bfs_init_depth, dim3(1024), dim3(256), 0, R.stream, depth, nv, source);
    GTAP_HIP_TRY(hipGetLastError());
    int32_t rs[2];
    GTAP_HIP_TRY(hipMemcpy(rs, row + source, 2 * sizeof(int32_t), hipMemcpyDeviceToHost));
    if (rs[0] < 0 || rs[1] < rs[0] || (int64_t)rs[1] > ne) return host::invalid_argument("gtap_bfs: bad source row offsets");
    bfs::BfsArg root{source, rs[0], rs[1], 0};
    const uint32_t q = (num_queues == 4) ? bfs::degree_bucket(rs[1] - rs[0]) : 0u;
    gtap_job job = host::make_job(bfs::F_BFS, q, &root, sizeof(root));
    bfs::BfsArgs a{row, col, depth, nv, split, ne, -1};
    // Large graphs may have no hubs (lane_scan): a range is one where degrees drawn at random around
    // the mean would hardly ever reach.
    const double mean = (double)ne / nv;
    if (nv > (num_queues == 1 ? 3 << 18 : 1 << 19) && (num_queues == 1 || mean >= 8.0)) {
        a.hub = (int32_t)std::min(mean + 6.0 * std::sqrt(mean) + 8.0, 1e9);
    }
    if (num_queues == 4) return host::run_single_job<Bfs4>(a, job, nullptr, stats, GTAP_TERM_QUIESCE);
    if (split <= bfs::kShortSplit) return host::run_single_job<Bfs1Short>(a, job, nullptr, stats, GTAP_TERM_QUIESCE);
    return host::run_single_job<Bfs1>(a, job, nullptr, stats, GTAP_TERM_QUIESCE);
}

// The block-mode BFS (one vertex task per 256-thread workgroup) over a CSR graph in device
// memory; same arguments and result as gtap_bfs. Replaces the program of
// examples/asynchronous_bfs/asynchronous_bfs_block.cu:17-37.
extern "C" int gtap_bfs_block(const int32_t* row, const int32_t* col, int32_t nv, int64_t ne, int32_t source,
                              int32_t* depth, gtap_run_stats* stats) {
    using namespace gtap;
    if (!row || !col || !depth || nv <= 0 || source < 0 || source >= nv || ne < 0)
        return host::invalid_argument("gtap_bfs_block: bad graph arguments");
    host::Runtime& R = host::rt();
    if (!R.initialized) {
        int st = gtap_initialize();
        if (st) return st;
    }
    hipLaunchKernelGGL(bfs_init_depth, dim3(1024), dim3(256), 0, R.stream, depth, nv, source);
    GTAP_HIP_TRY(hipGetLastError());
    int32_t rs[2];
    GTAP_HIP_TRY(hipMemcpy(rs, row + source, 2 * sizeof(int32_t), hipMemcpyDeviceToHost));
    if (rs[0] < 0 || rs[1] < rs[0] || (int64_t)rs[1] > ne)
        return host::invalid_argument("gtap_bfs_block: bad source row offsets");
    bfs::BfsArg root{source, rs[0], rs[1], 0};
    gtap_job job = host::make_job(bfs::F_BFS, 0, &root, sizeof(root));
    bfs::BfsArgs a{row, col, depth, nv, 0, ne, 0};
    return host::run_single_block_job<bfs::BlockProgram>(a, job, nullptr, stats, GTAP_TERM_QUIESCE);
}

// Host-pointer convenience: copies the CSR in, runs gtap_bfs, copies depth out.
extern "C" int gtap_bfs_host(const int32_t* row, const int32_t* col, int32_t nv, int64_t ne, int32_t source,
                             int32_t* depth_out, int32_t num_queues, int32_t split, gtap_run_stats* stats) {
    if (!row || !col || !depth_out || nv <= 0 || ne < 0) return gtap::host::invalid_argument("gtap_bfs_host");
    if (int st = gtap::host::check_csr_rows(row, nv, ne, "gtap_bfs_host")) return st;
    int32_t *drow = nullptr, *dcol = nullptr, *ddep = nullptr;
    GTAP_HIP_TRY(hipMalloc(&drow, (size_t)(nv + 1) * sizeof(int32_t)));
    GTAP_HIP_TRY(hipMalloc(&dcol, (size_t)(ne > 0 ? ne : 1) * sizeof(int32_t)));
    GTAP_HIP_TRY(hipMalloc(&ddep, (size_t)nv * sizeof(int32_t)));
    int st = 0;
    hipError_t e = hipMemcpy(drow, row, (size_t)(nv + 1) * sizeof(int32_t), hipMemcpyHostToDevice);
    if (e == hipSuccess && ne > 0) e = hipMemcpy(dcol, col, (size_t)ne * sizeof(int32_t), hipMemcpyHostToDevice);
    if (e != hipSuccess) st = gtap::host::hip_status(e, "gtap_bfs_host copy-in");
    if (!st) st = gtap_bfs(drow, dcol, nv, ne, source, ddep, num_queues, split, stats);
    if (!st) {
        e = hipMemcpy(depth_out, ddep, (size_t)nv * sizeof(int32_t), hipMemcpyDeviceToHost);
        if (e != hipSuccess) st = gtap::host::hip_status(e, "gtap_bfs_host copy-out");
    }
    (void)hipFree(drow);
    (void)hipFree(dcol);
    (void)hipFree(ddep);
    return st;
}
