// prog_nq.hip -- n-queens as a thread-executed task program.
//
// Source program (the task shape of the reference's evaluation/2-comparison/nq/gtap_nq.cu:25-55,
// with no cutoff and with every count returned to the parent through a taskwait and an
// int64 sum instead of a global atomicAdd):
//
//   #pragma gtap function
//   __device__ int64_t nq(int row, uint32_t cols, uint32_t diag, uint32_t anti) {
//       if (row == N) return 1;
//       uint32_t avail = mask & ~(cols | diag | anti);
//       int64_t counts[16]; int k = 0;
//       while (avail) {
//           uint32_t p = avail & -avail; avail -= p;
//           #pragma gtap task
//           counts[k++] = nq(row + 1, cols | p, (diag | p) << 1, (anti | p) >> 1);
//       }
//       #pragma gtap taskwait
//       int64_t s = 0; for (int i = 0; i < k; ++i) s += counts[i];
//       return s;
//   }
//
// Two lowerings of this program:
//  * additive join (Program, the default): the counts are only summed after the taskwait,
//    so each child adds its count to the parent's join word with the atomic that counts the
//    join down; frame = { int32 row; uint32 cols, diag, anti; }, the parent resumes with
//    the sum.
//  * result slots (SlotProgram): frame = { int32 row; uint32 cols, diag, anti; int32 k;
//    int32 pad[3]; int64 counts[16]; }; each child stores its count into counts[i], then
//    counts the join down. The first six words (the arguments and k) are loaded when the
//    task starts, so the resumed task knows k without another load; counts[] is 16-byte
//    aligned and read two at a time.
#include "../device/gtap_abi.hpp"
#include "../host/gtap_launch.hpp"

namespace gtap {
namespace nq {

enum : uint32_t { F_NQ = 1 };
struct NqArg {
    int32_t row;
    uint32_t cols;
    uint32_t diag;
    uint32_t anti;
};
constexpr int kOffK = 16;
constexpr int kOffCounts = 32;
constexpr int kMaxN = 16;

template <bool kSum>
struct ProgramT {
    static constexpr int kQueues = 1;
    // the default form is also built with the global-queue and Chase-Lev schedulers
    static constexpr bool kSchedVariants = kSum;
    static constexpr bool kCoop = kSum;  // a round's children are spawned by run_coop
    static constexpr int kWavesPerSimd = kSum ? 4 : 1;
    static constexpr int kFrameWords = kSum ? 4 : 6;  // row, cols, diag, anti (, k, pad)
    static constexpr uint32_t kMaxFunc = F_NQ;
    static constexpr uint32_t kFrameBytes = kSum ? 16 : kOffCounts + 8 * kMaxN;
    struct Args {
        int32_t n;
    };
    template <class L>
    __device__ __forceinline__ static void run(L& lane);
    template <class L, class S>
    __device__ __forceinline__ static void run_coop(L& lane, uint64_t mask, S* sh);
};
using Program = ProgramT<true>;
using SlotProgram = ProgramT<false>;

template <bool kSum, class L>
__device__ __forceinline__ void nq_task(L& lane) {
    const int32_t N = lane.args->n;
    switch (__gtap_get_task_state(lane)) {
        case 0: {
            const int32_t row = lane.template arg<int32_t>(0);
            const uint32_t cols = lane.template arg<uint32_t>(4);
            const uint32_t diag = lane.template arg<uint32_t>(8);
            const uint32_t anti = lane.template arg<uint32_t>(12);
            if (row == N) {
                __gtap_return(lane, (int64_t)1);
                return;
            }
            const uint32_t mask = (N < 32) ? ((1u << N) - 1u) : 0xFFFFFFFFu;
            uint32_t avail = mask & ~(cols | diag | anti);
            int32_t k = 0;
            if constexpr (kSum) {
                k = popc32(avail);
                lane.coop = k != 0;  // the children: run_coop
                lane.coop_arg = avail;
                lane.will_spawn_sum((uint32_t)k);
            } else {
                while (avail) {
                    const uint32_t p = avail & (0u - avail);
                    avail -= p;
                    const NqArg child{row + 1, cols | p, (diag | p) << 1, (anti | p) >> 1};
                    __gtap_spawn_task(lane, F_NQ, 0, kOffCounts + 8 * k, child);
                    ++k;
                }
            }
            if (k == 0) {  // dead end: no legal column in this row
                __gtap_return(lane, (int64_t)0);
                return;
            }
            if constexpr (kSum) {
                if (__gtap_set_state_for_join_sum(lane, 1, 0)) return;
            } else {
                lane.template frame_st<int32_t>(kOffK, k);
                if (__gtap_set_state_for_join(lane, 1, 0)) return;
            }
        }
            [[fallthrough]];
        case 1: {
            if constexpr (kSum) {
                __gtap_return(lane, __gtap_get_join_sum(lane));
            } else {
                const int32_t k = lane.template arg<int32_t>(kOffK);
                int64_t s = 0;
                for (int32_t i = 0; i < k; i += 2) {
                    int64_t a, b;
                    lane.template frame_ld2<int64_t>(kOffCounts + 8 * i, a, b);
                    s += a + (i + 1 < k ? b : 0);
                }
                __gtap_return(lane, s);
            }
            return;
        }
        default:
            GTAP_DEVICE_ERROR(*lane.dev, GTAP_ERROR_INVALID_TASKWAIT, lane.tid, 0, lane.state, 1);
            lane.finish();
            return;
    }
}

template <bool kSum>
template <class L>
__device__ __forceinline__ void ProgramT<kSum>::run(L& lane) {
    nq_task<kSum>(lane);
}

// One child per free column of the task's row, lowest first.
template <bool kSum>
template <class L, class S>
__device__ __forceinline__ void ProgramT<kSum>::run_coop(L& lane, uint64_t mask, S* sh) {
    (void)mask;
    (void)sh;
    uint32_t avail = lane.coop ? lane.coop_arg : 0u;
    const int32_t row = (int32_t)lane.frame[0];
    const uint32_t cols = lane.frame[1], diag = lane.frame[2], anti = lane.frame[3];
    spawn_round<ProgramT<kSum>, 0, true, NqArg>(lane, (uint32_t)popc32(avail), [&](uint32_t) {
        const uint32_t p = avail & (0u - avail);
        avail -= p;
        return NqArg{row + 1, cols | p, (diag | p) << 1, (anti | p) >> 1};
    });
}

}  // namespace nq
}  // namespace gtap

namespace gtap {
namespace nq {

// The reference's evaluation program at its own settings (evaluation/2-comparison/nq/
// gtap_nq.cu:10-56): tasks down to row `cutoff`, a sequential search below it, detached
// spawns (no taskwait) and one count. The sequential search here is a depth-first walk; each
// lane sums the counts of its tasks, and the sums leave with the wave's statistics at the end
// of the launch. (The reference adds 1 per solution to one int32. Adding each task's count to
// one word was bound by that word's line: n = 14 took 752 us, against 500 us without.) Unlike
// the reference, a task that reaches row N counts a solution even above the cutoff, so
// N <= cutoff + 1 is also correct.
struct CutoffArgs {
    int32_t n;
    int32_t cutoff;
};

// A lane's share of the sequential search: a depth-first walk that lives in registers. The two
// diagonal sets are kept in board coordinates (bit col - row + n - 1 and bit col + row, at most
// bit 30 for n <= 16), so a step back is the same exclusive or as the step forward, and the
// columns of the path are 4 bits each in one 64-bit word: no stack in memory (with one, as four
// private arrays, every step waited for scratch memory and the walks of a round took 113 us at
// n = 15). The walk starts at `base` with the columns `rem` of that row to try, and may lose some of
// those it has not come to (another lane takes them). Placements in row n - 2 are not stepped
// into: the last row's free columns are counted from there.
struct Walk {
    uint32_t cols, dl, dr, avail, rem;
    uint64_t path;
    int32_t r, base;

    __device__ __forceinline__ bool active() const { return avail != 0u || r != base; }
    __device__ __forceinline__ void start(int32_t row, uint32_t c, uint32_t l, uint32_t d, uint32_t todo) {
        base = r = row;
        cols = c;
        dl = l;
        dr = d;
        rem = avail = todo;
        path = 0;
    }
    // One placement or one step back; returns the solutions it counted.
    __device__ __forceinline__ int32_t step(int32_t top, uint32_t mask) {
        const bool fwd = avail != 0u;
        const int32_t at = fwd ? r : r - 1;  // the row whose queen is placed or taken back
        const uint32_t c = fwd ? (uint32_t)__builtin_ctz(avail | 0x80000000u) : (uint32_t)path & 15u;
        const uint32_t p = 1u << c;
        const uint32_t cols1 = cols ^ p, dl1 = dl ^ (p << (top - at)), dr1 = dr ^ (p << at);
        const int32_t r1 = fwd ? r + 1 : at;
        const uint32_t free1 = mask & ~(cols1 | (dl1 >> (top - r1)) | (dr1 >> r1));
        rem = fwd && at == base ? rem ^ p : rem;
        if (fwd && r1 == top) {
            avail ^= p;
            return popc32(free1);
        }
        cols = cols1;
        dl = dl1;
        dr = dr1;
        r = r1;
        path = fwd ? (path << 4) | c : path >> 4;
        avail = fwd ? free1 : (r1 == base ? rem : free1 & (~1u << c));
        return 0;
    }
};
constexpr int kWalkSteps = 4;   // steps between two looks at the idle lanes
// Idle lanes that make the busy ones share: N = 14, 8 / 16 / 24: 429 / 415 / 411 us; N = 15: 1154 / 1147 /
// 1162 us (without sharing 465 and 1438 us).
constexpr int kWalkIdle = 16;

struct CutoffProgram {
    static constexpr int kQueues = 1;
    static constexpr bool kNoTaskwait = true;
    static constexpr uint32_t kIdleProbes = 2;
    static constexpr bool kLaneSum = true;
    static constexpr bool kCoop = true;  // children and searches: run_coop
    static constexpr int kWavesPerSimd = 4;
    static constexpr int kFrameWords = 4;  // row, cols, left, right
    static constexpr uint32_t kMaxFunc = F_NQ;
    static constexpr uint32_t kFrameBytes = 16;
    using Args = CutoffArgs;
    struct WaveShared {
        int32_t lane[kWave];  // the lanes that give a column away
    };
    template <class L>
    __device__ __forceinline__ static void run(L& lane) {
        const CutoffArgs& g = *lane.args;
        const int32_t row = lane.template arg<int32_t>(0);
        const uint32_t cols = lane.template arg<uint32_t>(4);
        const uint32_t left = lane.template arg<uint32_t>(8);
        const uint32_t right = lane.template arg<uint32_t>(12);
        const uint32_t avail = ((1u << g.n) - 1u) & ~(cols | left | right);
        if (row == g.n) {
            lane.total += 1u;
        } else if (row == g.n - 1 && row > g.cutoff) {
            lane.total += (uint32_t)popc32(avail);
        } else {
            lane.coop = avail != 0u;  // the children, or the search: run_coop
            lane.coop_arg = avail;
        }
        __gtap_finish_task(lane);
    }
    // Rows up to the cutoff: a child task per free column. Below it: the round's searches, on all
    // lanes. Their lengths differ (a mean of 50 steps and a longest of 134 in a round at n = 15,
    // cutoff 7), so once kWalkIdle lanes have nothing to do, each takes one of the first row's
    // columns that a busy lane has not come to.
    template <class L>
    __device__ __forceinline__ static void run_coop(L& lane, uint64_t mask, WaveShared* sh) {
        (void)mask;
        const CutoffArgs& g = *lane.args;
        const int32_t l = lane_id();
        const int32_t row = (int32_t)lane.frame[0];
        const uint32_t cols = lane.frame[1], left = lane.frame[2], right = lane.frame[3];
        const bool walks = lane.coop && row > g.cutoff;
        uint32_t avail = lane.coop && !walks ? lane.coop_arg : 0u;
        if (ballot(avail != 0u)) {
            spawn_round<CutoffProgram, 0, false, NqArg>(lane, (uint32_t)popc32(avail), [&](uint32_t) {
                const uint32_t p = avail & (0u - avail);
                avail -= p;
                return NqArg{row + 1, cols | p, (left | p) << 1, (right | p) >> 1};
            });
        }
        if (ballot(walks) == 0) return;
        const int32_t top = g.n - 1;
        const uint32_t board = (1u << g.n) - 1u;
        Walk w;
        w.start(0, 0u, 0u, 0u, 0u);
        uint32_t bc = 0, bl = 0, bd = 0;  // the board that w starts from
        if (walks) {
            bc = cols;
            bl = (left & board) << (top - row);
            bd = (right & board) << row;
            w.start(row, bc, bl, bd, lane.coop_arg);
        }
        uint32_t found = 0;
        while (true) {
#pragma unroll 1
            for (int k = 0; k < kWalkSteps; ++k)
                if (w.active()) found += (uint32_t)w.step(top, board);
            const uint64_t idle = ballot(!w.active());
            if (idle == ~0ull) break;
            if (popc(idle) < kWalkIdle) continue;
            const bool gives = w.active() && (w.r > w.base ? w.rem != 0u : (w.rem & (w.rem - 1u)) != 0u);
            const uint64_t donors = ballot(gives);
            if (donors == 0) continue;
            const int32_t pairs = popc(idle) < popc(donors) ? popc(idle) : popc(donors);
            const int32_t rank = w.active() ? rank_in(donors) : rank_in(idle);
            uint32_t part = 0;  // the column given away: the last one
            if (gives && rank < pairs) {
                part = 1u << (31 - __builtin_clz(w.rem));
                w.rem ^= part;
                if (w.r == w.base) w.avail = w.rem;
                lds(sh->lane)[rank] = l;
            }
            wave_sync();
            const bool takes = !w.active() && rank < pairs;
            const int32_t src = takes ? lds(sh->lane)[rank] : l;
            const uint32_t c1 = shfl(bc, src), l1 = shfl(bl, src), d1 = shfl(bd, src);
            const uint32_t what = shfl(part | ((uint32_t)w.base << 16), src);
            if (takes) {
                bc = c1;
                bl = l1;
                bd = d1;
                w.start((int32_t)(what >> 16), bc, bl, bd, what & 0xFFFFu);
            }
            wave_sync();
        }
        lane.total += found;
    }
};

}  // namespace nq
}  // namespace gtap

using NqProgram = gtap::nq::Program;
using NqSlotProgram = gtap::nq::SlotProgram;
static_assert(NqSlotProgram::kFrameBytes + gtap::kHdrBytes <= gtap::host::kBuiltinStride, "frame exceeds stride");

// Counts the n-queens placements of an n x n board as one persistent launch
// (reference program: evaluation/2-comparison/nq/gtap_nq.cu:57-99).
extern "C" int gtap_nqueens(int n, int64_t* result, gtap_run_stats* stats) {
    if (n < 1 || n > gtap::nq::kMaxN) return gtap::host::invalid_argument("gtap_nqueens: n must be in [1, 16]");
    gtap::nq::NqArg root{0, 0u, 0u, 0u};
    gtap_job job = gtap::host::make_job(gtap::nq::F_NQ, 0, &root, sizeof(root));
    int64_t r = 0;
    int st = gtap::host::run_single_job<NqProgram>(NqProgram::Args{n}, job, &r, stats, GTAP_TERM_JOBS);
    if (st == 0 && result) *result = r;
    return st;
}

// The same count with the result-slot join (each child stores its count into the parent's
// frame, then counts the join down), the form a slot-per-call lowering produces; work-
// stealing scheduler only.
extern "C" int gtap_nqueens_slots(int n, int64_t* result, gtap_run_stats* stats) {
    if (n < 1 || n > gtap::nq::kMaxN) return gtap::host::invalid_argument("gtap_nqueens_slots: n must be in [1, 16]");
    gtap::nq::NqArg root{0, 0u, 0u, 0u};
    gtap_job job = gtap::host::make_job(gtap::nq::F_NQ, 0, &root, sizeof(root));
    int64_t r = 0;
    int st = gtap::host::run_single_job<NqSlotProgram>(NqSlotProgram::Args{n}, job, &r, stats, GTAP_TERM_JOBS);
    if (st == 0 && result) *result = r;
    return st;
}

// The reference's n-queens benchmark at its own settings (evaluation/2-comparison/nq/
// gtap_nq.cu:57-99): tasks for rows 0..cutoff (the reference's default 7), a sequential search
// below, no taskwait, one count. Returns the solution count in *result.
extern "C" int gtap_nqueens_cutoff(int n, int cutoff, int64_t* result, gtap_run_stats* stats) {
    using namespace gtap;
    if (n < 1 || n > nq::kMaxN || cutoff < 0) return host::invalid_argument("gtap_nqueens_cutoff: n in [1, 16], cutoff >= 0");
    host::Runtime& R = host::rt();
    if (!R.initialized) {
        int st = gtap_initialize();
        if (st) return st;
    }
    nq::NqArg root{0, 0u, 0u, 0u};
    gtap_job job = host::make_job(nq::F_NQ, 0, &root, sizeof(root));
    int st = host::run_single_job<gtap::nq::CutoffProgram>(nq::CutoffArgs{n, cutoff}, job, nullptr, stats,
                                                            GTAP_TERM_QUIESCE);
    if (st) return st;
    if (result) *result = (int64_t)R.summary->sums[ST_PROGRAM];
    return 0;
}
