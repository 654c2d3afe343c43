// prog_spmv.hip -- divide-and-conquer sparse matrix-vector product y = A x (CSR, float64) as
// a thread-executed task program.
//
// Source program (the task shape of the reference's examples/spmv/spmv_thread.cu:34-66):
//
//   #pragma gtap function
//   __device__ void spmv_row(int i) {
//       double sum = 0.0;
//       for (int k = row_ptr[i]; k < row_ptr[i + 1]; ++k) sum = fma(val[k], x[col_idx[k]], sum);
//       y[i] = sum;
//   }
//   #pragma gtap function
//   __device__ void range_spmv(int begin, int end) {          // (in 4 pieces here)
//       if (end - begin <= CUTOFF) {
//           for (int i = begin; i < end; ++i) {
//               #pragma gtap task
//               spmv_row(i);
//           }
//       } else {
//           int mid = (begin + end) >> 1;
//           #pragma gtap task
//           range_spmv(begin, mid);
//           #pragma gtap task
//           range_spmv(mid, end);
//       }
//   }
//
// All spawns are detached (no taskwait); the launch ends by quiescence. The row sum is an
// explicit fused multiply-add chain in column order, so the result is the same bit pattern
// as a sequential fma loop over the row on any device (the reference writes `sum += v * x`,
// which a compiler may or may not contract).
#include <algorithm>
#include <cstring>
#include <thread>
#include <vector>

#include "../device/gtap_abi.hpp"
#include "../device/gtap_steps.hpp"
#include "../host/gtap_launch.hpp"

namespace gtap {
namespace spmv {

enum : uint32_t { F_RANGE = 1, F_ROW = 2 };
struct RangeArg {
    int32_t begin;
    int32_t end;
};
struct SpmvArgs {
    const int32_t* row_ptr;
    const int32_t* col_idx;
    const double* val;
    const double* x;
    double* y;
    int32_t rows;
    int32_t cols;
    int32_t cutoff;
    uint32_t batch;   // most tasks a wave takes at once
    int32_t fan;      // pieces a range is cut into
    int32_t nnz;  // row_ptr[rows]: a row's offsets must satisfy 0 <= row_ptr[i] <= row_ptr[i+1] <= nnz
};

constexpr int kPer = 8;        // entries of a row that a lane loads in one step
constexpr int kGroup = 8;      // most lanes per row while there are rows for all lanes
constexpr int kRowBegin = 2;   // frame words a row task keeps its offsets in
constexpr int kRowLength = 3;
typedef double Entry __attribute__((ext_vector_type(2)));  // a value and its x entry

struct Program {
    static constexpr int kQueues = 1;
    static constexpr bool kNoTaskwait = true;  // detached spawns only
    static constexpr uint32_t kIdleProbes = 2;
    static constexpr bool kCoop = true;        // the rows of a round are summed by run_coop
    static constexpr int kWavesPerSimd = 2;    // what the tile's LDS allows; 3 with kPer = 4: 4.26 against 4.01 ms
    static constexpr int kFrameWords = 2;      // begin, end (a row task uses begin)
    static constexpr uint32_t kMaxFunc = F_ROW;
    static constexpr uint32_t kFrameBytes = 16;
    using Args = SpmvArgs;
    struct WaveShared {
        Entry tile[kWave * kPer + kWave];  // kWave / g rows of kPer * g entries, each row padded by one
        int32_t src[kWave];                // lanes that hold the round's rows
    };
    __device__ __forceinline__ static uint32_t batch_cap(const Args& a) { return a.batch; }
    template <class L>
    __device__ __forceinline__ static void run(L& lane);
    template <class L>
    __device__ __forceinline__ static void run_coop(L& lane, uint64_t mask, WaveShared* sh);
};

// A row task checks its row's offsets and leaves the entries to run_coop.
template <class L>
__device__ __forceinline__ void row_task(L& lane) {
    const SpmvArgs& g = *lane.args;
    const int32_t i = lane.template arg<int32_t>(0);
    if (i < 0 || i >= g.rows) {
        GTAP_DEVICE_ERROR(*lane.dev, GTAP_ERROR_INVALID_ARGUMENT, lane.tid, -1, i, g.rows);
        __gtap_finish_task(lane);
        return;
    }
    const int32_t kb = g.row_ptr[i], ke = g.row_ptr[i + 1];
    if (kb < 0 || ke < kb || ke > g.nnz) {  // malformed offsets: never read past col_idx / val
        GTAP_DEVICE_ERROR(*lane.dev, GTAP_ERROR_INVALID_ARGUMENT, lane.tid, -1, i, g.nnz);
        __gtap_finish_task(lane);
        return;
    }
    lane.frame[kRowBegin] = (uint32_t)kb;
    lane.frame[kRowLength] = (uint32_t)(ke - kb);
    lane.coop = true;
    __gtap_finish_task(lane);
}

template <class L>
__device__ __forceinline__ void range_task(L& lane) {
    const SpmvArgs& g = *lane.args;
    const int32_t begin = lane.template arg<int32_t>(0);
    const int32_t end = lane.template arg<int32_t>(4);
    if (end - begin <= g.cutoff) {
        for (int32_t i = begin; i < end; ++i) __gtap_spawn_task_detached(lane, F_ROW, 0, RangeArg{i, 0});
    } else {
        const int64_t len = (int64_t)end - begin;
        for (int32_t i = 0; i < g.fan; ++i) {
            const int32_t ps = begin + (int32_t)(len * i / g.fan), pe = begin + (int32_t)(len * (i + 1) / g.fan);
            if (pe > ps) __gtap_spawn_task_detached(lane, F_RANGE, 0, RangeArg{ps, pe});
        }
    }
    __gtap_finish_task(lane);
}

// The entries of the kPer * g of a row's entries that one step takes: this lane's columns and
// values, entry j at offset first + j * g of a row of `length` entries from `begin`.
__device__ __forceinline__ void load_entries(const SpmvArgs& a, int32_t begin, uint32_t length, uint32_t first, uint32_t g,
                                             int32_t (&c)[kPer], double (&v)[kPer]) {
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const uint32_t e = first + (uint32_t)j * g;
        c[j] = e < length ? __builtin_nontemporal_load(a.col_idx + begin + e) : -1;
        v[j] = e < length ? __builtin_nontemporal_load(a.val + begin + e) : 0.0;
    }
}

// The rows of a round on all 64 lanes. One lane per row reads 64 separate lines with every
// load, uses 4 or 8 bytes of each and has lost them from the caches when it comes back, and a
// round lasts as long as its longest row: 6.6 ms for 1M rows of 300 entries (345 M lines from
// beyond the L2). Here g lanes load a row's entries together, kPer each per step: whole lines of
// columns and values are used at once and not kept (non-temporal), and the entries
// {value, x[column]} go through LDS to one lane per row, which runs the row's chain of fused
// multiply-adds in column order, so the sum has the same bits. g is the smallest power of two
// with kPer * g entries for the longest row, at most kGroup (4 / 8 / 16 with full batches: 4.55 /
// 4.01 / 3.95 ms at 300 entries a row, 409 / 395 / 428 us at 100) unless fewer rows leave lanes
// free. 3.72 ms, 1.02 TB/s of matrix: bound by the gathers of x (8 MB against 4 MB of L2 per
// XCD), 215 M lines at 58 G/s, about the rate of random reads that miss the L2 on this chip.
template <class L>
__device__ __forceinline__ void Program::run_coop(L& lane, uint64_t mask, WaveShared* sh) {
    const SpmvArgs& a = *lane.args;
    const int32_t l = lane_id();
    const int32_t m = popc(mask);
    int32_t longest = lane.coop ? (int32_t)lane.frame[kRowLength] : 0;
#pragma unroll
    for (int d = kWave / 2; d > 0; d >>= 1) {
        const int32_t o = shfl(longest, l ^ d);
        longest = o > longest ? o : longest;
    }
    int32_t g = 1;
    while (kPer * g < longest && (g < kGroup || 2 * g * m <= kWave) && g < kWave) g <<= 1;
    if (lane.coop) lds(sh->src)[rank_in(mask)] = l;
    wave_sync();
    const int32_t rows = kWave / g, step = kPer * g, stride = step + 1;
    const int32_t slot = l / g, sub = l & (g - 1);
    const uint32_t width = (uint32_t)g;
    lds_array<Entry> tile = lds(sh->tile);
    // The steps of all groups in one sequence, the next step's columns and values in flight
    // while the current one gathers and sums, over the end of a group too.
    int32_t p0 = 0;              // current step: the group's first row (of the m)
    int32_t begin;               // this lane loads entries sub, sub + g, ... of a step of row p0 + slot
    Steps load{0u, (uint32_t)step, 0u};
    int32_t row;                 // and, among the first `rows` lanes, sums a step of row p0 + l
    Steps add{0u, (uint32_t)step, 0u};
    bool sums;
    auto load_part = [&](int32_t p) {
        const bool on = p + slot < m;
        const int32_t src = lds(sh->src)[on ? p + slot : 0];
        begin = shfl((int32_t)lane.frame[kRowBegin], src);
        const uint32_t length = shfl(lane.frame[kRowLength], src);
        load.n = on ? length : 0u;
    };
    auto sum_part = [&](int32_t p) {
        sums = l < rows && p + l < m;
        const int32_t own = lds(sh->src)[sums ? p + l : 0];
        row = shfl((int32_t)lane.frame[0], own);
        const uint32_t length = shfl(lane.frame[kRowLength], own);
        add.n = sums ? length : 0u;
        add.at = 0u;
    };
    load_part(0);
    sum_part(0);
    double sum = 0.0;
    int32_t c[kPer];
    double v[kPer];
    load_entries(a, begin, load.n, (uint32_t)sub, width, c, v);
    while (true) {
        double xv[kPer];
        bool bad = false;
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const bool in = load.at + (uint32_t)j * width + (uint32_t)sub < load.n;
            const bool valid = (uint32_t)c[j] < (uint32_t)a.cols;
            bad |= in && !valid;
            xv[j] = in && valid ? a.x[c[j]] : 0.0;
        }
        if (ballot(bad)) {
            const int32_t src = lds(sh->src)[p0 + slot < m ? p0 + slot : 0];
            const int32_t bad_row = shfl((int32_t)lane.frame[0], src), bad_task = shfl((int32_t)lane.tid, src);
            if (bad) GTAP_DEVICE_ERROR(*lane.dev, GTAP_ERROR_INVALID_ARGUMENT, bad_task, -1, bad_row, a.cols);
        }
        const bool more = ballot(load.more()) != 0;
        load.at = more ? load.at + load.step : 0u;
        const int32_t p1 = more ? p0 : p0 + rows;
        if (!more && p1 < m) load_part(p1);
        int32_t c1[kPer];
        double v1[kPer];
        if (p1 < m) load_entries(a, begin, load.n, load.at + (uint32_t)sub, width, c1, v1);
        wave_sync();  // the previous step's entries have been read
#pragma unroll
        for (int j = 0; j < kPer; ++j) tile[slot * stride + j * g + sub] = Entry{v[j], xv[j]};
        wave_sync();
        // signed, so that the tile's addresses fold into one base (200003 rows of 100: 313 against 326 us)
        const int32_t left = (int32_t)(add.more() ? add.step : add.left());
        for (int32_t e = 0; e < left; e += kPer) {
            Entry t[kPer];
#pragma unroll
            for (int j = 0; j < kPer; ++j) t[j] = tile[l * stride + e + j];
#pragma unroll
            for (int j = 0; j < kPer; ++j)
                if (e + j < left) sum = __builtin_fma(t[j].x, t[j].y, sum);
        }
        add.next();
        if (!more) {
            if (sums) a.y[row] = sum;
            if (p1 >= m) break;
            sum = 0.0;
            sum_part(p1);
        }
        p0 = p1;
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            c[j] = c1[j];
            v[j] = v1[j];
        }
    }
}

template <class L>
__device__ __forceinline__ void Program::run(L& lane) {
    if (lane.func == F_ROW) row_task(lane);
    else range_task(lane);
}

}  // namespace spmv
}  // namespace gtap

using SpmvProgram = gtap::spmv::Program;
static_assert(SpmvProgram::kFrameBytes + gtap::kHdrBytes <= gtap::host::kBuiltinStride, "frame exceeds stride");

// y = A x for a CSR matrix already in device memory (row_ptr: rows+1 int32, col_idx: nnz
// int32, val: nnz float64, x: cols float64, y: rows float64). Rows are split in 4 pieces (in 2
// where full batches of `cutoff` rows do not fit the deque) down to ranges of at most `cutoff` rows
// (0 -> 16), whose rows become one task each.
// Replaces the program of examples/spmv/spmv_thread.cu:34-66.
extern "C" int gtap_spmv(const int32_t* row_ptr, const int32_t* col_idx, const double* val, const double* x,
                         double* y, int32_t rows, int32_t cols, int32_t cutoff, gtap_run_stats* stats) {
    using namespace gtap;
    if (!row_ptr || rows < 0 || cols < 0 || (rows > 0 && !y) || (cols > 0 && !x))
        return host::invalid_argument("gtap_spmv: bad arguments");
    if (cutoff <= 0) cutoff = 16;
    if (rows == 0) {
        if (stats) memset(stats, 0, sizeof(*stats));
        return 0;
    }
    int32_t nnz = 0;  // the entry count is row_ptr[rows]; every row range is checked against it
    GTAP_HIP_TRY(hipMemcpy(&nnz, row_ptr + rows, sizeof(int32_t), hipMemcpyDeviceToHost));
    if (nnz < 0) return host::invalid_argument("gtap_spmv: negative entry count");
    if (nnz > 0 && (!col_idx || !val)) return host::invalid_argument("gtap_spmv: bad arguments");
    if (int st = gtap_initialize()) return st;
    spmv::RangeArg root{0, rows};
    gtap_job job = host::make_job(spmv::F_RANGE, 0, &root, sizeof(root));
    spmv::SpmvArgs a{row_ptr, col_idx, val, x, y, rows, cols, cutoff, 64u, 2, nnz};
    // Rows per batch, by the mean row length: a batch's time is its entries', so with long rows
    // small batches spread better, and with short ones the round's own time counts. Measured (us,
    // batches of 64 / 32 / 16 / 8, ranges cut in 4): 1M rows of 300: 3870 / 3784 / 3737 / 3722;
    // 5000 rows of 200: 215 / 146 / 142 / 140; 200003 rows of 100: 363 / 328 / 332 / 358; 512K rows
    // of 40: 402 / 384 / 412 / 481; 1M rows of 5: 336 / 334 / 403 / 573. Ranges cut in 4 instead of
    // 2 reach full batches in half the rounds (1000 rows of 10: 83 -> 77 us). A cutoff whose full
    // batch of ranges does not fit the deque keeps full batches of halves: it ends in the
    // queue-overflow error as it always has.
    if (64ll * cutoff <= (int64_t)host::rt().cap - (int64_t)kMargin) {
        const int64_t mean = nnz / rows;
        a.batch = mean >= 160 ? 8u : (mean >= 96 ? 16u : 32u);
        a.fan = 4;
    }
    return host::run_single_job<SpmvProgram>(a, job, nullptr, stats, GTAP_TERM_QUIESCE);
}

// Host-buffer convenience: copies the matrix and x in, runs gtap_spmv, copies y out.
extern "C" int gtap_spmv_host(const int32_t* row_ptr, const int32_t* col_idx, const double* val, const double* x,
                              double* y, int32_t rows, int32_t cols, int32_t cutoff, gtap_run_stats* stats) {
    using namespace gtap;
    if (!row_ptr || rows < 0 || cols < 0 || (rows > 0 && !y) || (cols > 0 && !x))
        return host::invalid_argument("gtap_spmv_host: bad arguments");
    if (rows == 0) return gtap_spmv(row_ptr, col_idx, val, x, y, 0, cols, cutoff, stats);
    const int64_t nnz = row_ptr[rows];
    if (nnz < 0) return host::invalid_argument("gtap_spmv_host: negative entry count");
    if (int st = host::check_csr_rows(row_ptr, rows, nnz, "gtap_spmv_host")) return st;
    if (nnz > 0 && (!col_idx || !val)) return host::invalid_argument("gtap_spmv_host: bad arguments");
    int32_t *drp = nullptr, *dci = nullptr;
    double *dv = nullptr, *dx = nullptr, *dy = nullptr;
    int st = 0;
    hipError_t e = hipMalloc(&drp, (size_t)(rows + 1) * 4);
    if (e == hipSuccess) e = hipMalloc(&dci, (size_t)(nnz > 0 ? nnz : 1) * 4);
    if (e == hipSuccess) e = hipMalloc(&dv, (size_t)(nnz > 0 ? nnz : 1) * 8);
    if (e == hipSuccess) e = hipMalloc(&dx, (size_t)(cols > 0 ? cols : 1) * 8);
    if (e == hipSuccess) e = hipMalloc(&dy, (size_t)rows * 8);
    if (e == hipSuccess) e = hipMemcpy(drp, row_ptr, (size_t)(rows + 1) * 4, hipMemcpyHostToDevice);
    if (e == hipSuccess && nnz > 0) e = hipMemcpy(dci, col_idx, (size_t)nnz * 4, hipMemcpyHostToDevice);
    if (e == hipSuccess && nnz > 0) e = hipMemcpy(dv, val, (size_t)nnz * 8, hipMemcpyHostToDevice);
    if (e == hipSuccess && cols > 0) e = hipMemcpy(dx, x, (size_t)cols * 8, hipMemcpyHostToDevice);
    if (e != hipSuccess) st = host::hip_status(e, "gtap_spmv_host copy-in");
    if (!st) st = gtap_spmv(drp, dci, dv, dx, dy, rows, cols, cutoff, stats);
    if (!st) {
        e = hipMemcpy(y, dy, (size_t)rows * 8, hipMemcpyDeviceToHost);
        if (e != hipSuccess) st = host::hip_status(e, "gtap_spmv_host copy-out");
    }
    (void)hipFree(drp);
    (void)hipFree(dci);
    (void)hipFree(dv);
    (void)hipFree(dx);
    (void)hipFree(dy);
    return st;
}

namespace {

uint64_t spmv_mix(uint64_t z) {
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

}  // namespace

// A random CSR matrix of the shape of examples/spmv/spmv_thread.cu:89-107 (rows x rows;
// row i has 1 + (h mod (2*avg_nnz - 1)) column draws, sorted and deduplicated; values uniform
// in [-1, 1)), from a splitmix64 stream keyed by (seed, row, draw), so every row can be
// generated on its own: rows are generated by several host threads, twice (counts, then
// entries). Two calls: with row_ptr only (col_idx = val = NULL) it fills row_ptr and
// *nnz_out; with all buffers it fills the matrix.
extern "C" int gtap_spmv_random(int32_t rows, int32_t avg_nnz, uint64_t seed, int32_t* row_ptr, int32_t* col_idx,
                                double* val, int64_t* nnz_out) {
    if (rows < 0 || avg_nnz < 1 || avg_nnz > (1 << 24) || !row_ptr) return gtap::host::invalid_argument("gtap_spmv_random");
    const uint64_t span = 2ull * (uint64_t)avg_nnz - 1ull;
    // the sorted, deduplicated columns of row i in `cols`; returns the row's key
    auto row_cols = [&](int32_t i, std::vector<int32_t>& cols) {
        const uint64_t key = spmv_mix(seed ^ (0x9E3779B97F4A7C15ULL * ((uint64_t)i + 1)));
        const uint32_t cnt = 1u + (uint32_t)(key % span);
        cols.resize(cnt);
        for (uint32_t k = 0; k < cnt; ++k) cols[k] = (int32_t)(spmv_mix(key + 2ull * k + 1ull) % (uint64_t)rows);
        std::sort(cols.begin(), cols.end());
        cols.erase(std::unique(cols.begin(), cols.end()), cols.end());
        return key;
    };
    unsigned nth = std::thread::hardware_concurrency();
    nth = nth == 0 ? 1u : (nth > 32u ? 32u : nth);
    if ((int64_t)rows < 4096) nth = 1;
    auto parallel_rows = [&](auto&& body) {
        std::vector<std::thread> pool;
        const int64_t per = ((int64_t)rows + nth - 1) / nth;
        for (unsigned t = 0; t < nth; ++t) {
            const int32_t r0 = (int32_t)std::min<int64_t>((int64_t)t * per, rows);
            const int32_t r1 = (int32_t)std::min<int64_t>((int64_t)(t + 1) * per, rows);
            pool.emplace_back([&body, r0, r1] {
                std::vector<int32_t> cols;
                for (int32_t i = r0; i < r1; ++i) body(i, cols);
            });
        }
        for (auto& th : pool) th.join();
    };
    std::vector<int32_t> count((size_t)rows);
    parallel_rows([&](int32_t i, std::vector<int32_t>& cols) {
        row_cols(i, cols);
        count[(size_t)i] = (int32_t)cols.size();
    });
    int64_t nnz = 0;
    row_ptr[0] = 0;
    for (int32_t i = 0; i < rows; ++i) {
        nnz += count[(size_t)i];
        if (nnz > 0x7FFFFFFF) return gtap::host::invalid_argument("gtap_spmv_random: more than 2^31-1 entries");
        row_ptr[i + 1] = (int32_t)nnz;
    }
    if (col_idx && val) {
        parallel_rows([&](int32_t i, std::vector<int32_t>& cols) {
            const uint64_t key = row_cols(i, cols);
            const int64_t at = row_ptr[i];
            for (size_t k = 0; k < cols.size(); ++k) {
                col_idx[at + (int64_t)k] = cols[k];
                const uint64_t r = spmv_mix(key + 2ull * (uint64_t)cols[k] + 2ull);
                val[at + (int64_t)k] = (double)(r >> 11) * (2.0 / 9007199254740992.0) - 1.0;
            }
        });
    }
    if (nnz_out) *nnz_out = nnz;
    return 0;
}
