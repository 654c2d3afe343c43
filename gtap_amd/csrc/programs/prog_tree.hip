// prog_tree.hip -- the synthetic binary-tree workload: every node of a complete binary tree
// is a task that spawns its two children, waits for them, then does its own memory and
// arithmetic work and stores one float64 result (thread-executed, one task per lane).
//
// Source program (the task shape of the reference's examples/binary_tree/binary_tree_thread.cu:63-120):
//
//   __device__ double node_work(int node, int mem_ops, int compute_iters) {
//       uint32_t seed = xorshift32(node ^ 0x9e3779b9);
//       double acc = 0;
//       for (int m = 0; m < mem_ops; ++m)                       // random reads of the input
//           acc += input[xorshift32(seed + m * 747796405) & (input_n - 1)];
//       uint32_t mix = (0x9e3779b9 ^ node) + (uint32_t)acc;
//       for (int it = 0; it < compute_iters; ++it) {            // arithmetic
//           double y = fma((double)xorshift32(seed + it * 747796405), 1.0000001192092896,
//                          0.9999999403953552);
//           mix ^= (uint32_t)bits(y);
//       }
//       return (double)mix;
//   }
//   #pragma gtap function
//   __device__ void tree_work(int node, int height, int mem_ops, int compute_iters) {
//       if (height == 0) { out[node] = node_work(node, ...); return; }
//       #pragma gtap task
//       tree_work(2 * node + 1, height - 1, ...);
//       #pragma gtap task
//       tree_work(2 * node + 2, height - 1, ...);
//       #pragma gtap taskwait
//       out[node] = node_work(node, ...);
//   }
//
// `(uint32_t)acc` converts a double that may be negative. In C++ that is undefined; the
// reference's GPU converts with saturation (negative and NaN -> 0, above 2^32-1 -> 2^32-1),
// and so does sat_u32 here, explicitly, so the result does not depend on the compiler.
#include <cstring>

#include "../device/gtap_abi.hpp"
#include "../device/gtap_steps.hpp"
#include "../host/gtap_launch.hpp"

namespace gtap {
namespace tree {

enum : uint32_t { F_NODE = 1 };
struct NodeArg {
    int32_t node;
    int32_t height;
    int32_t mem_ops;
    int32_t compute_iters;
};
struct TreeArgs {
    const double* input;
    uint32_t input_mask;  // input_n - 1 (input_n a power of two)
    double* out;
    uint32_t batch;  // most nodes a wave takes at once
};

__host__ __device__ __forceinline__ uint32_t xs32(uint32_t x) {
    x ^= x << 13;
    x ^= x >> 17;
    x ^= x << 5;
    return x;
}

__device__ __forceinline__ uint32_t sat_u32(double v) {
    if (!(v > 0.0)) return 0u;  // negative, zero and NaN
    if (v >= 4294967295.0) return 0xFFFFFFFFu;
    return (uint32_t)v;
}

// One term of the arithmetic phase: the low word of fma(x, c, d). The terms are combined by
// exclusive or, so any lane may compute any of them.
__device__ __forceinline__ uint32_t mix_term(uint32_t seed, uint32_t it) {
    const double x = (double)xs32(seed + it * 747796405u);
    return (uint32_t)__builtin_bit_cast(uint64_t, __builtin_fma(x, 1.0000001192092896, 0.9999999403953552));
}

constexpr int kUnusedSlot = 16;  // frame bytes 16..23
constexpr int kCoopReads = 4;    // reads in flight per lane of a group

struct Program {
    static constexpr int kQueues = 1;
    static constexpr bool kCoop = true;    // node work is done by run_coop
    static constexpr int kFrameWords = 4;  // node, height, mem_ops, compute_iters
    static constexpr uint32_t kMaxFunc = F_NODE;
    static constexpr uint32_t kFrameBytes = 24;
    using Args = TreeArgs;
    struct WaveShared {
        double v[kCoopReads * kWave];  // the input values read in one step, in read order per node
        int32_t src[kWave];            // lanes that hold the round's nodes
    };
    __device__ __forceinline__ static uint32_t batch_cap(const Args& a) { return a.batch; }
    template <class L>
    __device__ __forceinline__ static void run(L& lane);
    template <class L>
    __device__ __forceinline__ static void run_coop(L& lane, uint64_t mask, WaveShared* sh);
};

template <class L>
__device__ __forceinline__ void Program::run(L& lane) {
    const int32_t node = lane.template arg<int32_t>(0);
    const int32_t height = lane.template arg<int32_t>(4);
    const int32_t mem_ops = lane.template arg<int32_t>(8);
    const int32_t iters = lane.template arg<int32_t>(12);
    switch (__gtap_get_task_state(lane)) {
        case 0:
            if (height > 0) {
                // the children return nothing: their result slot is an unused frame word
                __gtap_spawn_task(lane, F_NODE, 0, kUnusedSlot, NodeArg{2 * node + 1, height - 1, mem_ops, iters});
                __gtap_spawn_task(lane, F_NODE, 0, kUnusedSlot, NodeArg{2 * node + 2, height - 1, mem_ops, iters});
                if (__gtap_set_state_for_join(lane, 1, 0)) return;
            }
            [[fallthrough]];
        case 1:
            lane.coop = true;  // the node's work: run_coop
            __gtap_finish_task(lane);
            return;
        default:
            GTAP_DEVICE_ERROR(*lane.dev, GTAP_ERROR_INVALID_TASKWAIT, lane.tid, 0, lane.state, 1);
            __gtap_finish_task(lane);
            return;
    }
}

// The work of a round's m nodes on all 64 lanes. A level of the tree takes at least one node's
// work, and on one lane that is 64 reads 8 at a time and a chain of 512 steps, about 25 us: it
// bound the whole run (height 15, 64 reads, 512 steps: 663 us, with most waves idle). Here each
// node gets a group of g lanes, the largest power of two <= 64 / m: the reads go through LDS and
// every lane of the group sums them in order, so the sum has the same bits; the arithmetic terms
// are divided among the lanes and combined by exclusive or. With full batches 368 us, with the
// batches of at most 8 nodes that gtap_tree asks for 196 us, now bound by the rounds' own latency
// (the same tree without node work takes 135 us).
template <class L>
__device__ __forceinline__ void Program::run_coop(L& lane, uint64_t mask, WaveShared* sh) {
    const TreeArgs& a = *lane.args;
    const int32_t l = lane_id();
    const int32_t m = popc(mask);
    int32_t g = kWave;
    while (g * m > kWave) g >>= 1;
    const uint32_t width = (uint32_t)g;
    if (lane.coop) vst(&sh->src[rank_in(mask)], l);
    wave_sync();
    const int32_t grp = l / g, sub = l % g;
    const bool on = grp < m;
    const int32_t src = vld(&sh->src[on ? grp : 0]);
    const int32_t node = shfl((int32_t)lane.frame[0], src);
    int32_t mem_ops = shfl((int32_t)lane.frame[2], src);
    int32_t iters = shfl((int32_t)lane.frame[3], src);
    if (!on) mem_ops = iters = 0;
    const uint32_t seed = xs32((uint32_t)node ^ 0x9e3779b9u);
    double acc = 0.0;
    lds_array<double> buf = lds(&sh->v[grp * g * kCoopReads]);
    for (Steps reads{(uint32_t)mem_ops, width * kCoopReads, 0u}; ballot(reads.on()); reads.next()) {
        double v[kCoopReads];
#pragma unroll
        for (int j = 0; j < kCoopReads; ++j) {
            const uint32_t k = reads.at + (uint32_t)j * width + (uint32_t)sub;
            v[j] = k < reads.n ? a.input[xs32(seed + k * 747796405u) & a.input_mask] : 0.0;
        }
        wave_sync();  // the previous step's values have been read
#pragma unroll
        for (int j = 0; j < kCoopReads; ++j) buf[j * g + sub] = v[j];
        wave_sync();
        const uint32_t cnt = reads.more() ? reads.step : reads.left();
#pragma unroll 8
        for (uint32_t k = 0; k < cnt; ++k) acc += buf[k];
    }
    uint32_t mix = 0;
    const Steps its{(uint32_t)iters, width, (uint32_t)sub};
#pragma unroll 4
    for (uint32_t k = 0, n = its.steps(); k < n; ++k) mix ^= mix_term(seed, its.at + k * width);
    for (int32_t d = g / 2; d > 0; d >>= 1) mix ^= (uint32_t)shfl((int32_t)mix, l ^ d);
    mix ^= (0x9e3779b9u ^ (uint32_t)node) + sat_u32(acc);
    if (on && sub == 0) a.out[node] = (double)mix;
}

}  // namespace tree
}  // namespace gtap

using TreeProgram = gtap::tree::Program;
static_assert(TreeProgram::kFrameBytes + gtap::kHdrBytes <= gtap::host::kBuiltinStride, "frame exceeds stride");

// The binary-tree workload over a tree of the given height (2^(height+1) - 1 nodes). input
// (input_n float64, input_n a power of two) and out (one float64 per node) are device
// buffers. Replaces the program of examples/binary_tree/binary_tree_thread.cu:93-120.
extern "C" int gtap_tree(int32_t height, int32_t mem_ops, int32_t compute_iters, const double* input, int64_t input_n,
                         double* out, gtap_run_stats* stats) {
    using namespace gtap;
    if (height < 0 || height > 29 || mem_ops < 0 || compute_iters < 0 || !out || (mem_ops > 0 && !input) ||
        input_n < 1 || input_n > (int64_t)1 << 31 || (input_n & (input_n - 1)) != 0)
        return host::invalid_argument("gtap_tree: bad arguments (input_n must be a power of two)");
    tree::NodeArg root{0, height, mem_ops, compute_iters};
    gtap_job job = host::make_job(tree::F_NODE, 0, &root, sizeof(root));
    // Nodes per batch: a batch of c nodes takes the wave c / 64 of a full one's time, plus the
    // round's own 4 us or so. Measured (us, caps of 8 / 16 / 32 / 64): 64 reads + 512 steps a node
    // at height 15: 196 / 221 / 287 / 407, at height 20: 1473 / 1484 / 1577 / 1766; 24 reads +
    // 160 steps at height 15: 159 / 162 / 179, at height 20: 900 / 757 / 757; 8 reads + 32 steps
    // at height 15: 148 / 142 / 142 / 157, at height 20: 756 / 527 / 443 / 453. A read counts
    // like 8 steps; with enough nodes for every wave the round's own time decides.
    const int64_t node_steps = 8ll * mem_ops + compute_iters;
    const bool tall = height > 16;
    const uint32_t batch = node_steps >= 800 ? 8u : (node_steps >= 256 ? (tall ? 16u : 8u) : (tall ? 32u : 16u));
    tree::TreeArgs a{input, (uint32_t)(input_n - 1), out, batch};
    return host::run_single_job<TreeProgram>(a, job, nullptr, stats, GTAP_TERM_JOBS);
}

namespace {

uint64_t tree_mix(uint64_t z) {
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

}  // namespace

// The tree's input: n float64 uniform in [-1, 1) from a splitmix64 stream (the reference
// draws them with std::mt19937_64, binary_tree_thread.cu:139-144).
extern "C" int gtap_tree_input(uint64_t seed, int64_t n, double* out) {
    if (n < 0 || (n > 0 && !out)) return gtap::host::invalid_argument("gtap_tree_input");
    for (int64_t i = 0; i < n; ++i) {
        const uint64_t r = tree_mix(seed + 0x9E3779B97F4A7C15ULL * ((uint64_t)i + 1));
        out[i] = (double)(r >> 11) * (2.0 / 9007199254740992.0) - 1.0;
    }
    return 0;
}
