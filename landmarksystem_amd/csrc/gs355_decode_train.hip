// The anchor decode as training differentiates it (landmark/nerf_components/model_components/fields/
// anchor_decoder.py:147-242 under autograd; benchmarks/nerf/scaffold_gs/gs_trainer.py), forward and back, in fp32.  The
// feature bank is the caller's: it hands over mixed features.
//
//   rows      visible anchors per run of 128 and (scan) their ranks
//   inputs    the list of visible anchors and the heads' input rows [feat | view | dist or level]
//   heads     hidden = relu(W0 x + b0) and W1 hidden + b1, kept offsets (opacity pre-activation > 0) per group of 32 rows
//             and (scan) their output slots
//   emit      activations and compaction of the kept offsets
//   items     backward: cotangents of the outputs to those of the pre-activations, gradients of offsets and scales
//   layers    backward: a wavefront takes 32 rows at a time back through the layers to the features (and view directions),
//             the products of the weight gradients accumulated in registers over all of its tiles
//   sum       the workgroups' weight gradients added up in a fixed order
//
// Going forward the heads add in the order in which the framework's fp32 linear layers add over some thousand rows, and
// every operation around them rounds as the framework's own does (this file is compiled without contraction): a scene's
// opacities saturate, an anchor far from the camera has pre-activations of a hundred, and one more rounding in them moves
// the few unsaturated Gaussians across the rasterizer's thresholds.  With the library at hand the Gaussians of 5 000 to
// 200 000 anchors are the statements' to the bit; with few rows, where it splits a sum, opacities differ by up to 1.2e-7
// (1 and 880 rows).  Nothing relies on either: another library may add in another order.
//
// Backward, everything is transposed as in the inference decode: weights are the left operand of v_mfma_f32_32x32x2_f32
// (rows = units), anchors the columns, and the accumulator of one layer (lane = anchor, registers = units
// 8 b + 4 half + t) is the next product's right operand register by register, the weights being read in that order.  One
// matrix instruction takes 64 cycles, so its left operand comes from LDS, one dword per lane, rows of odd stride.
//
// As torch operations the backward pass alone was some thirty launches of skinny matrix products, index and reduction
// kernels.  A training step at 200k anchors with ten offsets, most of them visible, at 1080p: 3.48 ms with the statements
// in both directions, 1.50 with these kernels when they were written, 1.18 now, the rasterizer included.
#include "gs355_internal.h"

namespace gs355 {

namespace {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kFeat = 32;
constexpr int kRun = 128;           // anchors per run, as in the inference decode
constexpr int kW0Stride = 37;       // 36 inputs (35-wide heads: zero weight) and, in gradients, the bias
constexpr int kW1Stride = 33;       // 32 hidden units and, in gradients, the bias
constexpr int kRows = 112;          // outputs of the three heads, 11 n <= 110, padded
constexpr int kGroup = 32;          // rows per group of the kept offsets
constexpr int kMaxOffsets = 10;

struct TrainArgs {
    int A, n;
    uint32_t V;            // rows (visible anchors; going through the heads: as many as there is room for)
    int in_dim[3];
    const float* anchor;
    const float* feat;     // [A,32], or [V,32] with compact_feat
    const float* offset;
    const float* scaling;
    const uint8_t* visible;
    const float* campos;
    const float* level;    // replaces the distance
    int compact_feat;
    const float* w0[3];
    const float* b0[3];
    const float* w1[3];
    const float* b1[3];
    float* with_dist;      // [V,36] input rows, or NULL
    float* without;        // [V,35] input rows, or NULL
    const float* hidden[3];  // [V,32]
    const float* pre[3];     // [V,n] [V,7n] [V,3n] pre-activations
};

// The heads' weights in LDS (and, in the same shape, a workgroup's gradients of them with the biases' in the last
// columns).  Outputs are numbered through the heads: opacity [0, n), covariance [n, 8 n), colour [8 n, 11 n).
struct HeadParameters {
    float w0[3][32 * kW0Stride];
    float w1[kRows * kW1Stride];
};
constexpr int kGradFloats = 3 * 32 * kW0Stride + kRows * kW1Stride;

__device__ __forceinline__ int head_of(int o, int n) { return o < n ? 0 : o < 8 * n ? 1 : 2; }
__device__ __forceinline__ int head_base(int j, int n) { return j == 0 ? 0 : j == 1 ? n : 8 * n; }
__device__ __forceinline__ int head_outputs(int j, int n) { return j == 0 ? n : j == 1 ? 7 * n : 3 * n; }

// By a workgroup of 256: every thread requests all of its floats before it waits for the first (one after the other, a branch
// around each, they took 20 us).
__device__ __forceinline__ void load_parameters(HeadParameters& s, const TrainArgs& d)
{
    constexpr int kThreads = 256, kEach0 = (32 * 36 + kThreads - 1) / kThreads, kEach1 = (kFeat * 7 * kMaxOffsets + kThreads - 1) / kThreads;
    const int tid = threadIdx.x;
    auto from = [](const float* p, int count) {  // zeros past the last of the floats
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, 4 * count, 0x00020000);
    };
    float v0[3][kEach0], v1[3][kEach1];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const auto w0 = from(d.w0[j], 32 * d.in_dim[j]), w1 = from(d.w1[j], kFeat * head_outputs(j, d.n));
#pragma unroll
        for (int k = 0; k < kEach0; ++k)
            v0[j][k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(w0, 4 * tid, 4 * kThreads * k, 0));
#pragma unroll
        for (int k = 0; k < (j == 0 ? 2 : j == 1 ? kEach1 : 4); ++k)
            v1[j][k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(w1, 4 * tid, 4 * kThreads * k, 0));
    }
    static_assert(kFeat * kMaxOffsets <= 2 * kThreads && kFeat * 3 * kMaxOffsets <= 4 * kThreads, "");
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int w = d.in_dim[j], inv_w = (65536 + w - 1) / w;  // e / w == (e * inv_w) >> 16 for e < 32 w, w = 35 or 36
#pragma unroll
        for (int k = 0; k < kEach0; ++k) {
            const int e = k * kThreads + tid, r = (e * inv_w) >> 16;
            if (e < 32 * w) s.w0[j][r * kW0Stride + e - r * w] = v0[j][k];
        }
        if (tid < 32) {
            if (w < 36) s.w0[j][tid * kW0Stride + 35] = 0.0f;
            s.w0[j][tid * kW0Stride + 36] = 0.0f;
        }
#pragma unroll
        for (int k = 0; k < (j == 0 ? 2 : j == 1 ? kEach1 : 4); ++k) {
            const int e = k * kThreads + tid;
            if (e < kFeat * head_outputs(j, d.n)) s.w1[(head_base(j, d.n) + e / kFeat) * kW1Stride + e % kFeat] = v1[j][k];
        }
    }
}

__device__ __forceinline__ floatx16 mfma(float a, float b, floatx16 c)
{
    return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// Unit held by register v of an accumulator.
__device__ __forceinline__ int unit_of(int v, int half) { return 8 * (v >> 2) + 4 * half + (v & 3); }

// View direction and distance of an anchor; the norm adds its squares as the framework's row reduction does.
__device__ __forceinline__ float view_of(const TrainArgs& d, size_t a, float view[3])
{
    const float v[3] = {d.anchor[3 * a] - d.campos[0], d.anchor[3 * a + 1] - d.campos[1], d.anchor[3 * a + 2] - d.campos[2]};
    const float dist = sqrtf((v[0] * v[0] + v[2] * v[2]) + v[1] * v[1]);
#pragma unroll
    for (int k = 0; k < 3; ++k) view[k] = v[k] / dist;
    return dist;
}

// Positions (within the run) of a run's visible anchors, in order; returns their number.
__device__ __forceinline__ int list_visible(const TrainArgs& d, int run, int lane, uint8_t* __restrict__ list)
{
    const int a0 = run * kRun + lane, a1 = a0 + 64;
    const bool v0 = a0 < d.A && d.visible[a0] != 0, v1 = a1 < d.A && d.visible[a1] != 0;
    const uint64_t m0 = __ballot(v0), m1 = __ballot(v1);
    const int n0 = __popcll(m0);
    if (v0) list[lanes_below_in(m0)] = (uint8_t)lane;
    if (v1) list[n0 + lanes_below_in(m1)] = (uint8_t)(64 + lane);
    wave_lds_sync();
    return n0 + __popcll(m1);
}

__global__ __launch_bounds__(256) void train_rows_kernel(TrainArgs d, uint2* __restrict__ run_totals, int runs)
{
    const int run = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (run >= runs) return;
    const int a0 = run * kRun + lane, a1 = a0 + 64;
    const int nvis = __popcll(__ballot(a0 < d.A && d.visible[a0] != 0)) + __popcll(__ballot(a1 < d.A && d.visible[a1] != 0));
    if (lane == 0) run_totals[run] = make_uint2(0u, (uint32_t)nvis);
}

// A wavefront lists its run's visible anchors and writes their input rows, four lanes per row.
__global__ __launch_bounds__(256) void train_inputs_kernel(TrainArgs d, const uint2* __restrict__ run_base, int runs,
                                                           uint32_t* __restrict__ rows)
{
    __shared__ uint8_t s_list[4][kRun];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, run = blockIdx.x * 4 + wave;
    if (run >= runs) return;
    const int nvis = list_visible(d, run, lane, s_list[wave]);
    const uint32_t rank = run_base[run].y;
    const int part = lane & 3;
    for (int i = lane >> 2; i < nvis; i += 16) {
        const size_t a = (size_t)run * kRun + s_list[wave][i], r = (size_t)rank + i;
        if (r >= d.V) continue;  // (no room: the caller learns the number from the heads)
        const float4* __restrict__ f4 = reinterpret_cast<const float4*>(d.feat + (d.compact_feat ? r : a) * kFeat) + 2 * part;
        const float4 f0 = f4[0], f1 = f4[1];
        float extra[4];
        if (part == 0) {
            rows[r] = (uint32_t)a;
            extra[3] = view_of(d, a, extra);
            if (d.level) extra[3] = d.level[a];
        }
        if (d.with_dist) {  // (rows of 144 B)
            float4* __restrict__ x = reinterpret_cast<float4*>(d.with_dist + r * 36);
            x[2 * part] = f0;
            x[2 * part + 1] = f1;
            if (part == 0) x[8] = make_float4(extra[0], extra[1], extra[2], extra[3]);
        }
        if (d.without) {
            float* __restrict__ x = d.without + r * 35 + 8 * part;
            x[0] = f0.x, x[1] = f0.y, x[2] = f0.z, x[3] = f0.w, x[4] = f1.x, x[5] = f1.y, x[6] = f1.z, x[7] = f1.w;
            if (part == 0)
#pragma unroll
                for (int k = 0; k < 3; ++k) x[32 + k] = extra[k];
        }
    }
}

// The heads going forward: hidden = relu(W0 x + b0) and W1 hidden + b1 for every row, 32 rows (a group) per wavefront and
// step, and the number of kept offsets per group.  Both layers are v_mfma_f32_16x16x4_f32 with the weights (left operand,
// rows = units) in registers for the whole kernel and 16 rows as columns.  Each eight inputs are two steps, the even ones
// and the odd ones (lane quarter q: input 2 q, then 2 q + 1), the last four of 36 one more, and the bias is added last:
// the order in which the framework's fp32 linear layers add over some thousand rows (see the top of this file; a saturated
// opacity's gradient hangs on the last bits of its pre-activation).  The accumulator of the first layer (register r of lane quarter q = unit
// 4 q + r) becomes the second's right operand by two lane exchanges per pair of registers.  Outputs pass through LDS so
// that they leave in 16-byte stores (a row of 70 is not a multiple of that).
// Six library products, three activations and a counting pass took 250 us at 200k anchors (176k of them visible, ten
// offsets); this takes 59 us for the 170 MB it moves.
// The rows are as many as the device-side count of visible anchors says, `visible_rows`: nothing is read back before the
// number of kept offsets is.
constexpr int kHeadBlocks = 8;                           // of 16 outputs: opacity 1, covariance up to 5, colour up to 2
constexpr int kHeadOut = 16 * 11 * kMaxOffsets;          // floats of 16 rows' outputs
typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void swap_lane_halves(float& a, float& b)
{
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
    const u32x2 r = __builtin_amdgcn_permlane32_swap((unsigned)__float_as_int(a), (unsigned)__float_as_int(b), false, false);
    a = __int_as_float((int)r.x);
    b = __int_as_float((int)r.y);
}
__device__ __forceinline__ void swap_lane_rows(float& a, float& b)
{
    typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
    const u32x2 r = __builtin_amdgcn_permlane16_swap((unsigned)__float_as_int(a), (unsigned)__float_as_int(b), false, false);
    a = __int_as_float((int)r.x);
    b = __int_as_float((int)r.y);
}

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void train_heads_kernel(
    TrainArgs d, const uint32_t* __restrict__ visible_rows, uint32_t* __restrict__ visible_out, float* __restrict__ hidden0,
    float* __restrict__ hidden1, float* __restrict__ hidden2,
    float* __restrict__ pre0, float* __restrict__ pre1, float* __restrict__ pre2, uint2* __restrict__ totals)
{
    __shared__ float s_b0[3][32];
    __shared__ float s_b1[kHeadBlocks * 16];
    // the weights on their way to registers, then the outputs of each wavefront's 16 rows
    __shared__ __align__(16) float s_all[kGradFloats > 4 * kHeadOut ? kGradFloats : 4 * kHeadOut];
    HeadParameters& s_parameters = *reinterpret_cast<HeadParameters*>(s_all);
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, quarter = lane >> 4, col = lane & 15;
    const int n = d.n;
    const uint32_t groups = (d.V + kGroup - 1) / kGroup;  // that have a place in `totals`
    const uint32_t V = min(*visible_rows, d.V);
    if (visible_out && blockIdx.x == 0 && threadIdx.x == 0) *visible_out = *visible_rows;
    auto block_head = [](int blk) { return blk == 0 ? 0 : blk < 6 ? 1 : 2; };
    auto block_first = [](int blk) { return blk == 0 ? 0 : blk < 6 ? 16 * (blk - 1) : 16 * (blk - 6); };  // output within its head
    for (int i = threadIdx.x; i < 3 * 32; i += 256) s_b0[i / 32][i % 32] = d.b0[i / 32][i % 32];
    for (int i = threadIdx.x; i < kHeadBlocks * 16; i += 256) {
        const int j = block_head(i / 16), o = block_first(i / 16) + i % 16;
        s_b1[i] = o < head_outputs(j, n) ? d.b1[j][o] : 0.0f;
    }
    auto input_of = [&](int step) { return step < 8 ? 8 * (step / 2) + 2 * quarter + (step & 1) : 32 + quarter; };
    // (by way of LDS: a lane's own 118 loads from 64 places each took 15 to 20 us)
    load_parameters(s_parameters, d);
    __syncthreads();
    float w0[3][2][9], w1[kHeadBlocks][8];  // lane (quarter, column i): unit 16 block + i, input_of(step)
#pragma unroll
    for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int k = 0; k < 9; ++k) {
                const int in = input_of(k);
                w0[j][h][k] = s_parameters.w0[j][(16 * h + col) * kW0Stride + in];  // (zero past the head's inputs)
            }
#pragma unroll
    for (int blk = 0; blk < kHeadBlocks; ++blk) {
        const int j = block_head(blk), o = block_first(blk) + col;
#pragma unroll
        for (int k = 0; k < 8; ++k)
            w1[blk][k] = o < head_outputs(j, n) ? s_parameters.w1[(head_base(j, n) + o) * kW1Stride + input_of(k)] : 0.0f;
    }
    __syncthreads();
    float* const out = s_all + wave * kHeadOut;
    for (uint32_t tile = blockIdx.x * 4 + wave; tile < groups; tile += gridDim.x * 4) {
        const uint32_t row0 = tile * kGroup;
        if (row0 >= V) {  // (the scan goes over all places)
            if (lane == 0) totals[tile] = make_uint2(0u, 0u);
            continue;
        }
        uint32_t row[2];
        float x[2][2][9];  // [without, with distance][16 rows][step]
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            row[h] = row0 + 16u * h + (uint32_t)col;
            const size_t r = min(row[h], V - 1);
#pragma unroll
            for (int k = 0; k < 9; ++k) {  // (column 35 of a row of 35: any finite value, its weight is zero)
                x[0][h][k] = d.without ? d.without[r * 35 + min(input_of(k), 34)] : 0.0f;
                x[1][h][k] = d.with_dist ? d.with_dist[r * 36 + input_of(k)] : 0.0f;
            }
        }
        uint32_t kept = 0;
        float right[3][2][8];  // hidden units as the second layer's right operand
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const bool dist = d.in_dim[j] == 36;
            floatx4 acc[2][2] = {};
#pragma unroll
            for (int k = 0; k < 9; ++k)
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int u = 0; u < 2; ++u)
                        acc[h][u] = __builtin_amdgcn_mfma_f32_16x16x4f32(w0[j][u][k], dist ? x[1][h][k] : x[0][h][k], acc[h][u], 0, 0, 0);
            float* const dst = j == 0 ? hidden0 : j == 1 ? hidden1 : hidden2;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    float v[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float pre = acc[h][u][r] + s_b0[j][16 * u + 4 * quarter + r];
                        v[r] = pre > 0.0f || pre != pre ? pre : 0.0f;  // (NaN stays)
                    }
                    if (row[h] < V)
                        *reinterpret_cast<float4*>(dst + (size_t)row[h] * kFeat + 16 * u + 4 * quarter) =
                            make_float4(v[0], v[1], v[2], v[3]);
#pragma unroll
                    for (int r = 0; r < 2; ++r) {
                        swap_lane_rows(v[r], v[r + 2]);
                        swap_lane_halves(v[r], v[r + 2]);
                        right[j][h][4 * u + r] = v[r];
                        right[j][h][4 * u + 2 + r] = v[r + 2];
                    }
                }
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
#pragma unroll
            for (int blk = 0; blk < kHeadBlocks; ++blk) {
                const int j = block_head(blk), count = head_outputs(j, n), first = block_first(blk);
                if (first >= count) continue;  // uniform
                floatx4 acc = {};
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    acc = __builtin_amdgcn_mfma_f32_16x16x4f32(w1[blk][k], right[j][h][k], acc, 0, 0, 0);
                float* const dst = out + 16 * head_base(j, n) + col * count;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int o = first + 4 * quarter + r;
                    const float v = acc[r] + s_b1[16 * blk + 4 * quarter + r];
                    if (o < count) dst[o] = v;
                    if (blk == 0) kept += (uint32_t)__popcll(__ballot(o < count && row[h] < V && v > 0.0f));
                }
            }
            wave_lds_sync();
            const uint32_t first_row = row0 + 16u * h, rows = first_row < V ? min(16u, V - first_row) : 0u;
#pragma unroll
            for (int j = 0; j < 3; ++j) {
                const int count = head_outputs(j, n), floats = (int)rows * count;
                float* const dst = (j == 0 ? pre0 : j == 1 ? pre1 : pre2) + (size_t)first_row * count;
                const float* const src = out + 16 * head_base(j, n);
                for (int i = lane; i < floats / 4; i += 64)
                    reinterpret_cast<float4*>(dst)[i] = reinterpret_cast<const float4*>(src)[i];
                if (lane < (floats & 3)) dst[(floats & ~3) + lane] = src[(floats & ~3) + lane];
            }
            wave_lds_sync();
        }
        if (lane == 0) totals[tile] = make_uint2(kept, 0u);
    }
}

// The items (row, offset) of a group of 32 rows, row-major (the output order), one per thread of a workgroup of 32 n rounded
// up to wavefronts.  (Two rounds of 256 threads, the second mostly empty: emit 59 us, items 57; one round: 51 and 53.)
constexpr int kItemThreads = kGroup * kMaxOffsets;
static_assert(kItemThreads % 64 == 0, "");
int item_threads(int n) { return (kGroup * n + 63) / 64 * 64; }
struct GroupItem {
    int count;             // of the group
    uint32_t slot;         // this thread's, were its item kept
    bool kept;
    float pre;             // opacity pre-activation
};
__device__ __forceinline__ GroupItem group_item(const TrainArgs& d, uint32_t group, uint32_t first_slot)
{
    __shared__ uint32_t s_kept[kItemThreads / 64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, it = threadIdx.x;
    const size_t row0 = (size_t)group * kGroup;
    GroupItem g;
    g.count = (int)min((size_t)kGroup, (size_t)d.V - row0) * d.n;
    g.pre = d.pre[0][row0 * d.n + min(it, g.count - 1)];
    g.kept = it < g.count && g.pre > 0.0f;
    const uint64_t mask = __ballot(g.kept);
    if (lane == 0) s_kept[wave] = (uint32_t)__popcll(mask);
    __syncthreads();
    g.slot = first_slot + lanes_below_in(mask);
    for (int w = 0; w < wave; ++w) g.slot += s_kept[w];
    return g;
}

// Memory-bound: some 130 MB at 200k anchors.
__global__ __launch_bounds__(kItemThreads) void train_emit_kernel(TrainArgs d, const uint2* __restrict__ base, uint32_t capacity,
                                                         gs355_decoded out, const uint32_t* __restrict__ rows)
{
    const int n = d.n, inv_n = (65536 + n - 1) / n;  // item / n == (item * inv_n) >> 16 for item < 32 n
    const size_t row0 = (size_t)blockIdx.x * kGroup;
    const GroupItem g = group_item(d, blockIdx.x, base[blockIdx.x].x);
    const int it = threadIdx.x;
    if (it >= g.count) return;
    const int rl = (it * inv_n) >> 16, m = it - rl * n;
    const size_t item = row0 * n + it, pos = g.slot;
    const float t = tanhf(g.pre);
    out.neural_opacity[item] = t;
    out.mask[item] = g.kept ? 1 : 0;
    if (!g.kept || pos >= capacity) return;  // (the second cannot happen: capacity comes from the count pass)
    const size_t a = rows[row0 + rl];
    const float* __restrict__ c7 = d.pre[1] + 7 * item;
    const float* __restrict__ c3 = d.pre[2] + 3 * item;
    out.opacity[pos] = t;
    const float q[4] = {c7[3], c7[4], c7[5], c7[6]};
    const float norm = quaternion_norm(q);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        out.color[3 * pos + k] = logistic(c3[k]);
        out.scaling[3 * pos + k] = d.scaling[6 * a + 3 + k] * logistic(c7[k]);
        out.xyz[3 * pos + k] = d.anchor[3 * a + k] + d.offset[(a * n + m) * 3 + k] * d.scaling[6 * a + k];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) out.rot[4 * pos + k] = q[k] / norm;
}

// Cotangents of the outputs to those of the pre-activations (`d_pre`, shaped as d.pre), and what does not go through the
// heads: gradients of offsets and scales, and the anchors' part through the Gaussians' positions.  A row's sums over its
// offsets are taken in their order from LDS.  Memory-bound: some 210 MB at 200k anchors (inside the
// kernel below, a wavefront at a time, it was most of 389 us).
__global__ __launch_bounds__(kItemThreads) void train_items_kernel(TrainArgs d, const uint2* __restrict__ base,
                                                          const uint32_t* __restrict__ rows, gs355_decode_cotangents g,
                                                          gs355_decode_gradients out, float* __restrict__ d_op,
                                                          float* __restrict__ d_cov, float* __restrict__ d_col)
{
    __shared__ float s_part[kGroup * kMaxOffsets][9];  // an item's share of d scaling (6) and d anchor (3)
    const int n = d.n, inv_n = (65536 + n - 1) / n;
    const size_t row0 = (size_t)blockIdx.x * kGroup;
    const GroupItem items = group_item(d, blockIdx.x, base[blockIdx.x].x);
    const int it = threadIdx.x;
    if (it < items.count) {
        const int rl = (it * inv_n) >> 16, m = it - rl * n;
        const size_t item = row0 * n + it, pos = items.slot, a = rows[row0 + rl];
        float dt = g.neural_opacity ? g.neural_opacity[item] : 0.0f;
        float c7[7] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, c3[3] = {0.f, 0.f, 0.f}, d_off[3] = {0.f, 0.f, 0.f};
        float part[9] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        if (items.kept) {
            if (g.opacity) dt += g.opacity[pos];
            float sc[6];
#pragma unroll
            for (int k = 0; k < 6; ++k) sc[k] = d.scaling[6 * a + k];
#pragma unroll
            for (int k = 0; k < 7; ++k) c7[k] = d.pre[1][7 * item + k];
            const float q[4] = {c7[3], c7[4], c7[5], c7[6]};
            const float norm = quaternion_norm(q);
            float d_q[4] = {0.f, 0.f, 0.f, 0.f};
            if (g.rot) {
                float along = 0.0f;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    d_q[k] = g.rot[4 * pos + k];
                    along += d_q[k] * (q[k] / norm);
                }
                if (!(norm > 1e-12f)) along = 0.0f;  // (the norm is a constant there)
#pragma unroll
                for (int k = 0; k < 4; ++k) d_q[k] = (d_q[k] - (q[k] / norm) * along) / norm;
            }
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const float sig = logistic(c7[k]), colour = logistic(d.pre[2][3 * item + k]);
                const float d_s = g.scaling ? g.scaling[3 * pos + k] : 0.0f;
                const float d_c = g.color ? g.color[3 * pos + k] : 0.0f;
                const float d_x = g.xyz ? g.xyz[3 * pos + k] : 0.0f;
                part[k] = d_x * d.offset[(a * n + m) * 3 + k];
                part[3 + k] = d_s * sig;
                part[6 + k] = d_x;
                d_off[k] = d_x * sc[k];
                c7[k] = d_s * sc[3 + k] * (1.0f - sig) * sig;
                c3[k] = d_c * (1.0f - colour) * colour;
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) c7[3 + k] = d_q[k];
        }
        const float t = tanhf(items.pre);
        // (fused: close to saturation t * t rounded by itself would be wrong by a good part of the difference)
        d_op[item] = dt * __builtin_fmaf(-t, t, 1.0f);
#pragma unroll
        for (int k = 0; k < 7; ++k) d_cov[7 * item + k] = c7[k];
#pragma unroll
        for (int k = 0; k < 3; ++k) d_col[3 * item + k] = c3[k];
        if (out.offset)
#pragma unroll
            for (int k = 0; k < 3; ++k) out.offset[(a * n + m) * 3 + k] = d_off[k];
#pragma unroll
        for (int k = 0; k < 9; ++k) s_part[it][k] = part[k];
    }
    __syncthreads();
    for (int k = threadIdx.x; k < 9 * (items.count / n); k += (int)blockDim.x) {
        const int rl = k / 9, c = k % 9;
        float sum = 0.0f;
        for (int m = 0; m < n; ++m) sum += s_part[rl * n + m][c];
        const size_t a = rows[row0 + rl];
        if (c < 6 && out.scaling) out.scaling[6 * a + c] = sum;
        if (c >= 6 && out.anchor) out.anchor[3 * a + c - 6] = sum;  // (train_layers_kernel adds the view's part)
    }
}

constexpr int kBackwardWaves = 4;      // one per SIMD: 176 registers of weight gradients and as many again
constexpr int kBackwardMaxGroups = 256;
constexpr int kTilePre = kGroup * 11 * kMaxOffsets;  // floats of a tile's pre-activation gradients
constexpr int kHiddenStride = 36;      // of a row of hidden units in LDS (16-B reads of 32 rows at one unit on distinct banks)
// LDS of a wavefront: pre-activation gradients head by head as in memory, input rows, one head's hidden units by row, and
// their gradients
constexpr int kWaveIn = kTilePre, kWaveHidden = kWaveIn + kGroup * 36, kWaveUnit = kWaveHidden + kGroup * kHiddenStride;
constexpr int kWaveFloats = kWaveUnit + kGroup * kW1Stride;

// A run of kFloat4s * 64 float4 (or fewer) on its way through a wavefront's registers.
template <int kFloat4s>
struct InFlight {
    floatx4 v[kFloat4s];
    // The whole fours of `count` floats (both uniform): buffer loads, whose descriptor holds the address and gives zeros past
    // the last of them, so that no lane needs an address of its own.  No rows, no request, but no branch either: behind one
    // the compiler no longer knows how many loads are under way, and waits for all of them.
    __device__ __forceinline__ void request(const float* src, int count, int lane)
    {
        const auto from = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(src), 0, 4 * (count & ~3), 0x00020000);
#pragma unroll
        for (int i = 0; i < kFloat4s; ++i)
            v[i] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(from, 16 * lane, 1024 * i, 0));
    }
    __device__ __forceinline__ void store(float* dst, int space, int lane) const
    {
#pragma unroll
        for (int i = 0; i < kFloat4s; ++i)
            if (64 * i + lane < space / 4) reinterpret_cast<floatx4*>(dst)[64 * i + lane] = v[i];
    }
};
// The floats behind the last whole four of `count` (the last tile's rows may end in between).
__device__ __forceinline__ void copy_rest(const float* __restrict__ src, float* dst, int count, int lane)
{
    if (lane < (count & 3)) dst[(count & ~3) + lane] = src[(count & ~3) + lane];
}

// A wavefront keeps all 11 blocks of 32 x 32 weight gradients in registers, so there is one wavefront per SIMD and a
// workgroup per compute unit, each with its own quarter of the LDS for the tile's rows.  Nothing else hides the wait for a
// tile's rows: the next tile's are requested, into registers, as soon as this one's have gone to LDS, and arrive while it is
// worked on (copies straight to LDS make every later read of LDS wait for them).  200k anchors, 176k of them visible, ten
// offsets: 86 to 88 us.  37 us of that are matrix instructions.  A tile takes some 11 us, of which its matrix instructions
// are 7.4: the operands of the next one are read from LDS while one runs, and not earlier.  8 us go to the weights and 4 to
// adding up the gradients, and the last round of tiles fills a third of the wavefronts.  Rows requested when they are needed,
// weights one after the other, the last tile's rows too, and gradients added by one wavefront after the other: 145.
// kAnchor: the anchors' own gradient is wanted (the layers are then also walked back to view direction and distance).
// kOffsets: offsets per anchor, or 0 (d.n).  Ten, the decoder's default, has its loops unrolled and requests rows ahead; with
// the count a variable there are no registers for that (400 bytes per lane were spilled), and the rows are requested together
// when they are needed.  The same anchors: 88 us (105 with kAnchor) with ten offsets; with the variable count 123 (141) at
// eight and 98 (116) at four.
template <bool kAnchor, int kOffsets>
__global__ __launch_bounds__(64 * kBackwardWaves) void train_layers_kernel(
    TrainArgs d, const uint32_t* __restrict__ rows, const float* __restrict__ d_op, const float* __restrict__ d_cov,
    const float* __restrict__ d_col, gs355_decode_gradients out, float* __restrict__ partials)
{
    // the parameters, then the wavefronts' parts; at the end the wavefronts' weight gradients, one after the other
    __shared__ __align__(16) float s_all[kGradFloats + kBackwardWaves * kWaveFloats];
    static_assert(kGradFloats % 4 == 0 && kWaveFloats % 4 == 0 && kBackwardWaves * kGradFloats <= kGradFloats + kBackwardWaves * kWaveFloats, "");
    HeadParameters& s = *reinterpret_cast<HeadParameters*>(s_all);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, half = lane >> 5, col = lane & 31;
    const int n = kOffsets ? kOffsets : d.n;
    const int width = d.with_dist ? 36 : 35;
    const float* const input_rows = d.with_dist ? d.with_dist : d.without;
    // a tile's rows on their way
    InFlight<(kGroup * kMaxOffsets / 4 + 63) / 64> fly_op;
    InFlight<(kGroup * 7 * kMaxOffsets / 4 + 63) / 64> fly_cov;
    InFlight<(kGroup * 3 * kMaxOffsets / 4 + 63) / 64> fly_col;
    InFlight<(kGroup * 36 / 4 + 63) / 64> fly_in;
    InFlight<kGroup * kFeat / 4 / 64> fly_hidden;  // one head's
    constexpr bool kAhead = kOffsets != 0;         // (with loops of unknown length there are no registers for them)
    const uint32_t stride = gridDim.x * kBackwardWaves;
    auto rows_of = [&](uint32_t tile) { return (int)min(d.V - min(tile * kGroup, d.V), (uint32_t)kGroup); };
    auto request_rows = [&](uint32_t tile) {
        const size_t row0 = (size_t)tile * kGroup;
        const int count = rows_of(tile);
        fly_op.request(d_op + row0 * n, count * n, lane);
        fly_cov.request(d_cov + row0 * 7 * n, count * 7 * n, lane);
        fly_col.request(d_col + row0 * 3 * n, count * 3 * n, lane);
        fly_in.request(input_rows + row0 * width, count * width, lane);
    };
    auto request_hidden = [&](int j, uint32_t tile) {
        fly_hidden.request(d.hidden[j] + (size_t)tile * kGroup * kFeat, rows_of(tile) * kFeat, lane);
    };
    const uint32_t first_tile = blockIdx.x * kBackwardWaves + wave;
    if (kAhead) {
        request_rows(first_tile);
        request_hidden(0, first_tile);
    }
    static_assert(kBackwardWaves == 4, "");
    load_parameters(s, d);
    __syncthreads();

    floatx16 grad1[5] = {}, grad0[6] = {};  // dW1: opacity | covariance x 3 | colour; dW0: features, extras + bias per head
    float bias1[5] = {};                    // db1 of the rows of grad1, the even and the odd rows' in either half of the lanes
    const uint32_t tiles = (d.V + kGroup - 1) / kGroup;
    for (uint32_t tile = first_tile; tile < tiles; tile += stride) {
        const uint32_t row0 = tile * kGroup, r = min(row0 + (uint32_t)col, d.V - 1);
        const bool live = row0 + (uint32_t)col < d.V;
        const int tile_rows = rows_of(tile);  // uniform
        // (an offset that the compiler does not know: it would keep dozens of addresses in registers over the tiles)
        int from = 0;
        asm volatile("" : "+s"(from));
        float* const pre = s_all + kGradFloats + wave * kWaveFloats + from;
        float* const input = pre + kWaveIn;
        float* const hidden = pre + kWaveHidden;
        float* const unit = pre + kWaveUnit;
        const uint32_t target = d.compact_feat ? r : rows[r];  // the row of the features' gradient
        if (!kAhead) request_rows(tile);
        fly_op.store(pre, kGroup * n, lane);
        fly_cov.store(pre + kGroup * n, kGroup * 7 * n, lane);
        fly_col.store(pre + kGroup * 8 * n, kGroup * 3 * n, lane);
        fly_in.store(input, kGroup * width, lane);
        if (tile_rows < kGroup) {
            copy_rest(d_op + (size_t)row0 * n, pre, tile_rows * n, lane);
            copy_rest(d_cov + (size_t)row0 * 7 * n, pre + kGroup * n, tile_rows * 7 * n, lane);
            copy_rest(d_col + (size_t)row0 * 3 * n, pre + kGroup * 8 * n, tile_rows * 3 * n, lane);
            copy_rest(input_rows + (size_t)row0 * width, input, tile_rows * width, lane);
        }
        if (kAhead) request_rows(tile + stride);
        floatx16 d_feat = {}, d_extra = {};
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const int base = head_base(j, n), count = head_outputs(j, n);
            if (!kAhead) request_hidden(j, tile);
#pragma unroll
            for (int i = 0; i < kGroup * kFeat / 4 / 64; ++i)  // the lane's float4 of row 8 i + lane / 8
                *reinterpret_cast<floatx4*>(hidden + (8 * i + (lane >> 3)) * kHiddenStride + 4 * (lane & 7)) = fly_hidden.v[i];
            if (kAhead) request_hidden(j < 2 ? j + 1 : 0, j < 2 ? tile : tile + stride);
            wave_lds_sync();
            // the head's gradients: row stride `count`, conflict-free for the counts of ten offsets (twice an odd number)
            const float* const g = pre + kGroup * base;
            floatx16 dh = {};
            {
                const float* const w1 = s.w1 + base * kW1Stride + col + from;  // transposed: this lane's hidden unit
                const int steps = (count + 1) / 2;
                constexpr int kUnroll = kOffsets ? 35 : 1;
#pragma unroll kUnroll
                for (int k = 0; k < steps; ++k) {
                    const int o = 2 * k + half;
                    const bool in_head = kOffsets ? true : o < count;  // (the counts of ten offsets are even)
                    dh = mfma(w1[(in_head ? o : 0) * kW1Stride], in_head ? g[col * count + o] : 0.0f, dh);
                }
            }
#pragma unroll
            for (int b = 0; b < 4; ++b) {  // the hidden units of this lane's row, in accumulator order (only their sign is used)
                const floatx4 relu = *reinterpret_cast<const floatx4*>(hidden + col * kHiddenStride + 4 * (2 * b + half));
#pragma unroll
                for (int t = 0; t < 4; ++t) {
                    dh[4 * b + t] = relu[t] > 0.0f ? dh[4 * b + t] : 0.0f;
                    unit[col * kW1Stride + unit_of(4 * b + t, half)] = dh[4 * b + t];
                }
            }
            // dW1 and db1: products over the tile's rows
#pragma unroll
            for (int q = 0; q < (j == 1 ? 3 : 1); ++q) {
                if (32 * q >= count) break;  // uniform
                const int o = min(32 * q + col, count - 1);  // (rows past the head's last output are not used)
                const int at = j == 0 ? 0 : j == 1 ? 1 + q : 4;
#pragma unroll
                for (int k = 0; k < 16; ++k) {
                    const float left = g[(2 * k + half) * count + o];
                    grad1[at] = mfma(left, hidden[(2 * k + half) * kHiddenStride + col], grad1[at]);
                    bias1[at] += left;
                }
            }
            wave_lds_sync();
            // back to the inputs, and dW0
            const float* const w0 = s.w0[j] + from;
#pragma unroll
            for (int v = 0; v < 16; ++v) d_feat = mfma(w0[unit_of(v, half) * kW0Stride + col], dh[v], d_feat);
            if (kAnchor) {
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    d_extra = mfma(w0[unit_of(v, half) * kW0Stride + 32 + min(col, 4)], dh[v], d_extra);  // (rows past 3: unused)
            }
#pragma unroll
            for (int k = 0; k < 16; ++k) {
                const float left = unit[(2 * k + half) * kW1Stride + col];
                const float* const x = input + (2 * k + half) * width;
                // columns 32 .. 35 (34): view and distance; then the constant one of the bias
                const float extra = x[min(32 + col, width - 1)];
                grad0[2 * j] = mfma(left, x[col], grad0[2 * j]);
                grad0[2 * j + 1] = mfma(left, col < width - 32 ? extra : 1.0f, grad0[2 * j + 1]);
            }
            wave_lds_sync();
        }
        if (live && out.feat) {
            float4* const dst = reinterpret_cast<float4*>(out.feat + (size_t)target * kFeat);
#pragma unroll
            for (int b = 0; b < 4; ++b)
                dst[2 * b + half] = make_float4(d_feat[4 * b], d_feat[4 * b + 1], d_feat[4 * b + 2], d_feat[4 * b + 3]);
        }
        if (kAnchor && live && half == 0) {  // rows 0..3 of d_extra: view direction, distance (or level)
            const size_t a = rows[r];
            float view[3];
            const float dist = view_of(d, a, view);
            const float along = view[0] * d_extra[0] + view[1] * d_extra[1] + view[2] * d_extra[2];
            const float d_dist = d.level ? 0.0f : d_extra[3];
#pragma unroll
            for (int k = 0; k < 3; ++k)
                out.anchor[3 * a + k] += (d_extra[k] - view[k] * along) / dist + d_dist * view[k];
        }
    }

    // ---- the wavefronts' weight gradients side by side in LDS (what is no gradient is not read), then their sums in order ----
    __syncthreads();
    float* const mine = s_all + wave * kGradFloats;
    float* const mine1 = mine + 3 * 32 * kW0Stride;
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        const int base = head_base(j, n), count = head_outputs(j, n);
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            float* const dst = mine + j * 32 * kW0Stride + unit_of(v, half) * kW0Stride;
            dst[col] = grad0[2 * j][v];
            if (col < width - 32) dst[32 + col] = grad0[2 * j + 1][v];
            else if (col == width - 32) dst[36] = grad0[2 * j + 1][v];  // (the bias keeps its column)
            else if (col == 4) dst[35] = 0.0f;  // (no rows at all, and so no input rows that would tell their width)
        }
#pragma unroll
        for (int q = 0; q < (j == 1 ? 3 : 1); ++q)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int o = 32 * q + unit_of(v, half);
                if (o < count) mine1[(base + o) * kW1Stride + col] = grad1[j == 0 ? 0 : j == 1 ? 1 + q : 4][v];
            }
#pragma unroll
        for (int q = 0; q < (j == 1 ? 3 : 1); ++q) {
            const float part = bias1[j == 0 ? 0 : j == 1 ? 1 + q : 4], sum = part + __shfl_xor(part, 32, 64);
            if (half == 0 && 32 * q + col < count) mine1[(base + 32 * q + col) * kW1Stride + 32] = sum;
        }
    }
    __syncthreads();
    float* const to = partials + (size_t)blockIdx.x * kGradFloats;
    static_assert(kBackwardWaves == 4, "");
#pragma unroll 4
    for (int i = threadIdx.x; i < kGradFloats; i += 64 * kBackwardWaves)
        to[i] = ((s_all[i] + s_all[kGradFloats + i]) + s_all[2 * kGradFloats + i]) + s_all[3 * kGradFloats + i];
}

// Sixty-four elements of the weight gradients per workgroup, the workgroups' contributions split over 16 wavefronts.
__global__ __launch_bounds__(1024) void train_sum_kernel(TrainArgs d, const float* __restrict__ partials, int groups,
                                                         gs355_decode_gradients out)
{
    __shared__ float s_sum[16][64];
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, i = blockIdx.x * 64 + lane;
    float sum = 0.0f;
    if (i < kGradFloats)
#pragma unroll 4
        for (int g = wave; g < groups; g += 16) sum += partials[(size_t)g * kGradFloats + i];
    s_sum[wave][lane] = sum;
    __syncthreads();
    if (wave != 0 || i >= kGradFloats) return;
    sum = 0.0f;
#pragma unroll
    for (int w = 0; w < 16; ++w) sum += s_sum[w][lane];
    if (i < 3 * 32 * kW0Stride) {
        const int j = i / (32 * kW0Stride), unit = i % (32 * kW0Stride) / kW0Stride, c = i % kW0Stride;
        if (c < d.in_dim[j]) {
            if (out.w0[j]) out.w0[j][unit * d.in_dim[j] + c] = sum;
        } else if (c == 36 && out.b0[j]) {
            out.b0[j][unit] = sum;
        }
        return;
    }
    const int k = i - 3 * 32 * kW0Stride, o = k / kW1Stride, c = k % kW1Stride;
    if (o >= 11 * d.n) return;
    const int j = head_of(o, d.n), at = o - head_base(j, d.n);
    if (c < kFeat) {
        if (out.w1[j]) out.w1[j][at * kFeat + c] = sum;
    } else if (out.b1[j]) {
        out.b1[j][at] = sum;
    }
}

// Workspace kept from the forward to the backward pass: totals and bases (of the runs, then of the groups of rows), the
// list of visible anchors.
struct TrainLayout {
    size_t totals, visible, base, rows, total;
};
TrainLayout train_layout(int32_t A)
{
    auto up = [](size_t v) { return (v + 255) / 256 * 256; };
    const size_t groups = ((size_t)A + kGroup - 1) / kGroup;  // (at least as many as runs)
    TrainLayout L;
    L.totals = 0;
    L.visible = groups * sizeof(uint2);  // the number of rows, behind the totals
    L.base = up(groups * sizeof(uint2) + 8);
    L.rows = L.base + up(groups * sizeof(uint2) + 8);
    L.total = L.rows + up((size_t)A * sizeof(uint32_t) + 4);
    return L;
}

// Scratch of the backward pass: gradients of the pre-activations (each head's 256-byte aligned), then the workgroups'
// weight gradients.
struct TrainScratch {
    size_t d_pre[3], partials, total;
};

int backward_groups(int32_t V);
TrainScratch train_scratch(int32_t V, int n)
{
    auto up = [](size_t v) { return (v + 255) / 256 * 256; };
    TrainScratch t;
    size_t off = 0;
    for (int j = 0; j < 3; ++j) {
        t.d_pre[j] = off;
        off += up((size_t)V * (j == 0 ? 1 : j == 1 ? 7 : 3) * n * sizeof(float));
    }
    t.partials = off;
    t.total = off + (size_t)backward_groups(V) * kGradFloats * sizeof(float);
    return t;
}

int backward_groups(int32_t V) { return min(kBackwardMaxGroups, max(1, ((V + 31) / 32 + kBackwardWaves - 1) / kBackwardWaves)); }

int train_args(const gs355_decoder* dec, const gs355_anchors* an, const gs355_train_rows* rows, const void* workspace,
               size_t workspace_bytes, TrainArgs* out)
{
    const int rc = check_decoder(dec, an);
    if (rc) return rc;
    if (!rows) return set_error(GS355_EINVAL, "rows is NULL");
    if (dec->bank_in_dim != 0)
        return set_error(GS355_EINVAL, "the differentiable decode takes mixed features: the feature bank is the caller's");
    if (rows->num_visible < 0 || rows->num_visible > an->A)
        return set_error(GS355_EINVAL, "num_visible must be in [0, A] (got %d)", rows->num_visible);
    if (an->A > 0) {
        if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 255u) != 0)
            return set_error(GS355_EINVAL, "workspace must be given and 256-byte aligned");
        const TrainLayout L = train_layout(an->A);
        if (workspace_bytes < L.total)
            return set_error(GS355_ENOSPC, "decode workspace has %zu bytes, %zu needed", workspace_bytes, L.total);
    }
    TrainArgs a;
    a.A = an->A;
    a.n = dec->n_offsets;
    a.V = (uint32_t)rows->num_visible;
    a.anchor = an->anchor;
    a.feat = an->feat;
    a.offset = an->offset;
    a.scaling = an->scaling;
    a.visible = an->visible_mask;
    a.campos = an->campos;
    a.level = dec->add_level ? an->level : nullptr;
    a.compact_feat = rows->compact_feat;
    for (int j = 0; j < 3; ++j) {
        a.in_dim[j] = dec->in_dim[j];
        a.w0[j] = dec->w0[j];
        a.b0[j] = dec->b0[j];
        a.w1[j] = dec->w1[j];
        a.b1[j] = dec->b1[j];
        a.hidden[j] = rows->hidden[j];
        a.pre[j] = rows->pre[j];
    }
    a.with_dist = rows->with_dist;
    a.without = rows->without;
    *out = a;
    return GS355_OK;
}

}  // namespace

}  // namespace gs355

using namespace gs355;

extern "C" {

int gs355_decode_train_bytes(int32_t A, int32_t num_visible, int32_t n_offsets, size_t* workspace, size_t* scratch)
{
    if (!workspace || !scratch) return set_error(GS355_EINVAL, "workspace / scratch is NULL");
    if (A < 0 || num_visible < 0 || num_visible > A)
        return set_error(GS355_EINVAL, "A and num_visible out of range (got %d, %d)", A, num_visible);
    if (n_offsets < 1 || n_offsets > kMaxOffsets)
        return set_error(GS355_EINVAL, "anchor decode supports 1..10 offsets per anchor (got %d)", n_offsets);
    *workspace = train_layout(A).total;
    *scratch = train_scratch(num_visible, n_offsets).total;
    return GS355_OK;
}

int gs355_decode_train(const gs355_decoder* dec, const gs355_anchors* an, const gs355_train_rows* rows, int64_t capacity,
                       const gs355_decoded* out, void* workspace, size_t workspace_bytes, uint32_t phase, void* stream)
{
    TrainArgs a;
    int rc = train_args(dec, an, rows, workspace, workspace_bytes, &a);
    if (rc) return rc;
    if (capacity < 0 || capacity > 0xFFFFFFFFll)
        return set_error(GS355_EINVAL, "capacity must be in [0, 2^32) (got %lld)", (long long)capacity);
    if (!out) return set_error(GS355_EINVAL, "decoded outputs is NULL");
    hipStream_t s = static_cast<hipStream_t>(stream);
    char* ws = static_cast<char*>(workspace);
    const TrainLayout L = train_layout(a.A);
    const int runs = (a.A + kRun - 1) / kRun;
    const uint32_t groups = (a.V + kGroup - 1) / kGroup;
    uint2* totals = reinterpret_cast<uint2*>(ws + L.totals);
    uint2* base = reinterpret_cast<uint2*>(ws + L.base);
    uint32_t* list = reinterpret_cast<uint32_t*>(ws + L.rows);
    switch (phase) {
        case GS355_TRAIN_HEADS: {
            if (!out->num_visible || !out->count) return set_error(GS355_EINVAL, "num_visible / count is NULL");
            uint32_t* visible = reinterpret_cast<uint32_t*>(ws + L.visible);
            if (groups > 0) {
                if ((reinterpret_cast<uintptr_t>(a.with_dist) & 15u) != 0)
                    return set_error(GS355_EINVAL, "with_dist must be 16-byte aligned");
                for (int j = 0; j < 3; ++j)
                    if (!a.hidden[j] || !a.pre[j] || ((reinterpret_cast<uintptr_t>(a.hidden[j]) | reinterpret_cast<uintptr_t>(a.pre[j])) & 15u) != 0 ||
                        !a.b0[j] || !a.b1[j] || (a.in_dim[j] == 36 ? !a.with_dist : !a.without))
                        return set_error(GS355_EINVAL, "head %d: input rows, biases, hidden and pre-activations (16-byte aligned) are needed", j);
            } else {
                visible = nullptr;
            }
            if (runs > 0) hipLaunchKernelGGL(train_rows_kernel, dim3((runs + 3) / 4), dim3(256), 0, s, a, totals, runs);
            GS355_CHECK_LAUNCH("decode train: rows");
            rc = launch_run_scan(totals, base, (uint32_t)runs, nullptr, visible ? visible : out->num_visible, s);
            if (rc) return rc;
            if (groups > 0) {
                hipLaunchKernelGGL(train_inputs_kernel, dim3((runs + 3) / 4), dim3(256), 0, s, a, base, runs, list);
                GS355_CHECK_LAUNCH("decode train: inputs");
                float* const hidden[3] = {const_cast<float*>(a.hidden[0]), const_cast<float*>(a.hidden[1]), const_cast<float*>(a.hidden[2])};
                float* const pre[3] = {const_cast<float*>(a.pre[0]), const_cast<float*>(a.pre[1]), const_cast<float*>(a.pre[2])};
                // (two workgroups per compute unit: a wavefront's weights are 118 registers)
                hipLaunchKernelGGL(train_heads_kernel, dim3(min((groups + 3u) / 4u, 512u)), dim3(256), 0, s, a, visible,
                                   out->num_visible, hidden[0], hidden[1], hidden[2], pre[0], pre[1], pre[2], totals);
                GS355_CHECK_LAUNCH("decode train: heads");
            }
            return launch_run_scan(totals, base, groups, out->count, nullptr, s);
        }
        case GS355_TRAIN_EMIT:
            if (a.V == 0) return GS355_OK;
            if (!a.pre[0] || !a.pre[1] || !a.pre[2]) return set_error(GS355_EINVAL, "pre-activations must all be non-NULL");
            if (!out->neural_opacity || !out->mask ||
                (capacity > 0 && (!out->xyz || !out->color || !out->opacity || !out->scaling || !out->rot)))
                return set_error(GS355_EINVAL, "decoded outputs must all be non-NULL");
            hipLaunchKernelGGL(train_emit_kernel, dim3(groups), dim3(item_threads(a.n)), 0, s, a, base, (uint32_t)capacity, *out, list);
            GS355_CHECK_LAUNCH("decode train: emit");
            return GS355_OK;
        default: return set_error(GS355_EINVAL, "phase must be one of GS355_TRAIN_* (got 0x%x)", phase);
    }
}

int gs355_decode_train_backward(const gs355_decoder* dec, const gs355_anchors* an, const gs355_train_rows* rows,
                                const void* workspace, size_t workspace_bytes, const gs355_decode_cotangents* cotangents,
                                const gs355_decode_gradients* grads, void* scratch, size_t scratch_bytes, void* stream)
{
    TrainArgs a;
    int rc = train_args(dec, an, rows, workspace, workspace_bytes, &a);
    if (rc) return rc;
    if (!cotangents || !grads) return set_error(GS355_EINVAL, "cotangents / gradients is NULL");
    for (int j = 0; j < 3; ++j)
        if (a.V > 0 && (!a.pre[j] || !a.hidden[j] || (reinterpret_cast<uintptr_t>(a.hidden[j]) & 15u) != 0))
            return set_error(GS355_EINVAL, "head %d: hidden (16-byte aligned) and pre-activations are needed", j);
    if (a.V > 0 && !a.with_dist && !a.without) return set_error(GS355_EINVAL, "with_dist and without are NULL");
    if (grads->feat && (reinterpret_cast<uintptr_t>(grads->feat) & 15u) != 0)
        return set_error(GS355_EINVAL, "the gradient of the features must be 16-byte aligned");
    const int workgroups = backward_groups(rows->num_visible);
    const TrainScratch S = train_scratch(rows->num_visible, a.n);
    if (!scratch || (reinterpret_cast<uintptr_t>(scratch) & 255u) != 0 || scratch_bytes < S.total)
        return set_error(GS355_ENOSPC, "decode backward scratch: %zu bytes given, %zu needed, 256-byte aligned", scratch_bytes,
                         S.total);
    hipStream_t s = static_cast<hipStream_t>(stream);
    const TrainLayout L = train_layout(a.A);
    const char* ws = static_cast<const char*>(workspace);
    char* sc = static_cast<char*>(scratch);
    const uint32_t* list = reinterpret_cast<const uint32_t*>(ws + L.rows);
    const uint2* base = reinterpret_cast<const uint2*>(ws + L.base);
    float* d_pre[3];
    for (int j = 0; j < 3; ++j) d_pre[j] = reinterpret_cast<float*>(sc + S.d_pre[j]);
    float* partials = reinterpret_cast<float*>(sc + S.partials);
    if (a.V > 0) {
        hipLaunchKernelGGL(train_items_kernel, dim3((a.V + kGroup - 1) / kGroup), dim3(item_threads(a.n)), 0, s, a, base, list, *cotangents,
                           *grads, d_pre[0], d_pre[1], d_pre[2]);
        GS355_CHECK_LAUNCH("decode train: items");
    }
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(workgroups), dim3(64 * kBackwardWaves), 0, s, a, list, d_pre[0], d_pre[1], d_pre[2],
                           *grads, partials);
    };
    if (grads->anchor) {
        if (a.n == 10) launch(train_layers_kernel<true, 10>);
        else launch(train_layers_kernel<true, 0>);
    } else {
        if (a.n == 10) launch(train_layers_kernel<false, 10>);
        else launch(train_layers_kernel<false, 0>);
    }
    GS355_CHECK_LAUNCH("decode train: layers");
    hipLaunchKernelGGL(train_sum_kernel, dim3((kGradFloats + 63) / 64), dim3(1024), 0, s, a, partials, workgroups, *grads);
    GS355_CHECK_LAUNCH("decode train: weight gradients");
    return GS355_OK;
}

}  // extern "C"
