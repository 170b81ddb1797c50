// Scaffold-GS / Octree-GS anchor decode on the gfx950 matrix cores.
//
// Replaces AnchorDecoder.forward in eval mode (landmark/nerf_components/
// model_components/fields/anchor_decoder.py:108-242; MLP shapes :79-104; the
// reference's fused twin is fused_anchor_decoder.py:69-244, whose CUDA kernels
// are an empty submodule) for the configuration the Scaffold-GS model builds
// (scaffold_gs/gs_model.py:126-134): no feature bank, no level / appearance
// inputs, three two-layer MLPs  [feat(32) | view(3) | dist(1)] -> 32 -> ReLU ->
// {n, 7n, 3n}  with tanh / none / sigmoid, mask opacity > 0, then
// scaling = anchor_scaling[3:6] * sigmoid(cov[0:3]), rot = normalize(cov[3:7]),
// xyz = anchor + offset * anchor_scaling[0:3].
//
// Everything is computed transposed so that the two layers chain without any
// data movement: weights are the A operand (rows = output units), 32 anchors
// are the columns of one v_mfma_f32_32x32x16_f16 tile (the gfx950 form: 16
// k values per instruction, 8 per lane), and the accumulator layout of layer 1
// (lane = anchor, registers = hidden units 8b+4*half+t) feeds layer 2's B
// operand directly: which k value sits in which of a lane's 8 slots is free
// as long as both operands agree, so the weights of layer 2 are simply loaded
// in the order the accumulator registers come in.
//
// Precision: fp32 accumulation throughout.  Weights and anchor features that
// fp16 holds exactly (fp16 checkpoints) enter the matrix cores as one fp16
// operand; general fp32 weights and features, the four fp32-only inputs (view
// direction, distance) and the hidden activations enter as hi + lo fp16
// pairs (22 significant bits; the lo x lo products, 2^-22 of a term, are
// left out), so the result carries fp32-level accuracy either way.  A workgroup
// keeps the weights' fragments, high and low parts, in LDS.
//
// Work follows the visible anchors: the visible ones of every run of 128
// consecutive anchors are packed (in order) into dense tiles of 32, and a
// wavefront decodes one tile at a time.
//
// Output order is the reference's boolean-mask order: row-major over (visible
// anchor, offset).  Two launches: count kept offsets per anchor (opacity head
// only) -> exclusive scan -> emit (all heads; the opacity head is recomputed
// with the identical instruction sequence, so counts and emission agree).
#include <atomic>

#include "gs355_internal.h"

namespace gs355 {

namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kFeat = 32;

struct DecodeArgs {
    int A, n;       // anchors, offsets per anchor
    int in_dim[3];  // 35 or 36 per head (opacity, cov, color)
    const float* anchor;
    const float* feat;
    const float* offset;
    const float* scaling;
    const uint8_t* visible;
    const float* campos;
    const float* level;  // per-anchor level: the fourth fp32-only input instead of the distance (add_level), or NULL
    int split_feat;      // features enter as hi + lo fp16 pairs (fp32 features that fp16 cannot represent)
    int weights_lo;      // weights enter as hi + lo fp16 pairs (fp32 weights that fp16 cannot represent)
    const float* w0[3];
    const float* b0[3];
    const float* w1[3];
    const float* b1[3];
    // one-call decode (gs355_decode): the count pass leaves per-run totals behind, a one-workgroup scan (or the emit pass) turns
    // them into run bases, and the emit pass (which recomputes the opacity head: matrix instructions are cheap
    // here, registers and memory requests are not) places its Gaussians from those instead of per-anchor offsets
    uint2* run_totals;       // [runs] (kept offsets, visible anchors) per run of anchors, or NULL
    uint2* run_tiles;        // [runs] kept offsets of the run before each of its four tiles, 16 bits each (with run_totals)
    uint2* run_base;         // [runs] exclusive prefix of run_totals, or NULL
    int scan_here;           // the emit pass makes that prefix itself (runs <= kScanStripes * its workgroups), for a later one too, and the sums:
    uint32_t* num_emitted;   // of the kept offsets, or NULL
    uint32_t* num_visible;   // of the visible anchors, or NULL
    float* neural_opacity;   // [A_vis * n] tanh of every pre-activation, in visible-anchor order, or NULL
    uint8_t* kept_mask;      // [A_vis * n] pre-activation > 0, or NULL
};

typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef float float2_t __attribute__((ext_vector_type(2)));

// Eight floats as hi + lo fp16 pairs (hi = the value rounded to fp16, lo = what that rounding left over, rounded
// to fp16), converted two at a time (one packed conversion per pair and direction).
__device__ __forceinline__ void split_half8(const float v[8], half8_t& hi, half8_t& lo)
{
    half2_t h[4], l[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const float2_t x = {v[2 * j], v[2 * j + 1]};
        h[j] = __builtin_convertvector(x, half2_t);
        l[j] = __builtin_convertvector(x - __builtin_convertvector(h[j], float2_t), half2_t);
    }
    hi = (half8_t){h[0][0], h[0][1], h[1][0], h[1][1], h[2][0], h[2][1], h[3][0], h[3][1]};
    lo = (half8_t){l[0][0], l[0][1], l[1][0], l[1][1], l[2][0], l[2][1], l[3][0], l[3][1]};
}

__device__ __forceinline__ half8_t to_half8(const float v[8])
{
    half8_t h;
#pragma unroll
    for (int j = 0; j < 8; ++j) h[j] = (_Float16)v[j];
    return h;
}

// Eight entries of row `row` of a [rows x cols] row-major fp32 weight matrix, as one lane's share of an A
// operand: slots 0..3 hold columns ka..ka+3, slots 4..7 columns kb..kb+3 (zero outside the matrix).  Loads are
// unconditional at clamped (in-range) positions and masked afterwards, so that none of them waits for another:
// the fragments of a head are fetched with all loads in flight together.
__device__ __forceinline__ void weight_values(const float* __restrict__ w, int rows, int cols, int row, int ka, int kb,
                                              float v[8])
{
    const int r = min(row, rows - 1);
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = w[(size_t)r * cols + min((j < 4 ? ka : kb - 4) + j, cols - 1)];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (row < rows && (j < 4 ? ka : kb - 4) + j < cols) ? v[j] : 0.0f;
}

// Bias for an accumulator: register v = 4b + t holds row 8b + 4*half + t.  `bias` is the head's bias vector
// staged in LDS, zero-padded to a multiple of 32 rows.
__device__ __forceinline__ floatx16 bias_rows(const float* bias, int row0, int half)
{
    floatx16 c;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const float4 b = *reinterpret_cast<const float4*>(bias + row0 + 8 * g + 4 * half);
        c[4 * g] = b.x, c[4 * g + 1] = b.y, c[4 * g + 2] = b.z, c[4 * g + 3] = b.w;
    }
    return c;
}

// Weight fragments of one head: an A operand's share for each lane.
//   layer 1, k-steps 0 and 1: the 32 anchor features, slot j of half h <-> feature 16s + 8h + j
//   layer 1, k-step 2:        the four fp32-only inputs twice on half 0 (slots 0..3 meet their hi parts, slots
//                             4..7 their lo parts, both against W0[:, 32..35]); half 1 meets zero inputs
//   layer 2, k-step s:        slot j of half h <-> hidden unit 16s + 4h + j (j < 4) or 16s + 8 + 4h + (j - 4),
//                             the units held by accumulator registers 8s..8s+7 of that lane
// Every wavefront needs the same fragments, so a workgroup keeps one copy in LDS, hi parts and, for weights that
// fp16 cannot represent, lo parts: a head's fragments follow one another in the order w0[0..2], w1[0][0], w1[0][1],
// w1[1][0], ..., 64 lanes each but for w0[2], whose half 1 never matters and reads half 0's 32.
constexpr int kOpacityFrags = 0, kCovFrags = 288, kColourFrags = 832, kAllFrags = 1120;  // first lane entry of each head

__device__ __forceinline__ int frag_entry(int f, int lane)  // f: 0..2 layer 1, 3.. layer 2
{
    return f == 2 ? 128 + (lane & 31) : f < 2 ? 64 * f + lane : 160 + 64 * (f - 3) + lane;
}

// One wavefront computes fragment f of a head and stores its hi parts and (`lo` not NULL) its lo parts.
__device__ __forceinline__ void stage_fragment(const DecodeArgs& d, int head, int outputs, int f, int lane,
                                               half8_t* __restrict__ hi, half8_t* __restrict__ lo)
{
    const int row = lane & 31, half = lane >> 5;
    float v[8];
    if (f < 2) weight_values(d.w0[head], kFeat, d.in_dim[head], row, 16 * f + 8 * half, 16 * f + 8 * half + 4, v);
    else if (f == 2) weight_values(d.w0[head], kFeat, d.in_dim[head], row, 32, 32, v);
    else {
        const int r = (f - 3) >> 1, s = (f - 3) & 1;
        weight_values(d.w1[head], outputs, kFeat, 32 * r + row, 16 * s + 4 * half, 16 * s + 8 + 4 * half, v);
    }
    half8_t h, l;
    split_half8(v, h, l);
    const int at = frag_entry(f, lane);
    hi[at] = h;
    if (lo) lo[at] = l;
}

// One head for one tile of 32 anchors; `store(r, c)` receives row tile r of its outputs (rows = outputs
// 32r + 8b + 4*half + t, column = this lane's anchor), one accumulator live at a time.
// `hi`, `lo`: the head's fragments in LDS, read right before their matrix instruction.
template <int kTiles, bool kSplit, bool kWLo, class Store>
__device__ __forceinline__ void run_head(const half8_t* __restrict__ hi, const half8_t* __restrict__ lo, int lane,
                                         const float* bias0, const float* bias1, const half8_t X[kSplit ? 5 : 3],
                                         int half, Store store)
{
    // layer 1: hidden = W0 [32 x in] * X^T + b0  (X[3], X[4]: the low parts of features that fp16 cannot hold)
    floatx16 h = bias_rows(bias0, 0, half);
    half8_t w0[3];
#pragma unroll
    for (int s = 0; s < 3; ++s) w0[s] = hi[frag_entry(s, lane)];
#pragma unroll
    for (int s = 0; s < 3; ++s) h = __builtin_amdgcn_mfma_f32_32x32x16_f16(w0[s], X[s], h, 0, 0, 0);
    if constexpr (kSplit) {
#pragma unroll
        for (int s = 0; s < 2; ++s) h = __builtin_amdgcn_mfma_f32_32x32x16_f16(w0[s], X[3 + s], h, 0, 0, 0);
    }
    if constexpr (kWLo) {  // low parts of the weights against the high parts of the inputs
#pragma unroll
        for (int s = 0; s < 3; ++s)
            h = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo[frag_entry(s, lane)], X[s], h, 0, 0, 0);
    }
    // ReLU, then hi/lo split: registers 8s..8s+7 are the B operand of k-step s
    half8_t hh[2], hl[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        float r[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) r[j] = __builtin_amdgcn_fmed3f(h[8 * s + j], 0.0f, __builtin_inff());  // ReLU in one instruction
        split_half8(r, hh[s], hl[s]);
    }
    // layer 2: out = W1 [outputs x 32] * hidden + b1
#pragma unroll
    for (int r = 0; r < kTiles; ++r) {
        floatx16 c = bias_rows(bias1, 32 * r, half);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            const half8_t w1 = hi[frag_entry(3 + 2 * r + s, lane)];
            c = __builtin_amdgcn_mfma_f32_32x32x16_f16(w1, hh[s], c, 0, 0, 0);
            c = __builtin_amdgcn_mfma_f32_32x32x16_f16(w1, hl[s], c, 0, 0, 0);
            if constexpr (kWLo)
                c = __builtin_amdgcn_mfma_f32_32x32x16_f16(lo[frag_entry(3 + 2 * r + s, lane)], hh[s], c, 0, 0, 0);
        }
        store(r, c);
    }
}

// 1 / (1 + exp(-x)) from the hardware exp2 and reciprocal (each within 1 ulp; the product x log2(e) adds
// |x| 2^-24 to the exponent): relative error below 1e-6 for any x, against the 3e-5 the decode is held to.
__device__ __forceinline__ float fast_sigmoid(float x)
{
    return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(-1.4426950408889634f * x));
}

// Biases of the three heads in LDS, zero-padded: b0 at [head*32], b1 of opacity / cov / colour at 96 / 128 / 224.
__device__ __forceinline__ void stage_biases(const DecodeArgs& d, float* __restrict__ s_bias, int threads)
{
    const int n = d.n;
    for (int t = threadIdx.x; t < 256; t += threads) {
        float v = 0.0f;
        if (t < 96) v = d.b0[t >> 5][t & 31];
        else if (t < 128) v = (t - 96) < n ? d.b1[0][t - 96] : 0.0f;
        else if (t < 224) v = (t - 128) < 7 * n ? d.b1[1][t - 128] : 0.0f;
        else v = (t - 224) < 3 * n ? d.b1[2][t - 224] : 0.0f;
        s_bias[t] = v;
    }
}

// Anchors come in runs of kRun consecutive ones, whose visible ones are packed (in order) into dense tiles of 32; a
// wavefront runs the MLPs on one tile at a time: the work follows the number of visible anchors, not of anchors.
constexpr int kRun = 128, kRunTiles = kRun / 32;

// A run's visible anchors as bits, and as a list of their positions within the run, in order.
struct Visible {
    uint64_t m0, m1;
    __device__ __forceinline__ int count() const { return __popcll(m0) + __popcll(m1); }
    __device__ __forceinline__ void pack(int lane, uint8_t* __restrict__ list) const
    {
        const uint64_t below = (1ull << lane) - 1ull;
        if ((m0 >> lane) & 1ull) list[__popcll(m0 & below)] = (uint8_t)lane;
        if ((m1 >> lane) & 1ull) list[__popcll(m0) + __popcll(m1 & below)] = (uint8_t)(64 + lane);
    }
};

// The mask of a run's anchors, two a lane; requested well before it is looked at.
struct VisibleBytes {
    uint8_t b0 = 0, b1 = 0;
    __device__ __forceinline__ void load(const DecodeArgs& d, int base, int lane)
    {
        b0 = base + lane < d.A ? d.visible[base + lane] : 0;
        b1 = base + 64 + lane < d.A ? d.visible[base + 64 + lane] : 0;
    }
    __device__ __forceinline__ Visible look() const { return Visible{__ballot(b0 != 0), __ballot(b1 != 0)}; }
};

// Features, position and level of a tile's anchors.  Everything is requested without a condition: a lane without an
// anchor reads anchor 0's data, which nothing uses (matrix columns are independent, and only items of visible anchors
// are ever counted or emitted) -- conditional loads would each become a branch with its own wait.
struct TileInputs {
    float4 f[4];  // features 16s + 8*half .. +7 in f[2s], f[2s+1], s = 0..1
    float pos[3];
    float extra = 0.f;  // the anchor's level when it replaces the distance
    __device__ __forceinline__ void load(const DecodeArgs& d, int a, int half)
    {
        const float4* __restrict__ f4 = reinterpret_cast<const float4*>(d.feat + (size_t)a * kFeat);
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            f[2 * s] = f4[4 * s + 2 * half];
            f[2 * s + 1] = f4[4 * s + 2 * half + 1];
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) pos[k] = d.anchor[3 * (size_t)a + k];
        if (d.level) extra = d.level[a];
    }
    // B operand: X^T, column = anchor; slots as described at the weight fragments
    template <bool kSplit>
    __device__ __forceinline__ void operand(const DecodeArgs& d, float cx, float cy, float cz, bool vis, int half,
                                            half8_t X[kSplit ? 5 : 3]) const
    {
        float x8[8];
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            x8[0] = f[2 * s].x, x8[1] = f[2 * s].y, x8[2] = f[2 * s].z, x8[3] = f[2 * s].w;
            x8[4] = f[2 * s + 1].x, x8[5] = f[2 * s + 1].y, x8[6] = f[2 * s + 1].z, x8[7] = f[2 * s + 1].w;
            if constexpr (kSplit) split_half8(x8, X[s], X[3 + s]);  // the second: what the fp16 rounding left over
            else X[s] = to_half8(x8);
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) x8[j] = 0.0f;
        if (vis && half == 0) {
            float vx = pos[0] - cx, vy = pos[1] - cy, vz = pos[2] - cz;
            const float dist = sqrtf(vx * vx + vy * vy + vz * vz);
            vx /= dist;
            vy /= dist;
            vz /= dist;
            const float in4[4] = {vx, vy, vz, d.level ? extra : dist};
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const _Float16 top = (_Float16)in4[t];
                x8[t] = (float)top;
                x8[4 + t] = in4[t] - (float)top;
            }
        }
        X[2] = to_half8(x8);
    }
};

// Which of its anchor's offsets this lane's opacity rows keep (bit m: offset m; the mask opacity > 0 is the sign of
// the pre-activation: tanh is odd, monotone and tanh(x) = x for the smallest floats).  Rows that do not exist hold zero.
__device__ __forceinline__ uint32_t kept_rows(const floatx16& c, bool vis, int half)
{
    uint32_t mask = 0;
#pragma unroll
    for (int v = 0; v < 8; ++v) mask |= c[v] > 0.0f ? 1u << (8 * (v >> 2) + (v & 3)) : 0u;
    return vis ? mask << (4 * half) : 0u;
}

// kSplit: the features enter as hi + lo fp16 pairs (general fp32 features; two more matrix instructions per head).
// kWLo: so do the weights (general fp32 weights).
// The count pass: the opacity head of every visible anchor and how many offsets it keeps.  Four wavefronts per SIMD;
// a run's tiles are otherwise a chain of memory latencies, so the next tile's inputs are requested before the current
// tile's are waited for, and the next run's mask before the run is walked.  While there are fewer runs than workgroups
// (`shared_run`) the four wavefronts of a workgroup take a tile each of one run instead of a run each.
constexpr int kCountWaves = 4;
constexpr int kCountCap = 1024;  // workgroups: four per CU
static_assert(kCountWaves == kRunTiles, "a workgroup's wavefronts share a run tile by tile");

template <bool kSplit, bool kWLo>
__global__ __launch_bounds__(64 * kCountWaves, 4) void decode_count_kernel(DecodeArgs d, uint32_t* __restrict__ counts,
                                                                       int shared_run)
{
    __shared__ float s_bias[256];
    __shared__ half8_t s_hi[kCovFrags];
    __shared__ half8_t s_lo[kWLo ? kCovFrags : 1];
    __shared__ uint8_t s_list[kCountWaves][kRun];
    __shared__ uint32_t s_kept[kRunTiles];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, half = lane >> 5, col = lane & 31;
    const int runs = (d.A + kRun - 1) / kRun;
    const int step = shared_run ? gridDim.x : gridDim.x * kCountWaves;
    int run = shared_run ? blockIdx.x : wave * gridDim.x + blockIdx.x;
    const int first_entry = shared_run ? 32 * wave : 0, entry_step = shared_run ? kRun : 32;
    VisibleBytes next;
    if (run < runs) next.load(d, run * kRun, lane);
    stage_biases(d, s_bias, 64 * kCountWaves);
    for (int f = wave; f < 5; f += kCountWaves) stage_fragment(d, 0, d.n, f, lane, s_hi, kWLo ? s_lo : nullptr);
    __syncthreads();
    uint8_t* __restrict__ list = s_list[wave];
    const float cx = d.campos[0], cy = d.campos[1], cz = d.campos[2];

    for (; run < runs; run += step) {  // the same rounds for every wavefront where a run is shared
        const Visible now = next.look();
        const int base = run * kRun, nvis = now.count();
        if (run + step < runs) next.load(d, base + step * kRun, lane);
        now.pack(lane, list);
        if (counts) {  // anchors that are not decoded keep nothing
            if (!((now.m0 >> lane) & 1ull) && base + lane < d.A) counts[base + lane] = 0;
            if (!((now.m1 >> lane) & 1ull) && base + 64 + lane < d.A) counts[base + 64 + lane] = 0;
        }
        wave_lds_sync();
        uint32_t kept01 = 0, kept23 = 0;  // this lane's share of the kept offsets of the run's tiles, 16 bits each
        TileInputs ahead;
        int a_ahead = first_entry + col < nvis ? base + (int)list[first_entry + col] : 0;
        if (first_entry < nvis) ahead.load(d, a_ahead, half);
        for (int first = first_entry; first < nvis; first += entry_step) {  // dense tiles of the run
            const bool vis = first + col < nvis;  // lanes l and l+32 share entry first + l
            const TileInputs in = ahead;
            const int a = a_ahead;
            if (first + entry_step < nvis) {  // uniform
                a_ahead = first + entry_step + col < nvis ? base + (int)list[first + entry_step + col] : 0;
                ahead.load(d, a_ahead, half);
            }
            wave_lds_sync();  // the fragments are read again for every tile: kept across tiles they would spill
            half8_t X[kSplit ? 5 : 3];
            in.operand<kSplit>(d, cx, cy, cz, vis, half, X);
            run_head<1, kSplit, kWLo>(s_hi, s_lo, lane, s_bias, s_bias + 96, X, half, [&](int, const floatx16& c) {
                const uint32_t kept = (uint32_t)__popc(kept_rows(c, vis, half));
                const uint32_t field = kept << (first & 32 ? 16 : 0);
                (first & 64 ? kept23 : kept01) += field;
                if (counts) {
                    const uint32_t both = kept + (uint32_t)__shfl_xor((int)kept, 32, 64);
                    if (half == 0 && vis) counts[a] = both;
                }
            });
        }
        if (d.run_totals) {
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                kept01 += (uint32_t)__shfl_xor((int)kept01, off, 64);
                kept23 += (uint32_t)__shfl_xor((int)kept23, off, 64);
            }
            if (shared_run) {
                if (lane == 0) s_kept[wave] = (wave & 2 ? kept23 : kept01) >> (wave & 1 ? 16 : 0);
                __syncthreads();
                kept01 = s_kept[0] | s_kept[1] << 16;
                kept23 = s_kept[2] | s_kept[3] << 16;
                __syncthreads();
            }
            if (lane == 0 && (!shared_run || wave == 0)) {
                const uint32_t k0 = kept01 & 0xFFFFu, k1 = kept01 >> 16, k2 = kept23 & 0xFFFFu, k3 = kept23 >> 16;
                d.run_totals[run] = make_uint2(k0 + k1 + k2 + k3, (uint32_t)nvis);
                d.run_tiles[run] = make_uint2(k0 << 16, (k0 + k1) | (k0 + k1 + k2) << 16);
            }
        }
        wave_lds_sync();
    }
}

// The emit pass: all heads, then the activations of the kept (anchor, offset) items on dense wavefronts of survivors.
//
// What bounds it is how many tiles are in flight: a tile is a chain of memory and matrix latencies.  With all 11n head
// outputs of 32 anchors in LDS and part of the weights in registers a wavefront needed 27 KB and 256 registers: six
// wavefronts per CU.  Colours and covariances now pass through the same 72 words per anchor one after the other, all
// weights are shared through LDS, and the learned offsets are read for survivors only, so twelve wavefronts of 10 KB
// and at most 168 registers fill a CU with one workgroup; an anchor's rows are a multiple of 16 bytes apart, so that
// accumulators leave four rows at a time.
//
// A workgroup takes every gridDim.x-th run and its wavefronts deal out the tiles of those runs, not the runs: the
// count pass left the visible anchors and the tiles' first slots of every run behind.  A wavefront requests the inputs of
// its next tile before the current one's heads and turns them into matrix operands before the current one's stores: a wait for
// them after the stores would be a wait for the stores as well.
//
// Measured (fp32 weights and features, n = 10): 500k visible anchors that keep 3.9M offsets, 358 MB in and out, 120 ->
// 84 us; a million anchors behind a level-of-detail mask 59 -> 38 us; 60k anchors, where a wavefront has one tile, 31 -> 15.
constexpr int kEmitWaves = 12;
constexpr int kEmitCap = 256;  // workgroups: one per CU
// Up to this many runs per workgroup the emit pass adds up the runs' totals itself: a workgroup's k-th run needs the runs of
// the stripes before (gridDim.x runs each) and those before it in its own.  62 KB per workgroup at a million anchors, read
// while the weights are, in the place of a launch of one workgroup of 3 to 5 us: frames of 60k anchors 116 -> 113 us, of a
// million behind a level-of-detail mask 203 -> 200.6, of 500k 371 -> 369.  The bases go to the workspace all the same (8 B per run).
constexpr int kScanStripes = 32;
constexpr int kRowWords = 72;  // an anchor's words: first opacity, colour, offset scale, position; then covariance
constexpr int kRowColour = 16, kRowExtra = 48;

struct __align__(16) EmitWave {
    float rows[32][kRowWords];
    float scale[32][3];  // the anchor's Gaussian scale
    uint16_t list[320];  // kept items, in order: 16 * entry + offset
    uint8_t anchors[2][kRun];  // positions of the run's visible anchors: the current tile's run and the next tile's
};

// Rows 32r .. 32r + 31 of an accumulator to the anchor's words: groups of eight rows that hold an output.
__device__ __forceinline__ void store_rows(float* __restrict__ dst, int r, int outputs, int half, const floatx16& c)
{
#pragma unroll
    for (int g = 0; g < 4; ++g)
        if (32 * r + 8 * g < outputs)  // uniform
            *reinterpret_cast<float4*>(dst + 32 * r + 8 * g + 4 * half) =
                make_float4(c[4 * g], c[4 * g + 1], c[4 * g + 2], c[4 * g + 3]);
}

template <bool kSplit, bool kWLo>
__global__ __launch_bounds__(64 * kEmitWaves, 3) void decode_emit_kernel(DecodeArgs d, const uint32_t* __restrict__ offsets,
                                                                      uint32_t capacity, float* __restrict__ xyz,
                                                                      float* __restrict__ color, float* __restrict__ opacity,
                                                                      float* __restrict__ scaling_out, float* __restrict__ rot)
{
    __shared__ EmitWave s_wave[kEmitWaves];
    __shared__ float s_bias[256];
    __shared__ half8_t s_hi[kAllFrags];
    __shared__ half8_t s_lo[kWLo ? kAllFrags : 1];
    __shared__ uint4 s_stripe[kScanStripes];  // (kept offsets, visible anchors) of a stripe of runs, and of those before this workgroup's
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63, half = lane >> 5, col = lane & 31;
    const int n = d.n;
    const int runs = (d.A + kRun - 1) / kRun;
    if (d.scan_here) {
        static_assert(kEmitCap <= 4 * 64, "four runs of a stripe per lane");
        for (int k = wave; k * (int)gridDim.x < runs; k += kEmitWaves) {
            uint2 all = make_uint2(0u, 0u), before = make_uint2(0u, 0u);
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const int at = 64 * u + lane, r = k * (int)gridDim.x + at;
                const uint2 v = at < (int)gridDim.x && r < runs ? d.run_totals[r] : make_uint2(0u, 0u);
                all = make_uint2(all.x + v.x, all.y + v.y);
                if (at < (int)blockIdx.x) before = make_uint2(before.x + v.x, before.y + v.y);
            }
            const uint4 sums = make_uint4(wave_sum(all.x), wave_sum(all.y), wave_sum(before.x), wave_sum(before.y));
            if (lane == 0) s_stripe[k] = sums;
        }
    }
    stage_biases(d, s_bias, 64 * kEmitWaves);
    for (int f = wave; f < 19; f += kEmitWaves) {
        const int head = f < 5 ? 0 : f < 14 ? 1 : 2;
        const int at = head == 0 ? kOpacityFrags : head == 1 ? kCovFrags : kColourFrags;
        stage_fragment(d, head, (head == 0 ? 1 : head == 1 ? 7 : 3) * n, f - (head == 0 ? 0 : head == 1 ? 5 : 14), lane, s_hi + at,
                       kWLo ? s_lo + at : nullptr);
    }
    __syncthreads();
    EmitWave& my = s_wave[wave];
    const float cx = d.campos[0], cy = d.campos[1], cz = d.campos[2];

    // 64 of the workgroup's runs at a time, a lane's worth each: run first_run + lane * gridDim.x
    for (int first_run = blockIdx.x; first_run < runs; first_run += 64 * gridDim.x) {
        const int my_run = first_run + lane * (int)gridDim.x;
        uint32_t tiles = my_run < runs ? kRunTiles : 0;  // two-call decode: the visible anchors are not known here
        uint2 run_base = make_uint2(0u, 0u), run_tiles = make_uint2(0u, 0u);
        if (!offsets && my_run < runs) {
            tiles = (d.run_totals[my_run].y + 31u) >> 5;
            run_tiles = d.run_tiles[my_run];
            if (!d.scan_here) run_base = d.run_base[my_run];
        }
        if (d.scan_here) {  // (one round: a lane per stripe)
            const uint4 v = my_run < runs ? s_stripe[lane] : make_uint4(0u, 0u, 0u, 0u);
            const uint32_t x = wave_sum_scan(v.x), y = wave_sum_scan(v.y);
            run_base = make_uint2(x - v.x + v.z, y - v.y + v.w);
            if (wave == 0 && my_run < runs) d.run_base[my_run] = run_base;  // (for an emit phase that is repeated, with more room)
            if (blockIdx.x == 0 && wave == 0 && lane == 63) {
                if (d.num_emitted) *d.num_emitted = x;
                if (d.num_visible) *d.num_visible = y;
            }
        }
        uint32_t upto = tiles;
#pragma unroll
        for (int k = 1; k < 64; k <<= 1) {
            const uint32_t u = (uint32_t)__shfl_up((int)upto, k, 64);
            if (lane >= k) upto += u;
        }
        const int units = __builtin_amdgcn_readlane((int)upto, 63);
        // unit u of these runs: tile `first / 32` of the run whose anchors start at `base`
        auto locate = [&](int u, int& base, int& first, int& index) {
            index = min(__popcll(__ballot((int)upto <= u)), 63);
            base = (first_run + index * (int)gridDim.x) * kRun;
            first = 32 * (u - __builtin_amdgcn_readlane((int)(upto - tiles), index));
        };
        TileInputs ahead;
        float sc_ahead[3];  // half 0: scaling[0..2] (offset scale), half 1: scaling[3..5] (Gaussian scale)
        auto fetch = [&](const uint8_t* __restrict__ anchors, int base, int first, int nvis) {
            const int a = first + col < nvis ? base + (int)anchors[first + col] : 0;
            ahead.load(d, a, half);
#pragma unroll
            for (int k = 0; k < 3; ++k) sc_ahead[k] = d.scaling[6 * (size_t)a + 3 * half + k];
        };
        // the current tile, and the next: run, tile, visible anchors; `seen` is the next tile's
        int base = 0, first = 0, index = 0, nvis = 0, base1 = 0, first1 = 0, index1 = 0;
        Visible seen = {0ull, 0ull};
        half8_t X[kSplit ? 5 : 3];
        if (wave < units) {
            VisibleBytes bytes, bytes1;
            locate(wave, base, first, index);
            bytes.load(d, base, lane);
            if (wave + kEmitWaves < units) {
                locate(wave + kEmitWaves, base1, first1, index1);
                bytes1.load(d, base1, lane);
            }
            const Visible v = bytes.look();
            nvis = v.count();
            v.pack(lane, my.anchors[0]);
            wave_lds_sync();
            fetch(my.anchors[0], base, first, nvis);
            seen = bytes1.look();
            ahead.operand<kSplit>(d, cx, cy, cz, first + col < nvis, half, X);
        }
        int buffer = 0;
        for (int unit = wave; unit < units; unit += kEmitWaves, buffer ^= 1) {
            const bool vis = first + col < nvis;  // lanes l and l+32 share entry first + l
            const uint8_t* __restrict__ anchors = my.anchors[buffer];
            uint32_t slot, run_rank = 0;
            if (offsets) {  // two-call decode: the first anchor's slot is the tile's (past the last tile: not used)
                slot = first < nvis ? offsets[base + (int)anchors[first]] : 0u;
            } else {  // the run's first slot and the kept items of the tiles before; the rank of its first visible anchor
                const uint32_t before = first & 64 ? (uint32_t)__builtin_amdgcn_readlane((int)run_tiles.y, index)
                                                   : (uint32_t)__builtin_amdgcn_readlane((int)run_tiles.x, index);
                slot = (uint32_t)__builtin_amdgcn_readlane((int)run_base.x, index) + (first & 32 ? before >> 16 : before & 0xFFFFu);
                run_rank = (uint32_t)__builtin_amdgcn_readlane((int)run_base.y, index);
            }
            {
                float* __restrict__ extra = my.rows[col] + kRowExtra;
                if (half == 0) {
#pragma unroll
                    for (int k = 0; k < 3; ++k) {
                        extra[k] = sc_ahead[k];
                        extra[3 + k] = ahead.pos[k];
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < 3; ++k) my.scale[col][k] = sc_ahead[k];
                }
            }
            const int nvis1 = seen.count();
            int base2 = 0, first2 = 0, index2 = 0;
            VisibleBytes bytes;
            if (unit + kEmitWaves < units) {  // uniform
                seen.pack(lane, my.anchors[buffer ^ 1]);
                wave_lds_sync();
                fetch(my.anchors[buffer ^ 1], base1, first1, nvis1);
                if (unit + 2 * kEmitWaves < units) {
                    locate(unit + 2 * kEmitWaves, base2, first2, index2);
                    bytes.load(d, base2, lane);
                }
            }

            // ---- opacity head; the kept items in the reference's order (anchor-major) ----
            // tanh itself is only evaluated for the offsets that are kept
            uint32_t mask = 0;
            run_head<1, kSplit, kWLo>(s_hi + kOpacityFrags, s_lo + kOpacityFrags, lane, s_bias, s_bias + 96, X, half,
                                      [&](int r, const floatx16& c) {
                                          mask = kept_rows(c, vis, half);
                                          store_rows(my.rows[col], r, n, half, c);
                                      });
            const uint32_t both = mask | (uint32_t)__shfl_xor((int)mask, 32, 64);
            const uint32_t mine = (uint32_t)__popc(both);
            uint32_t end = mine;  // inclusive prefix over the 32 anchors, the same in both halves
            end += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)end, 0x111, 0xf, 0xf, false);  // row_shr 1, 2, 4, 8
            end += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)end, 0x112, 0xf, 0xf, false);
            end += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)end, 0x114, 0xf, 0xf, false);
            end += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)end, 0x118, 0xf, 0xf, false);
            end += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)end, 0x142, 0xa, 0xf, false);  // row_bcast 15
            const uint32_t total = (uint32_t)__builtin_amdgcn_readlane((int)end, 31);
            while (mask) {  // each half lists the rows it holds
                const int m = __builtin_ctz(mask);
                my.list[end - mine + (uint32_t)__popc(both & ((1u << m) - 1u))] = (uint16_t)(16 * col + m);
                mask &= mask - 1u;
            }
            wave_lds_sync();
            // Items are in output order and slots come from a prefix of the kept counts, so the survivors of a tile
            // occupy consecutive output slots: lanes write consecutive addresses.
            // The learned offset of the lane's next survivor is requested ahead of its use.
            float of[3];
            auto fetch_offset = [&](uint32_t s) {
                const int it = (int)my.list[s < total ? s : 0];
                const float* __restrict__ src =
                    d.offset + ((size_t)(base + (int)anchors[first + (it >> 4)]) * n + (it & 15)) * 3;
#pragma unroll
                for (int k = 0; k < 3; ++k) of[k] = src[k];
            };
            if (total > 0) fetch_offset(lane);

            // ---- colour head; opacity, colour and position of the survivors ----
            run_head<1, kSplit, kWLo>(s_hi + kColourFrags, s_lo + (kWLo ? kColourFrags : 0), lane, s_bias + 64, s_bias + 224, X,
                                      half, [&](int r, const floatx16& c) {
                                          store_rows(my.rows[col] + kRowColour, r, 3 * n, half, c);
                                      });
            // the next tile's operands, before this tile's stores
            half8_t X1[kSplit ? 5 : 3];
            ahead.operand<kSplit>(d, cx, cy, cz, first1 + col < nvis1, half, X1);
            seen = bytes.look();
            wave_lds_sync();
            // training-mode by-products: tanh of every pre-activation of the visible anchors and the mask, indexed by
            // (visible anchor, offset): the tile's entries are the run's visible anchors first .. first + 31
            if (d.neural_opacity || d.kept_mask) {
                const size_t row0 = ((size_t)run_rank + (size_t)first) * (size_t)n;
                const int inv_n = (65536 + n - 1) / n;  // item / n == (item * inv_n) >> 16 for item < 32 n, n <= 10
                const int items = min(32, nvis - first) * n;
                for (int it = lane; it < items; it += 64) {
                    const int al = (it * inv_n) >> 16, m = it - al * n;
                    const float v = my.rows[al][m];
                    if (d.neural_opacity) d.neural_opacity[row0 + (size_t)it] = tanhf(v);
                    if (d.kept_mask) d.kept_mask[row0 + (size_t)it] = v > 0.0f ? 1 : 0;
                }
            }
            for (uint32_t s0 = 0; s0 < total; s0 += 64) {  // uniform
                const uint32_t s = s0 + lane, pos = slot + s;
                const float now_of[3] = {of[0], of[1], of[2]};
                if (s0 + 64 < total) fetch_offset(s + 64);
                if (s >= total || pos >= capacity) continue;  // the second cannot happen when capacity comes from the count pass
                const int it = (int)my.list[s], m = it & 15;
                const float* __restrict__ o = my.rows[it >> 4];
                opacity[pos] = tanhf(o[m]);
#pragma unroll
                for (int k = 0; k < 3; ++k) {
                    color[3 * (size_t)pos + k] = fast_sigmoid(o[kRowColour + 3 * m + k]);
                    xyz[3 * (size_t)pos + k] = o[kRowExtra + 3 + k] + now_of[k] * o[kRowExtra + k];
                }
            }
            wave_lds_sync();

            // ---- covariance head, over the same words; scaling and rotation of the survivors ----
            run_head<3, kSplit, kWLo>(s_hi + kCovFrags, s_lo + (kWLo ? kCovFrags : 0), lane, s_bias + 32, s_bias + 128, X, half,
                                      [&](int r, const floatx16& c) { store_rows(my.rows[col], r, 7 * n, half, c); });
            wave_lds_sync();
            for (uint32_t s0 = 0; s0 < total; s0 += 64) {  // uniform
                const uint32_t s = s0 + lane, pos = slot + s;
                if (s >= total || pos >= capacity) continue;
                const int it = (int)my.list[s];
                const float* __restrict__ c7 = my.rows[it >> 4] + 7 * (it & 15);
#pragma unroll
                for (int k = 0; k < 3; ++k) scaling_out[3 * (size_t)pos + k] = my.scale[it >> 4][k] * fast_sigmoid(c7[k]);
                const float q0 = c7[3], q1 = c7[4], q2 = c7[5], q3 = c7[6];
                // q / max(|q|, 1e-12) with one reciprocal square root (1 ulp) instead of a root and four divisions
                const float inv = __builtin_amdgcn_rsqf(fmaxf(q0 * q0 + q1 * q1 + q2 * q2 + q3 * q3, 1e-24f));
                rot[4 * (size_t)pos + 0] = q0 * inv;
                rot[4 * (size_t)pos + 1] = q1 * inv;
                rot[4 * (size_t)pos + 2] = q2 * inv;
                rot[4 * (size_t)pos + 3] = q3 * inv;
            }
            wave_lds_sync();
            base = base1, first = first1, index = index1, nvis = nvis1;
            base1 = base2, first1 = first2, index1 = index2;
#pragma unroll
            for (int k = 0; k < (kSplit ? 5 : 3); ++k) X[k] = X1[k];
        }
    }
}

// One workgroup: exclusive prefix of the per-run totals (kept offsets, visible anchors) and the grand totals.
__global__ __launch_bounds__(1024) void run_scan_kernel(const uint2* __restrict__ totals, uint2* __restrict__ base,
                                                        uint32_t runs, uint32_t* __restrict__ num_emitted,
                                                        uint32_t* __restrict__ num_visible)
{
    // eight consecutive totals per thread: one round for a million anchors (one each: eight rounds of three barriers and a
    // memory latency, 13 us); 4.7 us there, 3.0 at 60k (7.6 and 3.7 with 8-byte accesses and a scan by exchanges through LDS)
    constexpr int kItems = 8;
    __shared__ uint2 s_wave[16];
    __shared__ uint2 s_carry;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (threadIdx.x == 0) s_carry = make_uint2(0u, 0u);
    __syncthreads();
    for (uint32_t first = 0; first < runs; first += 1024 * kItems) {
        const uint32_t j = first + threadIdx.x * kItems;
        uint2 v[kItems];
        uint32_t sx = 0, sy = 0;
        const bool full = j + kItems <= runs;  // (16-byte accesses: half as many addresses)
        if (full) {
#pragma unroll
            for (int k = 0; k < kItems; k += 2) {
                const uint4 two = *reinterpret_cast<const uint4*>(totals + j + k);
                v[k] = make_uint2(two.x, two.y);
                v[k + 1] = make_uint2(two.z, two.w);
            }
        } else {
#pragma unroll
            for (int k = 0; k < kItems; ++k) v[k] = j + k < runs ? totals[j + k] : make_uint2(0u, 0u);
        }
#pragma unroll
        for (int k = 0; k < kItems; ++k) {
            sx += v[k].x;
            sy += v[k].y;
        }
        const uint32_t ix = wave_sum_scan(sx), iy = wave_sum_scan(sy);
        if (lane == 63) s_wave[wave] = make_uint2(ix, iy);
        __syncthreads();
        uint2 before = s_carry, all = make_uint2(0u, 0u);
#pragma unroll
        for (int w = 0; w < 16; ++w) {
            const uint2 t = s_wave[w];
            before.x += w < wave ? t.x : 0u;
            before.y += w < wave ? t.y : 0u;
            all.x += t.x;
            all.y += t.y;
        }
        before.x += ix - sx;
        before.y += iy - sy;
#pragma unroll
        for (int k = 0; k < kItems; k += 2) {
            const uint2 one = before, two = make_uint2(one.x + v[k].x, one.y + v[k].y);
            if (full) {
                *reinterpret_cast<uint4*>(base + j + k) = make_uint4(one.x, one.y, two.x, two.y);
            } else {
                if (j + k < runs) base[j + k] = one;
                if (j + k + 1 < runs) base[j + k + 1] = two;
            }
            before = make_uint2(two.x + v[k + 1].x, two.y + v[k + 1].y);
        }
        __syncthreads();
        if (threadIdx.x == 0) s_carry = make_uint2(s_carry.x + all.x, s_carry.y + all.y);
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        if (num_emitted) *num_emitted = s_carry.x;
        if (num_visible) *num_visible = s_carry.y;
    }
}

// Feature bank (anchor_decoder.py:163-177): a small MLP of the view direction (and the level) gives three softmax
// weights per anchor that mix the feature vector with its 4x and 2x strided copies:
//     feat'[j] = feat[4 (j mod 8)] w0 + feat[2 (j mod 16)] w1 + feat[j] w2 .
// fp32 throughout; the decode then reads the mixed features.  A workgroup takes 512 anchors: it lists the visible ones,
// finds the weights of each in a thread, and moves their features eight lanes to a row (a thread per anchor left three of
// four lanes idle behind a level-of-detail mask and read its row 16 bytes at a time: 67 us at 1M anchors, a quarter of
// them visible; now 19 for the 70 MB it moves).
struct BankArgs {
    int A, in_dim;  // 3 = view direction, 4 = view direction and level
    const float* anchor;
    const float* feat;
    const uint8_t* visible;
    const float* campos;
    const float* level;
    const float* w0;  // [32, in_dim]
    const float* b0;  // [32]
    const float* w1;  // [3, 32]
    const float* b1;  // [3]
    float* mixed;     // [A, 32]
};

constexpr int kBankAnchors = 512;  // per workgroup

__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(6, 8))) void feature_bank_kernel(BankArgs k)
{
    __shared__ float4 s_unit[kFeat][2];  // a hidden unit's input weights (of the level: zero without it) | bias, output weights
    __shared__ float s_b1[3];
    __shared__ uint16_t s_list[kBankAnchors];
    __shared__ float s_mix[kBankAnchors][3];
    __shared__ uint32_t s_count;
    const size_t first = (size_t)blockIdx.x * kBankAnchors;
    bool seen[kBankAnchors / 256];  // (requested ahead of the weights)
#pragma unroll
    for (int u = 0; u < kBankAnchors / 256; ++u) {
        const size_t a = first + 256 * u + threadIdx.x;
        seen[u] = a < (size_t)k.A && k.visible[min(a, (size_t)k.A - 1)] != 0;
    }
    if (threadIdx.x < kFeat) {
        const int h = threadIdx.x;
        const float* __restrict__ w = k.w0 + h * k.in_dim;
        s_unit[h][0] = make_float4(w[0], w[1], w[2], k.in_dim > 3 ? w[3] : 0.0f);
        s_unit[h][1] = make_float4(k.b0[h], k.w1[h], k.w1[kFeat + h], k.w1[2 * kFeat + h]);
    }
    if (threadIdx.x < 3) s_b1[threadIdx.x] = k.b1[threadIdx.x];
    if (threadIdx.x == 0) s_count = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int u = 0; u < kBankAnchors / 256; ++u) {
        const int i = 256 * u + (int)threadIdx.x;
        const uint64_t m = __ballot(seen[u]);
        uint32_t at = 0;
        if (lane == 0) at = atomicAdd(&s_count, (uint32_t)__popcll(m));
        at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
        if (__builtin_amdgcn_inverse_ballot_w64(m)) s_list[lanes_below_in(m, at)] = (uint16_t)i;  // (any order)
    }
    __syncthreads();
    const int count = (int)s_count;
    if (count == 0) return;  // (uniform)
    // The rows to mix, eight lanes each, 32 rows a round: those of the first four rounds are requested here and arrive while the
    // weights are computed, each later one when its place is free.  (One round after the other behind the weights: 31 us
    // for 346k anchors, most of them visible, 20 for 1M with 230k visible; now 24 and 17.)
    const int q = lane & 7, base = lane & ~7, mine = (int)(threadIdx.x >> 3);
    auto row_of = [&](int e0) { return (first + s_list[min(e0 + mine, count - 1)]) * (kFeat / 4) + q; };
    constexpr int kAhead = 4;
    float4 ahead[kAhead];
#pragma unroll
    for (int u = 0; u < kAhead; ++u) ahead[u] = reinterpret_cast<const float4*>(k.feat)[row_of(32 * u)];
    for (int e = threadIdx.x; e < count; e += 256) {
        const size_t a = first + s_list[e];
        float in[4];
        {
            float vx = k.anchor[3 * a] - k.campos[0], vy = k.anchor[3 * a + 1] - k.campos[1],
                  vz = k.anchor[3 * a + 2] - k.campos[2];
            const float dist = sqrtf(vx * vx + vy * vy + vz * vz);
            in[0] = vx / dist;
            in[1] = vy / dist;
            in[2] = vz / dist;
            in[3] = k.in_dim > 3 ? k.level[a] : 0.0f;
        }
        float logit[3] = {s_b1[0], s_b1[1], s_b1[2]};
#pragma unroll 8
        for (int h = 0; h < kFeat; ++h) {
            const float4 w = s_unit[h][0], u = s_unit[h][1];
            float v = u.x;
            v += w.x * in[0];
            v += w.y * in[1];
            v += w.z * in[2];
            v += w.w * in[3];
            v = fmaxf(v, 0.0f);
            logit[0] += u.y * v;
            logit[1] += u.z * v;
            logit[2] += u.w * v;
        }
        const float top = fmaxf(logit[0], fmaxf(logit[1], logit[2]));
        float w[3] = {expf(logit[0] - top), expf(logit[1] - top), expf(logit[2] - top)};
        const float sum = w[0] + w[1] + w[2];
#pragma unroll
        for (int o = 0; o < 3; ++o) s_mix[e][o] = w[o] / sum;
    }
    __syncthreads();
    // lane q of an anchor's eight holds f[4 q .. 4 q + 3]: f[4 m] is the first of lane m, f[2 m] of lane m / 2 the first or third
    for (int e1 = 0; e1 < count; e1 += 32 * kAhead) {
#pragma unroll
        for (int u = 0; u < kAhead; ++u) {
            const int e0 = e1 + 32 * u, e = min(e0 + mine, count - 1);
            if (e0 >= count) break;  // (uniform: every lane takes part in the exchange)
            const size_t row = row_of(e0);
            const float4 v = ahead[u];
            if (e0 + 32 * kAhead < count) ahead[u] = reinterpret_cast<const float4*>(k.feat)[row_of(e0 + 32 * kAhead)];
            const float w0 = s_mix[e][0], w1 = s_mix[e][1], w2 = s_mix[e][2];
            const float f[4] = {v.x, v.y, v.z, v.w};
            float o4[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                const float quarter = __shfl(v.x, base + 4 * (q & 1) + t, 64);
                const float half = __shfl((t & 1) ? v.z : v.x, base + 2 * (q & 3) + (t >> 1), 64);
                o4[t] = quarter * w0 + half * w1 + f[t] * w2;
            }
            if (e0 + mine < count)
                reinterpret_cast<float4*>(k.mixed)[row] = make_float4(o4[0], o4[1], o4[2], o4[3]);
        }
    }
}

}  // namespace

int check_decoder(const gs355_decoder* dec, const gs355_anchors* an)
{
    if (!dec || !an) return set_error(GS355_EINVAL, "decoder / anchors is NULL");
    if (dec->feat_dim != kFeat)
        return set_error(GS355_EINVAL, "anchor decode supports feat_dim 32 only (got %d)", dec->feat_dim);
    if (dec->n_offsets < 1 || dec->n_offsets > 10)
        return set_error(GS355_EINVAL, "anchor decode supports 1..10 offsets per anchor (got %d)", dec->n_offsets);
    if (an->A < 0) return set_error(GS355_EINVAL, "A must be >= 0 (got %d)", an->A);
    for (int j = 0; j < 3; ++j) {
        if (dec->add_level) {
            // the reference concatenates [feat | view | level] for every head once a level is given
            // (anchor_decoder.py:181-182), so a head built with a distance column as well cannot be fed
            if (dec->in_dim[j] != kFeat + 4)
                return set_error(GS355_EINVAL, "head %d: with add_level the input is [feat | view | level], 36 wide "
                                 "(got %d; a head with add_*_dist expects a width the reference never provides)",
                                 j, dec->in_dim[j]);
        } else if (dec->in_dim[j] != kFeat + 3 && dec->in_dim[j] != kFeat + 4) {
            return set_error(GS355_EINVAL, "head %d: input width must be 35 or 36 (got %d)", j, dec->in_dim[j]);
        }
        if (!dec->w0[j] || !dec->b0[j] || !dec->w1[j] || !dec->b1[j])
            return set_error(GS355_EINVAL, "head %d: weight or bias pointer is NULL", j);
    }
    if (dec->bank_in_dim != 0) {
        if (dec->bank_in_dim != 3 && dec->bank_in_dim != 4)
            return set_error(GS355_EINVAL, "bank_in_dim must be 0, 3 or 4 (got %d)", dec->bank_in_dim);
        if (!dec->bank_w0 || !dec->bank_b0 || !dec->bank_w1 || !dec->bank_b1)
            return set_error(GS355_EINVAL, "feature bank: weight or bias pointer is NULL");
    }
    if (an->A > 0 && (!an->anchor || !an->feat || !an->offset || !an->scaling || !an->visible_mask || !an->campos))
        return set_error(GS355_EINVAL, "anchor inputs must all be non-NULL");
    if (an->A > 0 && (dec->add_level || dec->bank_in_dim == 4) && !an->level)
        return set_error(GS355_EINVAL, "anchors.level is NULL but the decoder takes the level as an input");
    if (an->A > 0 && (reinterpret_cast<uintptr_t>(an->feat) & 15u) != 0)
        return set_error(GS355_EINVAL, "anchor features must be 16-byte aligned");
    return GS355_OK;
}

static int fill_args(const gs355_decoder* dec, const gs355_anchors* an, bool allow_bank, DecodeArgs* out)
{
    if (dec && dec->bank_in_dim != 0 && !allow_bank)
        return set_error(GS355_EINVAL, "the feature bank is supported by gs355_decode only");
    const int rc = check_decoder(dec, an);
    if (rc) return rc;
    DecodeArgs a;
    a.A = an->A;
    a.n = dec->n_offsets;
    a.anchor = an->anchor;
    a.feat = an->feat;
    a.offset = an->offset;
    a.scaling = an->scaling;
    a.visible = an->visible_mask;
    a.campos = an->campos;
    a.level = dec->add_level ? an->level : nullptr;
    a.split_feat = (dec->fp32_features || dec->bank_in_dim != 0) ? 1 : 0;  // bank-mixed features are general floats
    a.weights_lo = dec->fp32_weights ? 1 : 0;
    for (int j = 0; j < 3; ++j) {
        a.in_dim[j] = dec->in_dim[j];
        a.w0[j] = dec->w0[j];
        a.b0[j] = dec->b0[j];
        a.w1[j] = dec->w1[j];
        a.b1[j] = dec->b1[j];
    }
    a.run_totals = nullptr;
    a.run_tiles = nullptr;
    a.run_base = nullptr;
    a.scan_here = 0;
    a.num_emitted = nullptr;
    a.num_visible = nullptr;
    a.neural_opacity = nullptr;
    a.kept_mask = nullptr;
    *out = a;
    return GS355_OK;
}

int launch_run_scan(const uint2* totals, uint2* base, uint32_t runs, uint32_t* num_emitted, uint32_t* num_visible,
                    hipStream_t s)
{
    hipLaunchKernelGGL(run_scan_kernel, dim3(1), dim3(1024), 0, s, totals, base, runs, num_emitted, num_visible);
    GS355_CHECK_LAUNCH("decode: run scan");
    return GS355_OK;
}

static uint32_t run_count(int A) { return (uint32_t)(((size_t)A + kRun - 1) / kRun); }

// Launch the count or the emit pass in the variant the features and the weights need.
// Persistent workgroups, at most what the chip holds at once: the weights are fetched once per resident workgroup.
static void launch_count(hipStream_t s, const DecodeArgs& a, uint32_t* counts)
{
    const uint32_t runs = run_count(a.A);
    const int shared_run = runs <= (uint32_t)kCountCap ? 1 : 0;
    const dim3 grid(runs < (uint32_t)kCountCap ? runs : (uint32_t)kCountCap), block(64 * kCountWaves);
#define GS355_COUNT(S, W) hipLaunchKernelGGL((decode_count_kernel<S, W>), grid, block, 0, s, a, counts, shared_run)
    if (a.split_feat && a.weights_lo) GS355_COUNT(true, true);
    else if (a.split_feat) GS355_COUNT(true, false);
    else if (a.weights_lo) GS355_COUNT(false, true);
    else GS355_COUNT(false, false);
#undef GS355_COUNT
}

static void launch_emit(hipStream_t s, const DecodeArgs& a, const uint32_t* offsets, uint32_t capacity, const gs355_decoded& o)
{
    const uint32_t runs = run_count(a.A);
    const dim3 grid(runs < (uint32_t)kEmitCap ? runs : (uint32_t)kEmitCap), block(64 * kEmitWaves);
#define GS355_EMIT(S, W)                                                                                              \
    hipLaunchKernelGGL((decode_emit_kernel<S, W>), grid, block, 0, s, a, offsets, capacity, o.xyz, o.color, o.opacity, \
                       o.scaling, o.rot)
    if (a.split_feat && a.weights_lo) GS355_EMIT(true, true);
    else if (a.split_feat) GS355_EMIT(true, false);
    else if (a.weights_lo) GS355_EMIT(false, true);
    else GS355_EMIT(false, false);
#undef GS355_EMIT
}

}  // namespace gs355

using namespace gs355;

// ---- gs355_decode_count for callers that cannot allocate -----------------------------------------------------
// The scan's block sums live in a file-scope device array instead of a caller-provided scratch buffer.  Every
// GPU holds its own copy of the array at its own address; host code never uses the array's name as an address
// (it is a host-side stand-in) but the pointer hipGetSymbolAddress returns for the current device, resolved
// once per device and kept.
constexpr int32_t kStaticCountMaxAnchors = 1 << 24;
constexpr size_t kStaticScratchWords = ((size_t)kStaticCountMaxAnchors / kScanTile) * 3 + 8 + 64;
static __device__ __align__(256) uint32_t scratch[kStaticScratchWords];

constexpr int kMaxDevices = 64;
static std::atomic<uint32_t*> g_scratch_ptr[kMaxDevices];

static int static_scratch(uint32_t** out)
{
    int dev = -1;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return set_error(GS355_EHIP, "hipGetDevice: %s", hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices) return set_error(GS355_EINVAL, "device index %d is outside [0, %d)", dev, kMaxDevices);
    uint32_t* p = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!p) {
        void* q = nullptr;
        e = hipGetSymbolAddress(&q, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !q)
            return set_error(GS355_EHIP, "hipGetSymbolAddress(scratch) on device %d: %s", dev, hipGetErrorString(e));
        p = static_cast<uint32_t*>(q);
        g_scratch_ptr[dev].store(p, std::memory_order_release);  // racing threads resolve the same address
    }
    *out = p;
    return GS355_OK;
}

extern "C" {

int gs355_decode_scratch_bytes(int32_t A, size_t* bytes)
{
    if (!bytes) return set_error(GS355_EINVAL, "bytes is NULL");
    if (A < 0) return set_error(GS355_EINVAL, "A must be >= 0 (got %d)", A);
    *bytes = scan_tmp_words((size_t)A) * sizeof(uint32_t) + 256;
    return GS355_OK;
}

int gs355_decode_count(const gs355_decoder* dec, const gs355_anchors* an, uint32_t* counts, uint32_t* offsets,
                       void* scratch_buf, size_t scratch_bytes, void* stream)
{
    DecodeArgs a;
    int rc = fill_args(dec, an, false, &a);
    if (rc) return rc;
    if (a.A == 0) return GS355_OK;
    if (!counts || !offsets || !scratch_buf) return set_error(GS355_EINVAL, "counts / offsets / scratch is NULL");
    size_t need = 0;
    gs355_decode_scratch_bytes(a.A, &need);
    if (scratch_bytes < need)
        return set_error(GS355_ENOSPC, "decode scratch has %zu bytes, %zu needed", scratch_bytes, need);
    hipStream_t s = static_cast<hipStream_t>(stream);
    launch_count(s, a, counts);
    GS355_CHECK_LAUNCH("decode: count");
    return launch_exclusive_scan(counts, offsets, (size_t)a.A, static_cast<uint32_t*>(scratch_buf), s);
}

int gs355_decode_count_static(const gs355_decoder* dec, const gs355_anchors* an, uint32_t* counts, uint32_t* offsets,
                              void* stream)
{
    DecodeArgs a;
    int rc = fill_args(dec, an, false, &a);
    if (rc) return rc;
    if (a.A > kStaticCountMaxAnchors)
        return set_error(GS355_ENOSPC, "gs355_decode_count_static handles at most %d anchors (got %d); use gs355_decode_count",
                         kStaticCountMaxAnchors, a.A);
    if (a.A == 0) return GS355_OK;
    if (!counts || !offsets) return set_error(GS355_EINVAL, "counts / offsets is NULL");
    static_assert(kStaticScratchWords * sizeof(uint32_t) >=
                      (((size_t)kStaticCountMaxAnchors + kScanTile - 1) / kScanTile * 3 + 8) * sizeof(uint32_t) + 256,
                  "static scratch covers the scan of the largest accepted anchor count");
    uint32_t* tmp = nullptr;
    if ((rc = static_scratch(&tmp))) return rc;
    hipStream_t s = static_cast<hipStream_t>(stream);
    launch_count(s, a, counts);
    GS355_CHECK_LAUNCH("decode: count");
    // the scan writes every block sum before it reads it: nothing in the array has to start at zero
    return launch_exclusive_scan(counts, offsets, (size_t)a.A, tmp, s);
}

int gs355_decode_emit(const gs355_decoder* dec, const gs355_anchors* an, const uint32_t* offsets, int64_t capacity,
                      const gs355_decoded* out, void* stream)
{
    DecodeArgs a;
    int rc = fill_args(dec, an, false, &a);
    if (rc) return rc;
    if (a.A == 0 || capacity == 0) return GS355_OK;
    if (capacity < 0 || capacity > 0xFFFFFFFFll)
        return set_error(GS355_EINVAL, "capacity must be in [0, 2^32) (got %lld)", (long long)capacity);
    if (!offsets) return set_error(GS355_EINVAL, "offsets is NULL");
    if (!out || !out->xyz || !out->color || !out->opacity || !out->scaling || !out->rot)
        return set_error(GS355_EINVAL, "decoded outputs must all be non-NULL");
    hipStream_t s = static_cast<hipStream_t>(stream);
    launch_emit(s, a, offsets, (uint32_t)capacity, *out);
    GS355_CHECK_LAUNCH("decode: emit");
    return GS355_OK;
}

namespace {
struct FusedLayout {
    size_t run_totals, run_tiles, run_base, mixed, total;
};
FusedLayout fused_layout(int32_t A, int32_t n, bool bank)
{
    auto up = [](size_t v) { return (v + 255) / 256 * 256; };
    const size_t runs = run_count(A);
    FusedLayout L;
    size_t off = 0;
    (void)n;
    L.run_totals = off;
    off = up(off + runs * sizeof(uint2) + 8);
    L.run_tiles = off;
    off = up(off + runs * sizeof(uint2) + 8);
    L.run_base = off;
    off = up(off + runs * sizeof(uint2) + 8);
    L.mixed = off;
    if (bank) off = up(off + (size_t)A * kFeat * sizeof(float) + 4);
    L.total = off;
    return L;
}
}  // namespace

int gs355_decode_workspace_bytes(int32_t A, int32_t n_offsets, int32_t with_feature_bank, size_t* bytes)
{
    if (!bytes) return set_error(GS355_EINVAL, "bytes is NULL");
    if (A < 0) return set_error(GS355_EINVAL, "A must be >= 0 (got %d)", A);
    if (n_offsets < 1 || n_offsets > 10)
        return set_error(GS355_EINVAL, "anchor decode supports 1..10 offsets per anchor (got %d)", n_offsets);
    *bytes = fused_layout(A, n_offsets, with_feature_bank != 0).total;
    return GS355_OK;
}

int gs355_decode(const gs355_decoder* dec, const gs355_anchors* an, int64_t capacity, const gs355_decoded* out,
                 void* workspace, size_t workspace_bytes, uint32_t phases, void* stream)
{
    if (phases == 0 || (phases & ~(uint32_t)(GS355_DECODE_COUNT | GS355_DECODE_EMIT)) != 0)
        return set_error(GS355_EINVAL, "phases must be GS355_DECODE_COUNT, GS355_DECODE_EMIT or both (got 0x%x)", phases);
    const bool do_count = (phases & GS355_DECODE_COUNT) != 0, do_emit = (phases & GS355_DECODE_EMIT) != 0;
    DecodeArgs a;
    int rc = fill_args(dec, an, true, &a);
    if (rc) return rc;
    if (capacity < 0 || capacity > 0xFFFFFFFFll)
        return set_error(GS355_EINVAL, "capacity must be in [0, 2^32) (got %lld)", (long long)capacity);
    if (!out) return set_error(GS355_EINVAL, "decoded outputs is NULL");
    if (do_emit && capacity > 0 && (!out->xyz || !out->color || !out->opacity || !out->scaling || !out->rot))
        return set_error(GS355_EINVAL, "decoded outputs must all be non-NULL");
    const bool bank = dec->bank_in_dim != 0;
    const FusedLayout L = fused_layout(a.A, a.n, bank);
    if (a.A > 0) {
        if (!workspace) return set_error(GS355_EINVAL, "workspace is NULL");
        if ((reinterpret_cast<uintptr_t>(workspace) & 255u) != 0)
            return set_error(GS355_EINVAL, "workspace must be 256-byte aligned");
        if (workspace_bytes < L.total)
            return set_error(GS355_ENOSPC, "decode workspace has %zu bytes, %zu needed", workspace_bytes, L.total);
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (a.A == 0) {
        if (do_count && out->count && (rc = launch_fill_u32(out->count, 1, 0u, s))) return rc;
        if (do_count && out->num_visible && (rc = launch_fill_u32(out->num_visible, 1, 0u, s))) return rc;
        return GS355_OK;
    }
    char* ws = static_cast<char*>(workspace);
    const uint32_t runs = run_count(a.A);
    if (bank) a.feat = reinterpret_cast<float*>(ws + L.mixed);  // written by the count phase, read by both passes
    uint2* run_base = reinterpret_cast<uint2*>(ws + L.run_base);
    a.run_totals = reinterpret_cast<uint2*>(ws + L.run_totals);
    a.run_tiles = reinterpret_cast<uint2*>(ws + L.run_tiles);
    const bool emits = do_emit && (capacity > 0 || out->neural_opacity || out->mask);
    a.scan_here = do_count && emits && runs <= (uint32_t)(kScanStripes * kEmitCap);
    if (do_count) {
        if (bank) {
            BankArgs b;
            b.A = a.A;
            b.in_dim = dec->bank_in_dim;
            b.anchor = a.anchor;
            b.feat = an->feat;
            b.visible = a.visible;
            b.campos = a.campos;
            b.level = an->level;
            b.w0 = dec->bank_w0;
            b.b0 = dec->bank_b0;
            b.w1 = dec->bank_w1;
            b.b1 = dec->bank_b1;
            b.mixed = reinterpret_cast<float*>(ws + L.mixed);
            hipLaunchKernelGGL(feature_bank_kernel, dim3((a.A + kBankAnchors - 1) / kBankAnchors), dim3(256), 0, s, b);
            GS355_CHECK_LAUNCH("decode: feature bank");
        }
        launch_count(s, a, nullptr);
        GS355_CHECK_LAUNCH("decode: count");
        if (!a.scan_here && (rc = launch_run_scan(a.run_totals, run_base, runs, out->count, out->num_visible, s))) return rc;
    }
    if (!emits) return GS355_OK;
    a.run_base = run_base;
    a.num_emitted = out->count;
    a.num_visible = out->num_visible;
    a.neural_opacity = out->neural_opacity;
    a.kept_mask = out->mask;
    launch_emit(s, a, nullptr, (uint32_t)capacity, *out);
    GS355_CHECK_LAUNCH("decode: emit");
    return GS355_OK;
}

}  // extern "C"
