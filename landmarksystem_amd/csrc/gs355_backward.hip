// Backward pass of the rasterizer for gfx950: the gradients the reference's training loop pulls through
// GaussianRasterizer.forward (loss.backward() at benchmarks/nerf/origin_gs/gs_trainer.py:117-124; the
// screen-space gradient of `means2D` feeds densification, landmark/nerf_components/model_components/fields/
// encodings/gaussian_encoding.py:729-743).
//
// Kernels over the forward pass's workspace (records, sorted values, ranges), in their order:
//   record_slots     where each Gaussian's records of the next kernel go: one per tile number of its region, side by side
//   blend_backward   per 16x16 tile, the forward blend's walk repeated FRONT TO BACK with the same per-block
//                    lists and the same per-pair decisions.  With f_i = colour_i . dL/dpixel, w_i = alpha_i T_i,
//                    prefix P_i = sum_{j<=i} w_j f_j and R = out_pixel . dL/dpixel - T_final dL/dalpha_out (all
//                    known from the forward outputs), dL/dalpha_i = T_i f_i - (R - P_i) / (1 - alpha_i): no
//                    division by a transmittance and no second, reversed walk.  Per-pair contributions are summed
//                    over the 16 pixels of a block four list entries at a time, added to the wavefront's own sums of
//                    the staged Gaussians in LDS (no atomics), and written once per batch of 64 as one 36-byte
//                    record (48 with a depth gradient) per (tile, Gaussian) key.  No global atomics (they cost
//                    more than the rest of the kernel): the records of a Gaussian are consecutive, in the order its tile region is
//                    walked, and are summed in that order, so gradients are identical from run to run.
//   sum_large        (scenes of up to 262144 Gaussians) the records of Gaussians of many tiles, summed by many lanes
//   preprocess_backward  per Gaussian: conic -> 2-D covariance -> Jacobian / 3-D covariance -> scale, rotation,
//                    mean; pixel position -> mean; colour -> SH coefficients and view direction -> mean.
// min(0.99, opacity * G) passes the gradient unchanged, and the `means2D` gradient is in normalised device units
// (pixel gradient times W/2, H/2), as the published backward pass of this rasterizer family does.
#include <type_traits>

#include "gs355_internal.h"

namespace gs355 {

namespace {

// Per-key record, three parts of N floats: (dpx, dpy, dconic x), (dconic y, dconic z, dopacity), (dr, dg, db), or where a
// gradient arrives for the depth plane (dpx, dpy, dconic x, dconic y), (dconic z, dopacity, dr, dg), (db, ddepth, 0, 0).
// 36 bytes in the place of 48 where the depth has none: preprocess backward of 6M Gaussians 724 -> 707 us, of 550k decoded
// ones 57 -> 54, record sums of 100k large splats 40 -> 38.
template <bool kDepth>
constexpr int kPartFloats = kDepth ? 4 : 3;
static_assert(3 * kPartFloats<true> == GS355_KEY_GRAD_FLOATS, "the scratch holds a record of the larger kind per key");
template <int N>
struct RecordPart {
    float v[N];
    static __device__ __forceinline__ RecordPart load(const float* __restrict__ p)
    {
        RecordPart r;
#pragma unroll
        for (int k = 0; k < N; ++k) r.v[k] = p[k];
        return r;
    }
    __device__ __forceinline__ void store(float* __restrict__ p) const
    {
#pragma unroll
        for (int k = 0; k < N; ++k) p[k] = v[k];
    }
    __device__ __forceinline__ void add(const RecordPart& o)
    {
#pragma unroll
        for (int k = 0; k < N; ++k) v[k] = v[k] + o.v[k];
    }
};

// Where a Gaussian's records lie: those of its tile region (TileRegion), by tile number, from some first slot on.  The blend
// needs the slot of one tile (tx, ty) per key: base + ty * width + tx with base = first - y0 * width - x0 (modulo 2^32),
// eight bytes from one place (first slot and rectangle took two cache lines per key, of the four to five that a key costs: blend
// backward 1109 -> 1013 us at 6M Gaussians, 1080p).
struct RecordSlots {
    uint32_t base, width;
};
// The records of a region: slot first + e for tile number e of n, of the tiles the region holds (the others have no key, and
// their slots are not written).
struct RecordRun {
    uint32_t first, n, mask;
    bool masked, spans;
    __device__ __forceinline__ uint32_t keys() const { return masked ? (uint32_t)__popc(mask) : n; }  // (an upper bound with spans)
};
__device__ __forceinline__ RecordRun record_run(RecordSlots s, const TileRegion& q)
{
    if (s.width == 0u) return {0u, 0u, 0u, false, false};  // no tiles, or a frame that overflowed
    return {s.base + (uint32_t)q.y0 * s.width + (uint32_t)q.x0, (uint32_t)q.area, q.mask, q.masked, q.spans};
}

// Slots of all Gaussians: a workgroup adds up the rectangles of its 8192 Gaussians and takes that many slots from one
// counter (1024 Gaussians per request: 73 us at 6M Gaussians, the requests being served one after the other).  Which
// workgroup gets which slots varies between runs, the order of a Gaussian's own records does not, and nothing else enters
// a sum.  A frame that overflowed its capacity has no records, and no room for them: no Gaussian has slots.
constexpr int kSlotItems = 8, kSlotThreads = 1024;
__global__ __launch_bounds__(kSlotThreads) void record_slots_kernel(int P, bool plain, const gs355_header* __restrict__ header,
                                                                    const uint64_t* __restrict__ rects,
                                                                    uint32_t* __restrict__ next,
                                                                    RecordSlots* __restrict__ slots)
{
    __shared__ uint32_t s_wave[kSlotThreads / 64], s_first;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int first = (int)blockIdx.x * kSlotItems * kSlotThreads + (int)threadIdx.x;
    const int end = header->overflow ? 0 : P;
    uint64_t rect[kSlotItems];
#pragma unroll
    for (int k = 0; k < kSlotItems; ++k) rect[k] = first + k * kSlotThreads < end ? rects[first + k * kSlotThreads] : 0ull;
    uint32_t sum = 0;
#pragma unroll
    for (int k = 0; k < kSlotItems; ++k) sum += (uint32_t)TileRegion(rect[k], plain).area;
    uint32_t inc = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t up = __shfl_up(inc, d, 64);
        if (lane >= d) inc += up;
    }
    if (lane == 63) s_wave[wave] = inc;
    __syncthreads();
    uint32_t before = 0, all = 0;
#pragma unroll
    for (int w = 0; w < kSlotThreads / 64; ++w) {
        before += w < wave ? s_wave[w] : 0u;
        all += s_wave[w];
    }
    if (threadIdx.x == 0) s_first = atomicAdd(next, all);
    __syncthreads();
    uint32_t at = s_first + before + inc - sum;
#pragma unroll
    for (int k = 0; k < kSlotItems; ++k) {
        const TileRegion q(rect[k], plain);
        const uint32_t width = (uint32_t)q.width;
        const RecordRun run = record_run({0u, width}, q);  // (its first: the slot of the region's corner)
        if (first + k * kSlotThreads < P) slots[first + k * kSlotThreads] = {at - run.first, width};
        at += run.n;
    }
}

// Value of lane `kLane` of each quad of lanes, in all four of them.
template <int kLane>
__device__ __forceinline__ float quad_lane(float v)
{
    constexpr int kCtrl = kLane * 0x55;  // quad_perm [k, k, k, k]
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xf, 0xf, false));
}

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// Sums over the four 16-lane rows, two values at a time: after the swap of lane halves (kLanes = 32) or of neighbouring
// rows (16) one register holds the first value's two parts where the other holds the second's, and one addition
// leaves the first value's partial sum in the lower half (even rows), the second's in the upper (odd rows).
template <int kLanes>
__device__ __forceinline__ float add_halves(float a, float b)
{
    const unsigned ua = (unsigned)__float_as_int(a), ub = (unsigned)__float_as_int(b);
    u32x2 r;
    if (kLanes == 32) r = __builtin_amdgcn_permlane32_swap(ua, ub, false, false);
    else r = __builtin_amdgcn_permlane16_swap(ua, ub, false, false);
    return __int_as_float((int)r.x) + __int_as_float((int)r.y);
}

// Lane layout of a wavefront's 8x8 quadrant: lane = 16 q + 4 b + i is pixel i of row q of the 4x4 block b.  Per step a
// block's pixels produce two values each, d = dL/dpower and w = alpha T, and ten sums over the sixteen pixels are wanted:
// the moments of d over the offsets from the splat's centre, and w against the four channels of dL/dpixel.  Four steps
// are reduced together:
//   - a matrix instruction per value and step (4x4x1, sixteen blocks of four lanes, K = 1; value times a one-hot row)
//     hands step s's four values of a quad to the quad's lane s, so that lane (q, b, s) holds row q of step s in four
//     registers: a transposition for eight cycles each;
//   - the sums over a row are then additions inside a lane, every one serving four steps;
//   - the sums over the rows pair up values through lane swaps (add_halves): ten values, sixteen instructions, and each
//     row ends with the totals of its own two or three.
// Reducing each step by itself with lane exchanges took 53 vector instructions per step, more than the gradient
// arithmetic; this takes about 20.  Blend backward at 6M Gaussians / 1080p: 1.34 -> 1.25 ms, 622M -> 491M vector
// instructions, LDS pipe 73 -> 37 % busy (493M and 38 % with the check for sums that are not finite, 0.4 % of a
// step).  Larger matrix instructions do not pay for the sums (1.45 ms): fp32 ones occupy the SIMD like the vector
// instructions they replace.
// kDepth: a gradient arrives for the depth plane.
template <bool kDepth>
__global__ __launch_bounds__(256) void blend_backward_kernel(
    FrameArgs f, const gs355_header* __restrict__ header, const uint32_t* __restrict__ ranges, const uint4* __restrict__ order,
    const uint32_t* __restrict__ values, const float* __restrict__ records, const float* __restrict__ image,
    const float* __restrict__ out_depth, const float* __restrict__ out_alpha, const float* __restrict__ g_image,
    const float* __restrict__ g_depth, const float* __restrict__ g_alpha, const RecordSlots* __restrict__ slots,
    float* __restrict__ key_grads)
{
    // staged Gaussians per round, four threads each (96 and 128 measured 1 and 9 % slower: fewer resident workgroups)
    constexpr int kBatch = 64;
    // (entry kBatch: the null record, zero conic and log2(opacity) = -inf, which no pixel accepts; nothing reads its sums)
    __shared__ float4 s_a[kBatch + 1];  // px, py, -conic_x / 2, -conic_y   (rescaled as the forward blend stages them)
    __shared__ float4 s_b[kBatch + 1];  // -conic_z / 2, log2(opacity), r, g
    __shared__ float4 s_c[kBatch + 1];  // b, depth, mask of the blocks it can reach, unused
    // Sums of each wavefront: of d, d dx | d dy, d dy^2 | d dx dy, green | red, blue | d dx^2, depth.  A wavefront owns
    // its sums and serves its four blocks one after the other, so plain reads and writes do: float atomics on sums
    // shared by the workgroup take almost two cycles per lane of the CU's one LDS pipe, which bounded the kernel
    // (LDS pipe busy 73 %, whatever the vector instructions were reduced to).
    __shared__ float2 s_sum[4][kBatch + 1][5];
    __shared__ uint32_t s_slot[kBatch];  // where each staged Gaussian's record goes
    __shared__ uint32_t s_wave_done[4];
    __shared__ __align__(4) uint8_t s_list[4][4][kBatch + 8];

    if (header->overflow) return;
    const BlendTile list(header, ranges, order);
    const int tile = (int)list.tile;
    const int tile_x = tile % f.grid_x, tile_y = tile / f.grid_x;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int row = lane >> 4, group = (lane >> 2) & 3, sub = lane & 3;
    const int qx0 = tile_x * kTile + (wave & 1) * 8, qy0 = tile_y * kTile + (wave >> 1) * 8;
    const int px = qx0 + (group & 1) * 4 + sub, py = qy0 + (group >> 1) * 4 + row;
    const bool inside = px < f.W && py < f.H;
    const float pxf = (float)px, pyf = (float)py;
    const int first_bit = 8 * (wave >> 1) + 2 * (wave & 1);  // the quadrant's first block in a record's mask
    constexpr uint64_t kBlockLanes = 0x000F000F000F000Full;  // block 0's lanes: four of each row

    float g0 = 0.f, g1 = 0.f, g2 = 0.f, g3 = 0.f;  // dL/d(r, g, b, depth) of this pixel
    float R = 0.f;                                 // out . g - T_final * dL/dalpha_out
    if (inside) {
        const size_t plane = (size_t)f.W * f.H;
        const size_t o = (size_t)py * f.W + px;
        g0 = g_image[o];
        g1 = g_image[plane + o];
        g2 = g_image[2 * plane + o];
        R = image[o] * g0 + image[plane + o] * g1 + image[2 * plane + o] * g2;
        if (kDepth) {
            g3 = g_depth[o];
            R += out_depth[o] * g3;
        }
        if (g_alpha) R -= (1.0f - out_alpha[o]) * g_alpha[o];
    }
    const f32x4 zero4 = {0.f, 0.f, 0.f, 0.f};
    const bool finite_g = __ballot(!(fabsf(g0) + fabsf(g1) + fabsf(g2) + fabsf(g3) < __builtin_inff())) == 0ull;
    // 1 in the lanes of a constant mask (one instruction, and no register held for it)
    auto ones = [](uint64_t lanes) { return __builtin_amdgcn_inverse_ballot_w64(lanes) ? 1.0f : 0.0f; };
    // staging: thread 4 k + part brings part `part` of the batch's Gaussian k (part 3: the slot of its record), and later
    // writes a third of its record
    const int staged = tid >> 2, part = tid & 3;
    const uint32_t lo = list.lo, hi = list.hi;
    float T = inside ? 1.0f : -1.0f, prefix = 0.0f;
    if (tid < 3)
        (tid == 0 ? s_a : tid == 1 ? s_b : s_c)[kBatch] = make_float4(0.f, tid == 1 ? -__builtin_inff() : 0.f, 0.f, 0.f);

    for (int k = tid; k < 4 * (kBatch + 1) * 5; k += 256) (&s_sum[0][0][0])[k] = make_float2(0.f, 0.f);

    uint32_t base = lo;
    // of this batch's Gaussian; requested one batch ahead (6M Gaussians 874 -> 861 us; the records themselves ahead, too, cost
    // a wavefront per SIMD: 870)
    uint32_t index = lo + staged < hi ? values[lo + staged] : 0u;
    for (; base < hi; base += kBatch) {
        const uint64_t live = __ballot(T > 0.0f);
        const bool wave_done = live == 0ull;
        if (lane == 0) s_wave_done[wave] = wave_done ? 1u : 0u;
        const int count = (int)min((uint32_t)kBatch, hi - base);
        if (staged < count) {
            const uint32_t g = index;
            if (base + kBatch + staged < hi) index = values[base + kBatch + staged];
            float4 v = reinterpret_cast<const float4*>(records + (size_t)g * kRecordFloats)[min(part, 2)];
            if (part == 3) {
                const RecordSlots at = slots[g];
                s_slot[staged] = at.base + (uint32_t)tile_y * at.width + (uint32_t)tile_x;
            }
            // thread `part` tests the tile's block row `part`
            const TileReach reach(quad_lane<0>(v.x), quad_lane<0>(v.y), quad_lane<0>(v.z), quad_lane<0>(v.w),
                                  quad_lane<1>(v.x), quad_lane<2>(v.z), quad_lane<2>(v.w), (float)(tile_x * kTile),
                                  (float)(tile_y * kTile));
            const float row_mask = __uint_as_float(reach.unless_infinite(reach.row((float)part), 0xFu) << (4 * part));
            const uint32_t mask = __float_as_uint(quad_lane<0>(row_mask)) | __float_as_uint(quad_lane<1>(row_mask)) |
                                  __float_as_uint(quad_lane<2>(row_mask)) | __float_as_uint(quad_lane<3>(row_mask));
            if (part == 0) {
                v.z *= -0.5f;
                v.w = -v.w;
            } else if (part == 1) {  // (as the forward blend: a negative opacity never blends)
                v.x *= -0.5f;
                v.y = __builtin_amdgcn_logf(v.y < 0.0f ? 0.0f : v.y);
            } else {
                v.z = __uint_as_float(mask);
            }
            if (part < 3) (part == 0 ? s_a : part == 1 ? s_b : s_c)[staged] = v;
        } else if (part == 2) {
            s_c[staged].z = 0.0f;  // (no record: reaches no block)
        }
        __syncthreads();
        if ((s_wave_done[0] & s_wave_done[1] & s_wave_done[2] & s_wave_done[3]) != 0u) break;
        if (!wave_done) {
            // ---- lists: which staged Gaussians reach which 4x4 block (lane = Gaussian), as the forward blend ----
            uint32_t len[4] = {0u, 0u, 0u, 0u};
            {
                const uint32_t reached = __float_as_uint(s_c[lane].z) >> first_bit;
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    if ((live & (kBlockLanes << (4 * b))) == 0ull) continue;  // (all of the block's pixels have finished)
                    const uint64_t m = __ballot((reached & (1u << (4 * (b >> 1) + (b & 1)))) != 0u);
                    if (__builtin_amdgcn_inverse_ballot_w64(m)) s_list[wave][b][lanes_below_in(m)] = (uint8_t)lane;
                    len[b] = (uint32_t)__popcll(m);
                }
            }
            const uint32_t longest = (uint32_t)__builtin_amdgcn_readfirstlane(
                (int)max(max(len[0], len[1]), max(len[2], len[3])));
            const uint32_t quads = (longest + 3u) / 4u;
            // every block's lanes pad its list with the null record up to the common length
            uint32_t own = len[0];
            own = group == 1 ? len[1] : own;
            own = group == 2 ? len[2] : own;
            own = group == 3 ? len[3] : own;
            for (uint32_t at = own + (uint32_t)(4 * row + sub); at < quads * 4u; at += 16u) s_list[wave][group][at] = (uint8_t)kBatch;
            wave_lds_sync();
            const uint32_t* __restrict__ mine = reinterpret_cast<const uint32_t*>(s_list[wave][group]);
            uint32_t next = mine[0];  // read ahead by one round (rounds past the end are never used)
            for (uint32_t i = 0; i < quads; ++i) {
                const uint32_t entries = next;
                next = mine[i + 1];
                float d[4], w[4];
                uint64_t any = 0ull;
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    // One entry per block.  b.y is log2(opacity): opacity * exp(power) is evaluated exactly as the
                    // forward blend evaluates it (decided on the exponent before the exp2), so both passes take the
                    // same decisions.  T carries the forward blend's state (sign = finished).
                    d[s] = w[s] = 0.0f;
                    const uint32_t k = (entries >> (8 * s)) & 0xFFu;
                    const float4 a = s_a[k], b = s_b[k];
                    const float dx = a.x - pxf, dy = a.y - pyf;
                    const float power = pair_exponent(dx, dy, a.z, a.w, b.x);
                    const float t = __builtin_fmaf(power, 1.4426950408889634f, b.y);
                    const uint64_t accept = __ballot(!(power > 0.0f)) & __ballot(!(t < kAlphaCut));
                    if (accept != 0ull) {
                        const float raw = __builtin_amdgcn_exp2f(t);  // opacity * exp(power)
                        const float alpha = fminf(0.99f, raw);
                        const float test_T = __builtin_fmaf(-alpha, T, T);  // T - alpha T, as the forward blend forms it
                        const uint64_t hit = accept & __ballot(test_T >= 0.0001f);
                        if (__builtin_amdgcn_inverse_ballot_w64(accept & ~hit)) T = -fabsf(T);
                        any |= hit;
                        if (__builtin_amdgcn_inverse_ballot_w64(hit)) {
                            const float2 c = *reinterpret_cast<const float2*>(&s_c[k]);
                            w[s] = alpha * T;
                            float fg = b.z * g0 + b.w * g1 + c.x * g2;
                            if (kDepth) fg = __builtin_fmaf(c.y, g3, fg);
                            prefix = __builtin_fmaf(w[s], fg, prefix);
                            const float dalpha = T * fg - (R - prefix) * __builtin_amdgcn_rcpf(1.0f - alpha);
                            d[s] = raw * dalpha;  // the gradient passes through min(0.99, .) unchanged
                            T = test_T;
                        }
                    }
                }
                if (any != 0ull) {
                    f32x4 D = zero4, W = zero4;  // lane (q, b, s): d and w of the row's pixels at step s
#pragma unroll
                    for (int s = 0; s < 4; ++s) {
                        const float one_hot = ones(0x1111111111111111ull << s);
                        D = __builtin_amdgcn_mfma_f32_4x4x1f32(d[s], one_hot, D, 0, 0, 0);
                        W = __builtin_amdgcn_mfma_f32_4x4x1f32(w[s], one_hot, W, 0, 0, 0);
                    }
                    float m = (D[0] + D[1]) + (D[2] + D[3]);  // sum d
                    // A d that is not finite times the zeros of the one-hot row is NaN in the quad's other columns, which
                    // are other Gaussians, and every column's sum shows it: then the values change lanes by themselves.
                    if (__ballot(!(fabsf(m) < __builtin_inff())) != 0ull) {
                        auto from_lane = [&](auto lane) {  // (value by value: all sixteen at once cost a wavefront per SIMD)
                            const float v[4] = {quad_lane<lane.value>(d[0]), quad_lane<lane.value>(d[1]),
                                                quad_lane<lane.value>(d[2]), quad_lane<lane.value>(d[3])};
                            return sub < 2 ? (sub == 0 ? v[0] : v[1]) : (sub == 2 ? v[2] : v[3]);
                        };
                        D[0] = from_lane(std::integral_constant<int, 0>{});
                        D[1] = from_lane(std::integral_constant<int, 1>{});
                        D[2] = from_lane(std::integral_constant<int, 2>{});
                        D[3] = from_lane(std::integral_constant<int, 3>{});
                        m = (D[0] + D[1]) + (D[2] + D[3]);
                    }
                    const uint32_t k = (entries >> (8 * sub)) & 0xFFu;  // the column's entry
                    const float2 at = *reinterpret_cast<const float2*>(&s_a[k]);
                    const float ax = at.x - (pxf - (float)sub), dy = at.y - pyf;  // from the row's first pixel
                    const float ax1 = ax - 1.0f, ax2 = ax - 2.0f, ax3 = ax - 3.0f;
                    const float u0 = D[0] * ax, u1 = D[1] * ax1, u2 = D[2] * ax2, u3 = D[3] * ax3;
                    const float mx = (u0 + u1) + (u2 + u3);                           // sum d dx
                    const float mxx = __builtin_fmaf(u3, ax3, __builtin_fmaf(u2, ax2, __builtin_fmaf(u1, ax1, u0 * ax)));
                    const float my = dy * m, myy = dy * my, mxy = dy * mx;
                    auto against = [&](float g) {  // the row's w against one channel of its pixels' gradients
                        f32x4 G = __builtin_amdgcn_mfma_f32_4x4x1f32(g, 1.0f, zero4, 0, 0, 0);
                        if (!finite_g)  // (a pixel that rejected the Gaussian, w = 0, keeps its gradient to itself)
#pragma unroll
                            for (int i = 0; i < 4; ++i) G[i] = W[i] != 0.0f ? G[i] : 0.0f;
                        return __builtin_fmaf(W[3], G[3], __builtin_fmaf(W[2], G[2], __builtin_fmaf(W[1], G[1], W[0] * G[0])));
                    };
                    const float red = against(g0), green = against(g1), blue = against(g2);
                    // rows 0..3 end with (sum d, d dy, d dx dy, red), (d dx, d dy^2, green, blue), (d dx^2, depth)
                    const float sum_a = add_halves<16>(add_halves<32>(m, mxy), add_halves<32>(my, red));
                    const float sum_b = add_halves<16>(add_halves<32>(mx, green), add_halves<32>(myy, blue));
                    float sum_c = add_halves<16>(mxx, kDepth ? against(g3) : mxx);
                    sum_c = add_halves<32>(sum_c, sum_c);
                    float2* __restrict__ sums = s_sum[wave][k];
                    float* __restrict__ last = reinterpret_cast<float*>(sums + 4) + (row & 1);
#pragma unroll
                    for (int b = 0; b < 4; ++b) {  // (two blocks may hold the same entry)
                        if ((any & (kBlockLanes << (4 * b))) == 0ull) continue;  // (uniform: nothing blended in the block)
                        if (group == b) {  // (rows 2 and 3 hold what rows 0 and 1 do for the last pair: one exchange with LDS, not two)
                            const float2 v = sums[row];
                            const float l = *last;
                            sums[row] = make_float2(v.x + sum_a, v.y + sum_b);
                            *last = l + sum_c;
                        }
                        wave_lds_sync();
                    }
                }
                if (__ballot(T > 0.0f) == 0ull) break;
            }
        }
        __syncthreads();
        // ---- this batch's records: the moments turned into gradients of position and conic ----
        float2 m = make_float2(0.f, 0.f);
        float l = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            float2* __restrict__ sums = s_sum[w][staged];
            const float2 v = sums[part];
            m = make_float2(m.x + v.x, m.y + v.y);
            sums[part] = make_float2(0.f, 0.f);
            if (part < 2) {
                float* __restrict__ last = reinterpret_cast<float*>(sums + 4) + part;
                l += *last;
                *last = 0.f;
            }
        }
        const float M = quad_lane<0>(m.x), my = quad_lane<1>(m.x), mxy = quad_lane<2>(m.x), red = quad_lane<3>(m.x);
        const float green = quad_lane<2>(m.y), blue = quad_lane<3>(m.y), depth = quad_lane<1>(l);
        if (staged < count && part < 3) {
            const float hx = s_a[staged].z, ny = s_a[staged].w, hz = s_b[staged].x;
            RecordPart<kPartFloats<kDepth>> v;
            // d power / d centre = -(conic_x dx + conic_y dy, conic_z dy + conic_y dx), with conic_x = -2 hx etc.
            // M = sum of opacity * dL/dopacity over the tile's pixels (zero, not 0 * inf, for a Gaussian that never
            // blended)
            if (part == 0) {
                v.v[0] = 2.0f * hx * m.y + ny * my;
                v.v[1] = 2.0f * hz * my + ny * m.y;
                v.v[2] = -0.5f * l;
                if (kDepth) v.v[3] = -mxy;
            } else if (part == 1) {
                const float d_opacity = M != 0.0f ? M * __builtin_amdgcn_exp2f(-s_b[staged].y) : 0.0f;
                v.v[0] = kDepth ? -0.5f * m.y : -mxy;
                v.v[1] = kDepth ? d_opacity : -0.5f * m.y;
                v.v[2] = kDepth ? red : d_opacity;
                if (kDepth) v.v[3] = green;
            } else {
                v.v[0] = kDepth ? blue : red;
                v.v[1] = kDepth ? depth : green;
                v.v[2] = kDepth ? 0.0f : blue;
                if (kDepth) v.v[3] = 0.0f;
            }
            v.store(key_grads + ((size_t)s_slot[staged] * 3 + part) * kPartFloats<kDepth>);
        }
    }
    // keys the tile never reached (every pixel finished before them) contribute nothing: every record is written
    for (uint32_t j = base + tid; j < hi; j += 256) {
        const RecordSlots at = slots[values[j]];
        const uint32_t slot = at.base + (uint32_t)tile_y * at.width + (uint32_t)tile_x;
        float* __restrict__ dst = key_grads + (size_t)slot * 3 * kPartFloats<kDepth>;
#pragma unroll
        for (int k = 0; k < 3 * kPartFloats<kDepth>; ++k) dst[k] = 0.0f;
    }
}

// The preprocess's backward pass reads its inputs once and writes gradients that nothing reads before the pass has ended.  In large
// scenes streaming accesses (kStreamed) leave the L2 to the records, which lanes pick out of lines a part at a time (streamed as
// well, they take the kernel to 1059 us).  6M Gaussians from stored parameters: stores 706 -> 674 us, the coefficients' copies 668,
// the other inputs 660; and the next frame's preprocess, which finds more of its lines unwritten, 326 -> 312.
// Smaller scenes' parameters and gradients are in the caches when the optimizer reads both next: Adam's step alone, behind a pass
// with ordinary and with streaming accesses, 30k Gaussians of sixteen coefficients 98 and 104 us, 100k of nine 87 and 108, of one
// 84 and 104.  Pass and step: 100k of nine 457 to 468 and 475 to 483 us, 150k of sixteen 482 and 473, 270k 629 and 631, 400k 760
// and 750, 1M 1191 and 1146.
constexpr int kStreamedFrom = 1 << 17;
template <bool kStreamed>
__device__ __forceinline__ void put(float4* p, const float4 v)
{
    const f32x4 x = {v.x, v.y, v.z, v.w};
    if (kStreamed) __builtin_nontemporal_store(x, reinterpret_cast<f32x4*>(p));
    else *p = v;
}
template <bool kStreamed>
__device__ __forceinline__ void put(float* p, float v)
{
    if (kStreamed) __builtin_nontemporal_store(v, p);
    else *p = v;
}
template <bool kStreamed>
__device__ __forceinline__ float get(const float* p)
{
    return kStreamed ? __builtin_nontemporal_load(p) : *p;
}
constexpr float kShC0 = 0.28209479177387814f;
constexpr float kShC1 = 0.4886025119029199f;
constexpr float kShC2[5] = {1.0925484305920792f, -1.0925484305920792f, 0.31539156525252005f, -1.0925484305920792f,
                            0.5462742152960396f};
constexpr float kShC3[7] = {-0.5900435899266435f, 2.890611442640554f, -0.4570457994644658f, 0.3731763325901154f,
                            -0.4570457994644658f, 1.445305721320277f, -0.5900435899266435f};

// Real SH basis (sh_utils.py:67-94) and its gradient with respect to the unit direction.
__device__ __forceinline__ void sh_basis_grad(int deg, float x, float y, float z, float b[16], float bx[16],
                                              float by[16], float bz[16])
{
#pragma unroll
    for (int k = 0; k < 16; ++k) b[k] = bx[k] = by[k] = bz[k] = 0.0f;
    b[0] = kShC0;
    if (deg < 1) return;
    b[1] = -kShC1 * y; by[1] = -kShC1;
    b[2] = kShC1 * z;  bz[2] = kShC1;
    b[3] = -kShC1 * x; bx[3] = -kShC1;
    if (deg < 2) return;
    const float xx = x * x, yy = y * y, zz = z * z, xy = x * y, yz = y * z, xz = x * z;
    b[4] = kShC2[0] * xy; bx[4] = kShC2[0] * y; by[4] = kShC2[0] * x;
    b[5] = kShC2[1] * yz; by[5] = kShC2[1] * z; bz[5] = kShC2[1] * y;
    b[6] = kShC2[2] * (2.0f * zz - xx - yy); bx[6] = kShC2[2] * -2.0f * x; by[6] = kShC2[2] * -2.0f * y;
    bz[6] = kShC2[2] * 4.0f * z;
    b[7] = kShC2[3] * xz; bx[7] = kShC2[3] * z; bz[7] = kShC2[3] * x;
    b[8] = kShC2[4] * (xx - yy); bx[8] = kShC2[4] * 2.0f * x; by[8] = kShC2[4] * -2.0f * y;
    if (deg < 3) return;
    b[9] = kShC3[0] * y * (3.0f * xx - yy); bx[9] = kShC3[0] * 6.0f * xy; by[9] = kShC3[0] * (3.0f * xx - 3.0f * yy);
    b[10] = kShC3[1] * xy * z; bx[10] = kShC3[1] * yz; by[10] = kShC3[1] * xz; bz[10] = kShC3[1] * xy;
    b[11] = kShC3[2] * y * (4.0f * zz - xx - yy); bx[11] = kShC3[2] * -2.0f * xy;
    by[11] = kShC3[2] * (4.0f * zz - xx - 3.0f * yy); bz[11] = kShC3[2] * 8.0f * yz;
    b[12] = kShC3[3] * z * (2.0f * zz - 3.0f * xx - 3.0f * yy); bx[12] = kShC3[3] * -6.0f * xz;
    by[12] = kShC3[3] * -6.0f * yz; bz[12] = kShC3[3] * (6.0f * zz - 3.0f * xx - 3.0f * yy);
    b[13] = kShC3[4] * x * (4.0f * zz - xx - yy); bx[13] = kShC3[4] * (4.0f * zz - 3.0f * xx - yy);
    by[13] = kShC3[4] * -2.0f * xy; bz[13] = kShC3[4] * 8.0f * xz;
    b[14] = kShC3[5] * z * (xx - yy); bx[14] = kShC3[5] * 2.0f * xz; by[14] = kShC3[5] * -2.0f * yz;
    bz[14] = kShC3[5] * (xx - yy);
    b[15] = kShC3[6] * x * (xx - 3.0f * yy); bx[15] = kShC3[6] * (3.0f * xx - 3.0f * yy); by[15] = kShC3[6] * -6.0f * xy;
}

constexpr int kShStride = 52;  // floats per Gaussian in the SH staging area (16-B reads of 64 lanes on distinct banks)

// A Gaussian's keys are consecutive records; they are added in a fixed order, so the result does not vary between runs.
// Up to kSerialRecords of them are added by the Gaussian's own lane, four requested at a time (indices past the last
// one re-read it and are not added).  A Gaussian of more keys would keep its whole wavefront waiting for one lane's
// chain of requests (a splat of an early training step covers hundreds of tiles: 245 us of kernel for 100k Gaussians,
// 112 with this), so those are served by all lanes, four Gaussians at a time: sixteen lanes take one, three per
// record, five records side by side and four such rounds in flight, and the partial sums meet in LDS.
constexpr uint32_t kSerialRecords = 8;
// Scenes of few Gaussians leave most of the chip idle even so (a wavefront per 64 Gaussians): up to this many, a kernel
// of its own gives every Gaussian of more than kSerialRecords keys a wavefront and leaves the sum in its first slot
// (100k Gaussians: 112 -> 67 us for both kernels).  Beyond, the launch of a wavefront per Gaussian costs more.
constexpr int kSumAheadMax = 1 << 18;
constexpr int kPartials = 4 * 15;  // float4 of LDS per wavefront

// (spans: how many of the tile numbers are keys is not known without evaluating them, and there are more than a few)
__device__ __forceinline__ bool summed_ahead(const RecordRun& run) { return run.spans || run.keys() > kSerialRecords; }

__device__ __forceinline__ TileSpans spans_of(const TileRegion& q, const float* __restrict__ splats, size_t i)
{
    TileSpans s;
    if (q.spans) s = TileSpans(splats + i * kRecordFloats, q.x0, q.y0);
    return s;
}

template <int N>
__device__ __forceinline__ void sum_records(const float* __restrict__ key_grads, const RecordRun run, uint64_t region, bool plain,
                                            const float* __restrict__ splats, size_t index, float4* __restrict__ partial,
                                            RecordPart<N> A[3])
{
    typedef RecordPart<N> Part;
    const int lane = threadIdx.x & 63, group = lane >> 4, sub = lane & 15;
#pragma unroll
    for (int q = 0; q < 3; ++q) A[q] = Part{};
    const uint32_t n = run.n;
    const bool serial = !summed_ahead(run);
    if (serial) {
        const float* __restrict__ rec = key_grads + (size_t)run.first * (3 * N);
        const uint32_t keys = run.keys();
        uint32_t left = run.masked ? run.mask : (1u << n) - 1u, last = 0;
        for (uint32_t k0 = 0; k0 < keys; k0 += 4) {
            Part r[4][3];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                last = left != 0u ? (uint32_t)__builtin_ctz(left) : last;
                left &= left - 1u;  // (0 stays 0)
#pragma unroll
                for (int q = 0; q < 3; ++q) r[u][q] = Part::load(rec + (3u * last + (uint32_t)q) * N);
            }
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                if (k0 + (uint32_t)u < keys) {
#pragma unroll
                    for (int q = 0; q < 3; ++q) A[q].add(r[u][q]);
                }
            }
        }
    }
    uint64_t left = __ballot(!serial);
    const int slot = sub / 3, part = sub % 3;  // (lane 15 of a group has no part)
    while (left != 0ull) {
        int lane_of[4], mine = -1;  // the lanes whose Gaussians the four groups take
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            lane_of[g] = left != 0ull ? (int)__ffsll((unsigned long long)left) - 1 : -1;
            left &= left - 1ull;  // (0 stays 0)
            mine = group == g ? lane_of[g] : mine;
        }
        const uint32_t n_of = (uint32_t)__shfl((int)n, max(mine, 0), 64);
        const uint32_t first_of = (uint32_t)__shfl((int)run.first, max(mine, 0), 64);
        const uint32_t n_mine = mine < 0 || sub == 15 ? 0u : n_of;
        const uint64_t region_of = (uint64_t)__shfl((long long)region, max(mine, 0), 64);
        const TileRegion q(region_of, plain);
        const TileSpans spans = spans_of(q, splats, (size_t)__shfl((long long)index, max(mine, 0), 64));
        auto held = [&](uint32_t k) {
            if (k >= n_mine) return false;
            int row, col;
            q.place((int)k, row, col);
            return q.holds((int)k, row, col, spans);
        };
        const float* __restrict__ rec = key_grads + ((size_t)first_of * 3 + part) * N;
        Part sum = {};
        for (uint32_t k0 = (uint32_t)slot; k0 < n_mine; k0 += 20) {
            Part r[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) r[u] = Part::load(rec + 3 * N * (size_t)min(k0 + 5u * (uint32_t)u, n_mine - 1));
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (held(k0 + 5u * (uint32_t)u)) sum.add(r[u]);
        }
        if (sub < 15) sum.store(reinterpret_cast<float*>(partial + 15 * group + sub));
        wave_lds_sync();
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            if (lane != lane_of[g]) continue;
#pragma unroll
            for (int k = 0; k < 5; ++k)
#pragma unroll
                for (int p = 0; p < 3; ++p) A[p].add(Part::load(reinterpret_cast<const float*>(partial + 15 * g + 3 * k + p)));
        }
        wave_lds_sync();
    }
}

// A wavefront takes eight Gaussians, a step 64 tile numbers of one: a lane each finds those that the region holds, and the
// held records are read sixteen side by side, three lanes each, up to four such rounds.  The next step, of the same Gaussian
// or the next, is requested before the current one is added.  The first record is overwritten once all of them have been
// read (its new value depends on every one).
// What bounds it is the instructions per tile number: with the three lanes of a record each asking for its tile number, a
// record that the region leaves out took its turn like the others, and 100k Gaussians of some 20 records each took 39 us; with
// one question per tile number and only held records in the rounds, 26.
constexpr int kSumPerWave = 8;
template <int N>
__global__ __launch_bounds__(256) void sum_large_kernel(int P, bool plain, const int32_t* __restrict__ radii,
                                                        const float* __restrict__ splats,
                                                        const uint64_t* __restrict__ rects,
                                                        const RecordSlots* __restrict__ slots, float* key_grads)
{
    __shared__ uint8_t s_held[4][2][64];  // tile numbers (from the step's first) of a step's records, this step's and the next's
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i0 = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * 4 + wave) * kSumPerWave);
    const int i = min(i0 + (lane & (kSumPerWave - 1)), P - 1);
    const int32_t radius = radii[i];
    const uint64_t region = rects[i];
    const TileRegion own(region, plain);
    const RecordRun run = record_run(slots[i], own);
    uint32_t left = (uint32_t)__ballot(lane < kSumPerWave && i0 + lane < P && radius > 0 && summed_ahead(run));
    if (left == 0u) return;
    const TileSpans own_spans = spans_of(own, splats, (size_t)i);
    const int slot = lane / 3, part = lane % 3;
    typedef RecordPart<N> Part;
    float* const all = key_grads + part * N;
    // the Gaussian whose records are requested next: slots first .. first + n - 1, and the step's first tile number
    uint32_t first = 0, n = 0, e0 = 0;
    TileRegion q(0ull, plain);
    TileSpans spans;
    auto next = [&]() {
        const int l = __builtin_ctz(left);
        left &= left - 1u;
        first = (uint32_t)__builtin_amdgcn_readlane((int)run.first, l);
        n = (uint32_t)__builtin_amdgcn_readlane((int)run.n, l);
        e0 = 0;
        q = TileRegion((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)region, l) |
                           ((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(region >> 32), l) << 32),
                       plain);  // (uniform, and so are its spans)
        auto of_lane = [&](float v) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); };
        spans.rho = of_lane(own_spans.rho), spans.across = of_lane(own_spans.across), spans.slack = of_lane(own_spans.slack);
        spans.rx = of_lane(own_spans.rx), spans.x = of_lane(own_spans.x), spans.y = of_lane(own_spans.y);
        spans.inv_y = of_lane(own_spans.inv_y);
    };
    // (the loads stand behind no branch, so that the compiler knows how many are under way; what they read past the last
    // record is not added)
    auto request = [&](uint8_t* held, Part r[4]) {
        const uint32_t e = e0 + (uint32_t)lane;
        bool holds = e < n;
        if (holds) {
            int row, col;
            q.place((int)e, row, col);
            holds = q.holds((int)e, row, col, spans);
        }
        const uint64_t m = __ballot(holds);
        if (holds) held[lanes_below_in(m)] = (uint8_t)lane;
        wave_lds_sync();
        const int count = __popcll(m);
        const uint8_t* const mine = held + min(slot, 15);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const uint32_t at = slot + 16 * u < count ? mine[16 * u] : 0u;
            r[u] = Part::load(all + ((size_t)first + e0 + at) * (3 * N));
        }
        return count;
    };
    next();
    Part r[4], sum = {};
    int count = request(s_held[wave][0], r);
    for (int buffer = 1;; buffer ^= 1) {  // (uniform; ends with the last Gaussian's last step)
        const uint32_t first0 = first;
        const bool last = e0 + 64u >= n;
        const bool more = !last || left != 0u;
        if (!last) e0 += 64u;
        else if (more) next();
        Part r1[4];
        const int count1 = request(s_held[wave][buffer], r1);  // (behind the last step: once more, and not used)
#pragma unroll
        for (int u = 0; u < 4; ++u)
            if (slot < 16 && slot + 16 * u < count) sum.add(r[u]);
        if (last) {
#pragma unroll
            for (int d = 24; d >= 3; d >>= 1) {
                Part other;
#pragma unroll
                for (int k = 0; k < N; ++k) other.v[k] = __shfl_down(sum.v[k], d, 64);
                sum.add(other);  // (lanes past the last slot hold zeros; sums other than the first slot's are not used)
            }
            // (into the slot of the region's first record; a mask's first tile may be past number 0)
            if (slot == 0) sum.store(all + (size_t)first0 * (3 * N));
            sum = Part{};
        }
        if (!more) break;
        count = count1;
#pragma unroll
        for (int u = 0; u < 4; ++u) r[u] = r1[u];
    }
}

// kMode 0: SH blocks (if any) are read and written by their own lanes.  1 and 2: 16-coefficient blocks, 16-byte
// aligned, staged through LDS; 2 also fetches the coefficients (needed for degree > 0 only).  kStored: g holds the
// vanilla model's stored parameters, and the gradients are theirs (activations' derivatives included); the rows of the
// SH coefficients behind the first are then staged back to back, 3 (M - 1) floats each, as they lie in memory: a
// wavefront's 64 rows start on a 256-B boundary whatever their length.
template <int kMode, bool kStored, bool kDepth, bool kStreamed>
__global__ __launch_bounds__(256, kStored ? 3 : 1) void preprocess_backward_kernel(FrameArgs f, gs355_gaussians g,
                                                                  const int32_t* __restrict__ radii,
                                                                  const float* __restrict__ records,
                                                                  const uint64_t* __restrict__ rects,
                                                                  const RecordSlots* __restrict__ slots,
                                                                  const uint8_t* __restrict__ lit,
                                                                  const float* __restrict__ key_grads,
                                                                  gs355_gradients out, ParameterArgs par, bool summed)
{
    // Full 16-coefficient SH blocks travel through LDS: each wavefront moves the 12 KB of its 64 Gaussians'
    // coefficients (in) and coefficient gradients (out) with coalesced 16-B accesses; a lane works on its own row.
    // (kStored: rows of at most 45 floats back to back, filled by whole-wavefront copies of 1 KB, twelve at most)
    constexpr int kWaveRows = kMode == 0 ? 0 : kStored ? 12 * 64 : 64 * kShStride / 4;  // float4 per wavefront
    // the partial record sums have their place behind the rows where those may be in flight, else inside them
    constexpr int kPartialsAt = kStored ? kWaveRows : 0;
    constexpr int kWaveLds = kPartialsAt + kPartials > kWaveRows ? kPartialsAt + kPartials : kWaveRows;
    __shared__ float4 s_sh[4 * kWaveLds];

    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool valid = i < g.P;
    const size_t si = (size_t)(valid ? i : g.P - 1);
    const int M = f.sh_coeffs;
    const bool alive = valid && radii[si] > 0;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const size_t wave_first = (size_t)blockIdx.x * blockDim.x + (size_t)wave * 64;
    const int count = (int)min((size_t)64, (size_t)g.P > wave_first ? (size_t)g.P - wave_first : (size_t)0);
    constexpr bool staged = kMode != 0, fetch_sh = kMode == 2;
    const int rest_row = 3 * (M - 1);  // floats per Gaussian in par.rest
    float4* __restrict__ mine = s_sh + wave * kWaveLds;
    float* __restrict__ my_row = reinterpret_cast<float*>(mine) + (staged ? lane * (kStored ? rest_row : kShStride) : 0);

    float dmean[3] = {0.f, 0.f, 0.f}, d2[3] = {0.f, 0.f, 0.f}, dscale[3] = {0.f, 0.f, 0.f};
    float drot[4] = {0.f, 0.f, 0.f, 0.f}, dcov[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, dcol[3] = {0.f, 0.f, 0.f};
    float dop = 0.f;
    float gcol[3] = {0.f, 0.f, 0.f};
    float nx = 0.f, ny = 0.f, nz = 0.f, inv_len = 0.f;
    int K = 0;
    const uint64_t region = alive ? rects[si] : 0ull;
    RecordRun run = record_run(slots[si], TileRegion(region, f.plain_regions));
    if (summed && summed_ahead(run)) run = {run.first, 1u, 0u, false, false};  // (sum_large_kernel has added them into the first)
    // kStored: the wavefront's rows as one run of float4, and the up to three floats behind the last whole one.  They
    // travel from memory to LDS without passing through registers, requested before anything else is waited for: held
    // in registers the 48 of them left two wavefronts per SIMD, requested later their latency came on top of the
    // records' (6M Gaussians: 1.10 -> 0.76 ms, 3.5 GB at the rate of a large copy).
    const int run4 = kStored ? count * rest_row / 4 : 0, run_tail = kStored ? count * rest_row % 4 : 0;
    const size_t run_first = wave_first * (size_t)rest_row;
    float tail = 0.f;
    if (fetch_sh && kStored) {
        typedef __attribute__((address_space(1))) const void global_void;
        typedef __attribute__((address_space(3))) void lds_void;
        constexpr int kPolicy = kStreamed ? 2 : 0;  // (of the copies: nontemporal, or as ordinary loads)
        const float4* src = reinterpret_cast<const float4*>(par.rest + run_first);
#pragma unroll
        for (int it = 0; it < 12; ++it)
            if (it * 64 + lane < run4)  // (lane l of a copy writes float4 l behind the uniform LDS address)
                __builtin_amdgcn_global_load_lds((global_void*)(src + it * 64 + lane), (lds_void*)(mine + it * 64), 16, 0, kPolicy);
        if (lane < run_tail) tail = par.rest[run_first + 4 * run4 + lane];
    }
    // the Gaussian's own inputs are requested before its records are waited for, too
    float in_mean[3] = {0.f, 0.f, 0.f}, in_scale[3] = {0.f, 0.f, 0.f}, in_rot[4] = {0.f, 0.f, 0.f, 0.f};
    float in_opacity = 0.f;
    uint32_t in_lit = 0u;
    if (alive) {
#pragma unroll
        for (int k = 0; k < 3; ++k) in_mean[k] = get<kStreamed>(&g.means3D[3 * si + k]);
        if (kStored || !g.cov3D_precomp) {
#pragma unroll
            for (int k = 0; k < 3; ++k) in_scale[k] = get<kStreamed>(&g.scales[3 * si + k]);
#pragma unroll
            for (int k = 0; k < 4; ++k) in_rot[k] = get<kStreamed>(&g.rotations[4 * si + k]);
        }
        if (kStored) in_opacity = get<kStreamed>(&g.opacities[si]);
        if (g.shs) in_lit = lit[si];
    }
    constexpr int N = kPartFloats<kDepth>;
    RecordPart<N> A[3];
    sum_records<N>(key_grads, run, region, f.plain_regions, records, si, mine + kPartialsAt, A);
    if (alive) {
        const float* __restrict__ V = f.viewmatrix;
        const float* __restrict__ Pm = f.projmatrix;
        const float g_px = A[0].v[0], g_py = A[0].v[1], gA = A[0].v[2];
        const float gB = kDepth ? A[0].v[N - 1] : A[1].v[0], gC = kDepth ? A[1].v[0] : A[1].v[1];
        dop = kDepth ? A[1].v[1] : A[1].v[2];
        dcol[0] = kDepth ? A[1].v[2] : A[2].v[0];
        dcol[1] = kDepth ? A[1].v[N - 1] : A[2].v[1];
        dcol[2] = kDepth ? A[2].v[0] : A[2].v[2];
        const float g_depth = kDepth ? A[2].v[1] : 0.0f;
        const float x = in_mean[0], y = in_mean[1], z = in_mean[2];

        // ---- pixel position ----
        const float phx = Pm[0] * x + Pm[4] * y + Pm[8] * z + Pm[12];
        const float phy = Pm[1] * x + Pm[5] * y + Pm[9] * z + Pm[13];
        const float phw = Pm[3] * x + Pm[7] * y + Pm[11] * z + Pm[15];
        const float pw = 1.0f / (phw + 0.0000001f);
        d2[0] = g_px * 0.5f * (float)f.W;
        d2[1] = g_py * 0.5f * (float)f.H;
        const float d_phx = d2[0] * pw, d_phy = d2[1] * pw;
        const float d_phw = -(pw * pw) * (phx * d2[0] + phy * d2[1]);
#pragma unroll
        for (int k = 0; k < 3; ++k) dmean[k] = Pm[4 * k] * d_phx + Pm[4 * k + 1] * d_phy + Pm[4 * k + 3] * d_phw;

        // ---- 3-D covariance, Jacobian of the projection, 2-D covariance, conic: in double precision ----
        // An elongated splat (axes 50:1) hides its thin axes in the low bits of the fp32 covariance, and its 2-D
        // determinant is a difference of nearly equal products; the gradients of scale and rotation are small
        // differences of terms built from them.  fp64 vector arithmetic runs at the fp32 rate on this chip and
        // the kernel waits for memory, so the chain costs nothing in double and loses nothing.
        typedef double real;
        real S[6], s[3] = {0., 0., 0.}, q[4] = {0., 0., 0., 0.}, R[3][3] = {};
        float norm = 1.f;
        if (!kStored && g.cov3D_precomp) {
#pragma unroll
            for (int k = 0; k < 6; ++k) S[k] = g.cov3D_precomp[6 * si + k];
        } else {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                const float v = in_scale[k];
                s[k] = (real)f.scale_modifier * (real)(kStored ? expf(v) : v);
            }
            if (kStored) norm = quaternion_norm(in_rot);
#pragma unroll
            for (int k = 0; k < 4; ++k) q[k] = kStored ? in_rot[k] / norm : in_rot[k];
            const real r = q[0], qx = q[1], qy = q[2], qz = q[3];
            R[0][0] = 1. - 2. * (qy * qy + qz * qz); R[0][1] = 2. * (qx * qy - r * qz); R[0][2] = 2. * (qx * qz + r * qy);
            R[1][0] = 2. * (qx * qy + r * qz); R[1][1] = 1. - 2. * (qx * qx + qz * qz); R[1][2] = 2. * (qy * qz - r * qx);
            R[2][0] = 2. * (qx * qz - r * qy); R[2][1] = 2. * (qy * qz + r * qx); R[2][2] = 1. - 2. * (qx * qx + qy * qy);
            int n = 0;
#pragma unroll
            for (int a = 0; a < 3; ++a)
#pragma unroll
                for (int c = a; c < 3; ++c)
                    S[n++] = R[a][0] * s[0] * R[c][0] * s[0] + R[a][1] * s[1] * R[c][1] * s[1] + R[a][2] * s[2] * R[c][2] * s[2];
        }
        const real Sm[3][3] = {{S[0], S[1], S[2]}, {S[1], S[3], S[4]}, {S[2], S[4], S[5]}};

        real Vd[12];  // the three columns of the view matrix the chain uses, rows 0..2
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            Vd[3 * k] = V[4 * k];
            Vd[3 * k + 1] = V[4 * k + 1];
            Vd[3 * k + 2] = V[4 * k + 2];
        }
        const real xd = x, yd = y, zd = z;
        const real pvx = Vd[0] * xd + Vd[3] * yd + Vd[6] * zd + (real)V[12];
        const real pvy = Vd[1] * xd + Vd[4] * yd + Vd[7] * zd + (real)V[13];
        const real tz = Vd[2] * xd + Vd[5] * yd + Vd[8] * zd + (real)V[14];
        const real fx = (real)f.W / (2. * (real)f.tanfovx), fy = (real)f.H / (2. * (real)f.tanfovy);
        const real limx = 1.3 * (real)f.tanfovx, limy = 1.3 * (real)f.tanfovy;
        const real itz = 1. / tz, itz2 = itz * itz;
        const real rx = pvx * itz, ry = pvy * itz;
        const real cx = rx > limx ? limx : rx < -limx ? -limx : 0.;  // non-zero: clamped to +-lim
        const real cy = ry > limy ? limy : ry < -limy ? -limy : 0.;
        const real tx = cx != 0. ? cx * tz : pvx, ty = cy != 0. ? cy * tz : pvy;
        const real J00 = fx * itz, J02 = -(fx * tx) * itz2;
        const real J11 = fy * itz, J12 = -(fy * ty) * itz2;
        real a0[3], a1[3], Sa0[3], Sa1[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            a0[k] = J00 * Vd[3 * k] + J02 * Vd[3 * k + 2];
            a1[k] = J11 * Vd[3 * k + 1] + J12 * Vd[3 * k + 2];
        }
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            Sa0[k] = Sm[k][0] * a0[0] + Sm[k][1] * a0[1] + Sm[k][2] * a0[2];
            Sa1[k] = Sm[k][0] * a1[0] + Sm[k][1] * a1[1] + Sm[k][2] * a1[2];
        }
        const real ca = a0[0] * Sa0[0] + a0[1] * Sa0[1] + a0[2] * Sa0[2] + 0.3;
        const real cb = a0[0] * Sa1[0] + a0[1] * Sa1[1] + a0[2] * Sa1[2];
        const real cc = a1[0] * Sa1[0] + a1[1] * Sa1[1] + a1[2] * Sa1[2] + 0.3;
        const real D = 1. / (ca * cc - cb * cb), D2 = D * D;
        // conic = (cc, -cb, ca) / det; with det - ca cc = -cb^2 the derivatives need no difference of near-equal terms
        const real gAd = gA, gBd = gB, gCd = gC;
        const real d_ca = D2 * (-cc * cc * gAd + cb * cc * gBd - cb * cb * gCd);
        const real d_cb = D2 * (2. * cb * cc * gAd - (ca * cc + cb * cb) * gBd + 2. * ca * cb * gCd);
        const real d_cc = D2 * (-cb * cb * gAd + ca * cb * gBd - ca * ca * gCd);
        // symmetric gradient of the 3-D covariance, packed with the off-diagonal entries counted once each
        real dS[3][3];
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
            for (int l = 0; l < 3; ++l)
                dS[k][l] = d_ca * a0[k] * a0[l] + d_cb * 0.5 * (a0[k] * a1[l] + a1[k] * a0[l]) + d_cc * a1[k] * a1[l];
        real d_J00 = 0., d_J02 = 0., d_J11 = 0., d_J12 = 0.;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const real d_a0 = 2. * d_ca * Sa0[k] + d_cb * Sa1[k];
            const real d_a1 = 2. * d_cc * Sa1[k] + d_cb * Sa0[k];
            d_J00 += d_a0 * Vd[3 * k];
            d_J02 += d_a0 * Vd[3 * k + 2];
            d_J11 += d_a1 * Vd[3 * k + 1];
            d_J12 += d_a1 * Vd[3 * k + 2];
        }
        const real itz3 = itz2 * itz;
        const real d_tx = d_J02 * (-fx * itz2), d_ty = d_J12 * (-fy * itz2);
        const real d_tz = d_J00 * (-fx * itz2) + d_J11 * (-fy * itz2) + d_J02 * (2. * fx * tx * itz3) +
                          d_J12 * (2. * fy * ty * itz3);
        const real d_pvx = cx != 0. ? 0. : d_tx, d_pvy = cy != 0. ? 0. : d_ty;
        const real d_pvz = d_tz + cx * d_tx + cy * d_ty + (real)g_depth;
#pragma unroll
        for (int k = 0; k < 3; ++k)
            dmean[k] += (float)(Vd[3 * k] * d_pvx + Vd[3 * k + 1] * d_pvy + Vd[3 * k + 2] * d_pvz);

        if (!kStored && g.cov3D_precomp) {
            dcov[0] = (float)dS[0][0]; dcov[1] = (float)(2. * dS[0][1]); dcov[2] = (float)(2. * dS[0][2]);
            dcov[3] = (float)dS[1][1]; dcov[4] = (float)(2. * dS[1][2]); dcov[5] = (float)dS[2][2];
        } else {
            // Sigma = L L^T with L = R diag(s): dL = 2 dS L
            real dR[3][3];
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                real ds = 0.;
#pragma unroll
                for (int a = 0; a < 3; ++a) {
                    const real dL = 2. * (dS[a][0] * R[0][k] + dS[a][1] * R[1][k] + dS[a][2] * R[2][k]) * s[k];
                    ds += dL * R[a][k];
                    dR[a][k] = dL * s[k];
                }
                dscale[k] = (float)(ds * (kStored ? s[k] : (real)f.scale_modifier));  // (d s / d log s = s)
            }
            const real r = q[0], qx = q[1], qy = q[2], qz = q[3];
            drot[0] = (float)(2. * (-qz * dR[0][1] + qy * dR[0][2] + qz * dR[1][0] - qx * dR[1][2] - qy * dR[2][0] + qx * dR[2][1]));
            drot[1] = (float)(2. * (qy * dR[0][1] + qz * dR[0][2] + qy * dR[1][0] - 2. * qx * dR[1][1] - r * dR[1][2] +
                                    qz * dR[2][0] + r * dR[2][1] - 2. * qx * dR[2][2]));
            drot[2] = (float)(2. * (-2. * qy * dR[0][0] + qx * dR[0][1] + r * dR[0][2] + qx * dR[1][0] + qz * dR[1][2] -
                                    r * dR[2][0] + qz * dR[2][1] - 2. * qy * dR[2][2]));
            drot[3] = (float)(2. * (-2. * qz * dR[0][0] - r * dR[0][1] + qx * dR[0][2] + r * dR[1][0] - 2. * qz * dR[1][1] +
                                    qy * dR[1][2] + qx * dR[2][0] + qy * dR[2][1]));
            if (kStored) {  // through q / max(|q|, 1e-12): the part along q drops out, unless the norm is the constant
                const float along = norm > 1e-12f ? (float)(drot[0] * r + drot[1] * qx + drot[2] * qy + drot[3] * qz) : 0.f;
                drot[0] = (drot[0] - (float)r * along) / norm;
                drot[1] = (drot[1] - (float)qx * along) / norm;
                drot[2] = (drot[2] - (float)qy * along) / norm;
                drot[3] = (drot[3] - (float)qz * along) / norm;
            }
        }
        if (kStored) {
            const float o = logistic(in_opacity);
            dop = dop * ((1.0f - o) * o);
        }

        // ---- colour: view direction, SH basis and its gradient ----
        if (g.shs) {
            const float dirx = x - f.campos[0], diry = y - f.campos[1], dirz = z - f.campos[2];
            inv_len = 1.0f / sqrtf(dirx * dirx + diry * diry + dirz * dirz);
            nx = dirx * inv_len;
            ny = diry * inv_len;
            nz = dirz * inv_len;
            K = (f.sh_degree + 1) * (f.sh_degree + 1);
            // the forward pass clamped the colour at zero: a channel at zero gets no gradient
#pragma unroll
            for (int c = 0; c < 3; ++c) gcol[c] = ((in_lit >> c) & 1u) != 0u ? dcol[c] : 0.0f;
        }
    }

    // ---- SH coefficients: their part of the mean's gradient (through the view direction), and their own ----
    if (g.shs) {
        if (fetch_sh && kStored) {
            if (lane < run_tail) reinterpret_cast<float*>(mine)[4 * run4 + lane] = tail;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the copies have landed
            wave_lds_sync();
        } else if (fetch_sh) {
            // coefficients of the wavefront's Gaussians: all loads in flight together, then into the rows (slots
            // past the last Gaussian re-read it)
            float4 sh_in[12];
#pragma unroll
            for (int it = 0; it < 12; ++it) {
                const int q4 = it * 64 + lane;
                const size_t e = min(wave_first + (size_t)(q4 / 12), (size_t)g.P - 1);
                sh_in[it] = reinterpret_cast<const float4*>(g.shs + e * 48)[q4 % 12];
            }
#pragma unroll
            for (int it = 0; it < 12; ++it) {
                const int q4 = it * 64 + lane;
                mine[(q4 / 12) * (kShStride / 4) + q4 % 12] = sh_in[it];
            }
            wave_lds_sync();
        }
        // (the basis is evaluated after the coefficients have arrived: its 64 values held across the wait would cost a
        // wavefront per SIMD)
        float b[16], bx[16], by[16], bz[16];
        sh_basis_grad(f.sh_degree, nx, ny, nz, b, bx, by, bz);
        if (alive && f.sh_degree > 0) {
            constexpr int kSkip = kStored ? 3 : 0;  // (the first coefficient is stored apart)
            const float* __restrict__ sh = staged ? my_row : kStored ? par.rest + si * rest_row : g.shs + si * M * 3;
            float dn[3] = {0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 1; k < 16; ++k) {
                if (k < K) {
                    const float* __restrict__ c = sh + (3 * k - kSkip);
                    const float t = gcol[0] * c[0] + gcol[1] * c[1] + gcol[2] * c[2];
                    dn[0] += t * bx[k];
                    dn[1] += t * by[k];
                    dn[2] += t * bz[k];
                }
            }
            const float dot = nx * dn[0] + ny * dn[1] + nz * dn[2];
            dmean[0] += (dn[0] - nx * dot) * inv_len;
            dmean[1] += (dn[1] - ny * dot) * inv_len;
            dmean[2] += (dn[2] - nz * dot) * inv_len;
        }
        if (kStored) {
            if (out.shs && valid)
#pragma unroll
                for (int c = 0; c < 3; ++c) put<kStreamed>(&out.shs[3 * si + c], alive ? b[0] * gcol[c] : 0.0f);
            if (par.d_rest && staged) {
                wave_lds_sync();  // rows were read above
#pragma unroll
                for (int k = 1; k < 16; ++k) {
                    if (k < M) {
                        const float bk = (alive && k < K) ? b[k] : 0.0f;
#pragma unroll
                        for (int c = 0; c < 3; ++c) my_row[3 * (k - 1) + c] = bk * gcol[c];
                    }
                }
                wave_lds_sync();
                float4* __restrict__ dst = reinterpret_cast<float4*>(par.d_rest + run_first);
#pragma unroll
                for (int it = 0; it < 12; ++it)
                    if (it * 64 + lane < run4) put<kStreamed>(&dst[it * 64 + lane], mine[it * 64 + lane]);
                if (lane < run_tail) par.d_rest[run_first + 4 * run4 + lane] = reinterpret_cast<float*>(mine)[4 * run4 + lane];
            } else if (par.d_rest && valid) {
#pragma unroll
                for (int k = 1; k < 16; ++k) {
                    if (k < M) {
                        const float bk = (alive && k < K) ? b[k] : 0.0f;
#pragma unroll
                        for (int c = 0; c < 3; ++c) par.d_rest[si * rest_row + 3 * (k - 1) + c] = bk * gcol[c];
                    }
                }
            }
        } else if (out.shs) {
            if (staged) {
                wave_lds_sync();  // rows were read above
#pragma unroll
                for (int k = 0; k < 16; ++k) {
                    const float bk = (alive && k < K) ? b[k] : 0.0f;
                    my_row[3 * k] = bk * gcol[0];
                    my_row[3 * k + 1] = bk * gcol[1];
                    my_row[3 * k + 2] = bk * gcol[2];
                }
                wave_lds_sync();
#pragma unroll
                for (int it = 0; it < 12; ++it) {
                    const int q4 = it * 64 + lane;
                    const int e = q4 / 12, m = q4 % 12;
                    if (e < count) put<kStreamed>(reinterpret_cast<float4*>(out.shs + (wave_first + e) * 48) + m, mine[e * (kShStride / 4) + m]);
                }
            } else if (valid) {
                float* __restrict__ o = out.shs + si * M * 3;
#pragma unroll
                for (int k = 0; k < 16; ++k) {
                    if (k < M) {
                        const float bk = (alive && k < K) ? b[k] : 0.0f;
                        o[3 * k] = bk * gcol[0];
                        o[3 * k + 1] = bk * gcol[1];
                        o[3 * k + 2] = bk * gcol[2];
                    }
                }
                for (int k = 48; k < 3 * M; ++k) o[k] = 0.0f;  // coefficient rows beyond degree 3
            }
        }
    }
    if (!valid) return;

    if (out.means3D)
#pragma unroll
        for (int k = 0; k < 3; ++k) put<kStreamed>(&out.means3D[3 * si + k], dmean[k]);
    if (out.means2D)
#pragma unroll
        for (int k = 0; k < 3; ++k) put<kStreamed>(&out.means2D[3 * si + k], d2[k]);
    if (out.opacities) put<kStreamed>(&out.opacities[i], dop);
    if (out.colors_precomp)
#pragma unroll
        for (int k = 0; k < 3; ++k) put<kStreamed>(&out.colors_precomp[3 * si + k], dcol[k]);
    if (out.scales)
#pragma unroll
        for (int k = 0; k < 3; ++k) put<kStreamed>(&out.scales[3 * si + k], dscale[k]);
    if (out.rotations)
#pragma unroll
        for (int k = 0; k < 4; ++k) put<kStreamed>(&out.rotations[4 * si + k], drot[k]);
    if (out.cov3D_precomp)
#pragma unroll
        for (int k = 0; k < 6; ++k) put<kStreamed>(&out.cov3D_precomp[6 * si + k], dcov[k]);
}

}  // namespace

int launch_render_backward(const FrameArgs& f, const gs355_gaussians& g, const gs355_header* header,
                           const uint32_t* ranges, const uint4* order, const uint32_t* values, const float* records,
                           const uint64_t* rects, const uint8_t* lit, const gs355_backward_inputs& in, uint2* record_slots, uint32_t* next_slot,
                           float* key_grads, const gs355_gradients& out, const ParameterArgs* par, hipStream_t s)
{
    if (g.P == 0) return GS355_OK;
    int rc = launch_fill_u32(next_slot, 1, 0u, s);
    if (rc) return rc;
    RecordSlots* slots = reinterpret_cast<RecordSlots*>(record_slots);
    hipLaunchKernelGGL(record_slots_kernel, dim3((g.P + kSlotThreads * kSlotItems - 1) / (kSlotThreads * kSlotItems)),
                       dim3(kSlotThreads), 0, s, g.P, (bool)f.plain_regions, header, rects, next_slot, slots);
    GS355_CHECK_LAUNCH("record slots");
    const int tiles = f.grid_x * f.grid_y;
    auto blend = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(tiles), dim3(256), 0, s, f, header, ranges, order, values, records, in.image, in.depth,
                           in.alpha, in.dL_dimage, in.dL_ddepth, in.dL_dalpha, slots, key_grads);
    };
    if (in.dL_ddepth)
        blend(blend_backward_kernel<true>);
    else
        blend(blend_backward_kernel<false>);
    GS355_CHECK_LAUNCH("blend backward");
    const bool staged = g.shs != nullptr && f.sh_coeffs == 16 && (reinterpret_cast<uintptr_t>(g.shs) & 15u) == 0 &&
                        (out.shs == nullptr || (reinterpret_cast<uintptr_t>(out.shs) & 15u) == 0);
    const dim3 grid((g.P + 255) / 256), block(256);
    const bool summed = g.P <= kSumAheadMax;
    auto finish = [&](auto with_depth) {
        constexpr bool kDepth = with_depth.value;
        if (summed) {
            hipLaunchKernelGGL(sum_large_kernel<kPartFloats<kDepth>>, dim3((g.P + 4 * kSumPerWave - 1) / (4 * kSumPerWave)), dim3(256),
                               0, s, g.P, (bool)f.plain_regions, in.radii, records, rects, slots, key_grads);
            GS355_CHECK_LAUNCH("record sums");
        }
        auto launch = [&](auto kernel, const ParameterArgs& p) {
            hipLaunchKernelGGL(kernel, grid, block, 0, s, f, g, in.radii, records, rects, slots, lit, key_grads, out, p, summed);
        };
        auto pass = [&](auto streamed) {
            constexpr bool kStreamed = streamed.value;
            if (par) {
                if ((reinterpret_cast<uintptr_t>(par->rest) & 15u) != 0 || (reinterpret_cast<uintptr_t>(par->d_rest) & 15u) != 0)
                    launch(preprocess_backward_kernel<0, true, kDepth, kStreamed>, *par);
                else if (f.sh_degree == 0)
                    launch(preprocess_backward_kernel<1, true, kDepth, kStreamed>, *par);
                else
                    launch(preprocess_backward_kernel<2, true, kDepth, kStreamed>, *par);
            } else if (!staged) {
                launch(preprocess_backward_kernel<0, false, kDepth, kStreamed>, ParameterArgs());
            } else if (f.sh_degree == 0) {
                launch(preprocess_backward_kernel<1, false, kDepth, kStreamed>, ParameterArgs());
            } else {
                launch(preprocess_backward_kernel<2, false, kDepth, kStreamed>, ParameterArgs());
            }
        };
        if (g.P >= kStreamedFrom) pass(std::true_type{});
        else pass(std::false_type{});
        GS355_CHECK_LAUNCH("preprocess backward");
        return (int)GS355_OK;
    };
    return in.dL_ddepth ? finish(std::true_type{}) : finish(std::false_type{});
}

}  // namespace gs355
