// Per-tile range identification and front-to-back alpha blending for gfx950:
// the last two stages of the rasterizer behind GaussianRasterizer.forward
// (benchmarks/nerf/origin_gs/gs_model.py:211-220; output consumed as a
// [3,H,W] image at tests/test_inference_framework/test_inference.py:195-197).
//
// Blending: one 256-thread workgroup per 16x16 pixel tile, each of its four
// wavefronts owning an 8x8 pixel quadrant, each group of 16 lanes a 4x4 block
// of it.  The tile's depth-sorted Gaussians are staged through LDS in batches
// of 252 records (48 B each, rescaled while staging so that the per-pixel
// arithmetic needs no constant multiplies); every 4x4 block gets its own list
// of the staged Gaussians that can reach it, and the four lane groups of a
// wavefront walk their lists side by side, four entries per round, so one
// pass of the pixel arithmetic serves four different Gaussians.  A wavefront
// stops as soon as a ballot shows all of its 64 pixels finished, and the
// workgroup stops fetching batches once all four wavefronts have.
#include <type_traits>

#include "gs355_internal.h"

namespace gs355 {

namespace {

__global__ void fill_u32_kernel(uint32_t* __restrict__ p, size_t n, uint32_t v)
{
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ __launch_bounds__(256) void ranges_kernel(const gs355_header* __restrict__ header,
                                                     const uint64_t* __restrict__ keys, uint32_t* __restrict__ ranges,
                                                     uint32_t tiles)
{
    if (header->overflow) return;
    const uint32_t n = header->num_keys;
    const size_t j = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    const uint32_t t = (uint32_t)(keys[j] >> 32);
    if (t >= tiles) return;  // cannot happen for keys made by the duplicate stage
    if (j == 0) {
        ranges[2 * t] = 0;
    } else {
        const uint32_t tp = (uint32_t)(keys[j - 1] >> 32);
        if (tp != t) {
            if (tp < tiles) ranges[2 * tp + 1] = (uint32_t)j;
            ranges[2 * t] = (uint32_t)j;
        }
    }
    if (j == n - 1) ranges[2 * t + 1] = n;
}

// One (pixel, Gaussian) pair: exponent, alpha, the three discrete tests and the
// accumulation.  The staged record carries hx = -conic_x / 2, ny = -conic_y and
// hz = -conic_z / 2, so the exponent
//     power = hx dx^2 + ny dx dy + hz dy^2
// is two nested multiply-adds (pair_exponent: five instructions), and the
// opacity enters through its base-2 logarithm:
//     alpha = min(0.99, exp2(power * log2(e) + log2(opacity))),
// one more multiply-add and the hardware exp2.  Fused multiply-adds round
// once where the scalar formula rounds twice, so `power` agrees with a scalar
// evaluation to the rounding of its terms, not bit for bit: a pair whose alpha
// lies within that distance of 1/255 may be decided either way (the checker
// counts those pairs per pixel).
//
// Nothing here is conditional per lane: a rejected pair goes through with
// exp2(-inf) = 0, and a pixel that has finished (its next T would fall below
// 1e-4) with T = 0, so that w = alpha T is zero for both and T - alpha T is T.
// `limit` is 1e-4 while the pixel is live and -1 afterwards (a finished
// pixel cannot finish again), `last` the T it finished with.
//
// The lists' walk (walk_lists) evaluates the four entries of a round side by
// side, without a branch: T never grows, so one test behind the round finds
// the pixels that finish in it, and the round is then repeated entry by entry
// from its alphas; and a batch whose records are all definite() needs no test
// for exponents above zero.  A branch per entry and
// test held up the issue of the next entry's instructions, above all with one
// wavefront per SIMD: blend of 10k Gaussians at 256x256 20.4 -> 15.7 us, 1M
// large splats at 1080p 145 -> 134, 6M 292 -> 276, 20M at 4K 706 -> 676.
// Batches with a record that is not definite make that test for each entry,
// behind one branch per round that all lanes take alike (within 1 % of no
// branch for the others, where a second copy of the walk spills registers and
// the test for every batch costs up to 5 %).  One long needle is staged by many
// tiles, and a walk entry by entry took such a scene from 151 to 203 us; this
// one to 157.
//
// The accumulation itself, four channels times w, is one matrix instruction of
// sixteen 4x4x1 products: the four lanes of a quad hold w of four consecutive
// pixels (left operand) and one channel each of their common Gaussian (right
// operand), so lane j collects channel j of the quad's pixels, pixel i in
// register i.  It takes the time of two vector instructions where the four
// multiply-adds took that of four, and each lane reads one channel of the
// record instead of all.
// Blend of 1M Gaussians at 1080p 202 -> 198 us (issue-bound), of 10k at 256x256, one wavefront per SIMD, 38 -> 31 us.
typedef float f32x4 __attribute__((ext_vector_type(4)));

template <int kLane>
__device__ __forceinline__ float quad_lane(float v)  // value of lane kLane of each quad, in all four of them
{
    constexpr int kCtrl = kLane * 0x55;
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), kCtrl, 0xf, 0xf, false));
}

struct PixelState {
    float T, limit, last;
    f32x4 sums;
};

// One entry by itself: batches with channels that are not finite, and the verification variant.
// a = px, py, hx, ny;  b = hz, log2(opacity);  c = this lane's channel of (r, g, b, depth).  kPlain: every channel of the
// batch's records is finite.  Otherwise a pixel that rejects a Gaussian must not meet its channels even with w = 0.
template <bool kCutOnExponent, bool kPlain>
__device__ __forceinline__ void blend_one(PixelState& p, float pxf, float pyf, const float4 a, const float2 b, float c)
{
    const float dx = a.x - pxf, dy = a.y - pyf;
    const float power = pair_exponent(dx, dy, a.z, a.w, b.x);
    float t = __builtin_fmaf(power, 1.4426950408889634f, b.y);
    float alpha;
    if (kCutOnExponent) {
        const uint64_t accept = __ballot(!(power > 0.0f)) & __ballot(!(t < kAlphaCut));
        if (accept == 0ull) return;
        t = __builtin_amdgcn_inverse_ballot_w64(accept) ? t : -__builtin_inff();
        alpha = fminf(0.99f, __builtin_amdgcn_exp2f(t));
    } else {
        alpha = fminf(0.99f, __builtin_amdgcn_exp2f(t));
        if (power > 0.0f || alpha < 1.0f / 255.0f) alpha = 0.0f;
    }
    const float before = p.T;
    float w = alpha * p.T;
    p.T = __builtin_fmaf(-alpha, p.T, p.T);  // the transmittance behind the pair, rounded once
    const uint64_t finished = __ballot(p.T < p.limit);
    if (finished != 0ull) {  // (once in a pixel's life)
        if (__builtin_amdgcn_inverse_ballot_w64(finished)) {
            p.last = before;
            p.limit = -1.0f;
            w = p.T = 0.0f;
        }
    }
    if (kPlain) {
        p.sums = __builtin_amdgcn_mfma_f32_4x4x1f32(w, c, p.sums, 0, 0, 0);
    } else {
        const float ws[4] = {quad_lane<0>(w), quad_lane<1>(w), quad_lane<2>(w), quad_lane<3>(w)};
#pragma unroll
        for (int i = 0; i < 4; ++i) p.sums[i] = ws[i] != 0.0f ? __builtin_fmaf(ws[i], c, p.sums[i]) : p.sums[i];
    }
}

using ListEntry = uint16_t;
// Records staged per round: so many that eight workgroups fit into a CU's LDS, with at most 64 registers eight wavefronts per
// SIMD in the place of seven (256, and room behind the lists for one round more).  Blend of 1M large splats at 1080p 133.5 ->
// 129.5 us, of 6M 288 -> 283, octree frame 47.8 -> 45.3; with the next batch's indices requested a batch ahead (a latency less
// per batch: 10k Gaussians, a wavefront per SIMD, 16.1 -> 15.6) and the lists padded by their own lane groups side by side.
constexpr int kBatch = 252;
constexpr uint32_t kNullEntry = kBatch * 16;  // list entry of the null record (opacity 0: rejected by every pixel)
constexpr int kListWords = kBatch + 4;  // entries per list: a batch, padded to a multiple of four, one round read ahead

// kCull: staging a record also finds which of the tile's sixteen 4x4 blocks its
// alpha >= 1/255 ellipse can reach (TileReach), and each wavefront appends the
// Gaussians that reach its four blocks, in depth order, to the blocks' lists.  A (block, Gaussian) pair
// that is left out is one whose 16 pixels would all have taken the
// `alpha < 1/255` branch, and every pixel still sees its Gaussians front to
// back with the same arithmetic, so both variants produce identical images.
// List entries are the byte offsets of the staged records (16 x record number)
// in 16 bits (32-bit entries would serve as LDS addresses as they are, but the
// larger lists cost two workgroups per CU and 20 % of the kernel's speed); the
// lists are padded with the null record to a common length that is a multiple
// of four, so the walk needs no per-entry length test and reads four entries at
// a time.
template <bool kCull>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(8, 8))) void blend_kernel(FrameArgs f, const gs355_header* __restrict__ header,
                                                    const uint32_t* __restrict__ ranges,
                                                    const uint4* __restrict__ order,
                                                    const uint32_t* __restrict__ values,
                                                    const float* __restrict__ records, float* __restrict__ image,
                                                    float* __restrict__ out_depth, float* __restrict__ out_alpha)
{
    __shared__ float4 s_a[kBatch + 1];  // px, py, -conic_x / 2, -conic_y          (+ the null record)
    __shared__ float4 s_b[kBatch + 1];  // -conic_z / 2, log2(opacity), mask of the blocks it can reach, unused
    __shared__ float4 s_c[kBatch + 1];  // r, g, b, depth
    // bit 0: all pixels of the wavefront finished; it staged 1: a channel that is not finite, 2: a record that is not definite
    __shared__ uint32_t s_wave_state[4];
    // per wavefront and 4x4 block: byte offsets of the staged records of the Gaussians that can reach the block
    __shared__ __align__(8) ListEntry s_list[kCull ? 4 : 1][4][kListWords];

    if (header->overflow) return;
    const BlendTile list(header, ranges, order);
    const int tile = (int)list.tile;
    const int tile_x = tile % f.grid_x, tile_y = tile / f.grid_x;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const int group = lane >> 4, sub = lane & 15;  // 4x4 block within the quadrant, pixel within the block
    const int qx0 = tile_x * kTile + (wave & 1) * 8, qy0 = tile_y * kTile + (wave >> 1) * 8;
    const int px = qx0 + (group & 1) * 4 + (sub & 3), py = qy0 + (group >> 1) * 4 + (sub >> 2);
    const bool inside = px < f.W && py < f.H;
    const float pxf = (float)px, pyf = (float)py;
    const int first_bit = 8 * (wave >> 1) + 2 * (wave & 1);  // the quadrant's first block in a record's block mask

    const uint32_t lo = list.lo, hi = list.hi;
    PixelState p = {inside ? 1.0f : 0.0f, inside ? 0.0001f : -1.0f, 1.0f, {0.f, 0.f, 0.f, 0.f}};
    if (tid == 0) {  // the null record: zero conic and log2(opacity) = -inf give alpha = 0
        s_a[kBatch] = make_float4(0.f, 0.f, 0.f, 0.f);
        s_b[kBatch] = make_float4(0.f, -__builtin_inff(), 0.f, 0.f);
        s_c[kBatch] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    const char* const rec_a = reinterpret_cast<const char*>(s_a);
    const char* const rec_b = reinterpret_cast<const char*>(s_b);
    const char* const rec_c = reinterpret_cast<const char*>(s_c);
    const uint32_t channel = 4u * (uint32_t)(lane & 3);
    struct Staged {
        float4 a;
        float2 b;
        float c;
    };
    auto fetch = [&](uint32_t entry) {
        return Staged{*reinterpret_cast<const float4*>(rec_a + entry), *reinterpret_cast<const float2*>(rec_b + entry),
                      *reinterpret_cast<const float*>(rec_c + entry + channel)};
    };
    // the four lane groups walk their lists side by side, four entries per round
    auto walk_lists = [&](bool all_definite, uint32_t quads) {
        const uint2* __restrict__ mine = reinterpret_cast<const uint2*>(s_list[wave][group]);
        uint2 next = mine[0];  // read ahead by one round (rounds past the end are never used)
        for (uint32_t left = quads; left != 0u; --left) {
            const Staged e[4] = {fetch(next.x & 0xFFFFu), fetch(next.x >> 16), fetch(next.y & 0xFFFFu), fetch(next.y >> 16)};
            next = *++mine;
            float power[4], t[4], alpha[4], w[4], T = p.T;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float dx = e[q].a.x - pxf, dy = e[q].a.y - pyf;
                power[q] = pair_exponent(dx, dy, e[q].a.z, e[q].a.w, e[q].b.x);
                t[q] = __builtin_fmaf(power[q], 1.4426950408889634f, e[q].b.y);
            }
            if (!all_definite) {
#pragma unroll
                for (int q = 0; q < 4; ++q) t[q] = power[q] > 0.0f ? -__builtin_inff() : t[q];
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) alpha[q] = fminf(0.99f, __builtin_amdgcn_exp2f(t[q] < kAlphaCut ? -__builtin_inff() : t[q]));
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                w[q] = alpha[q] * T;
                T = __builtin_fmaf(-alpha[q], T, T);
            }
            // T never grows, so that a pixel that finishes within the round shows at its end
            if (__ballot(T < p.limit) != 0ull) {
                T = p.T;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float behind = __builtin_fmaf(-alpha[q], T, T);
                    const bool finishes = behind < p.limit;
                    if (finishes) {
                        p.last = T;
                        p.limit = -1.0f;
                    }
                    w[q] = finishes ? 0.0f : alpha[q] * T;
                    T = finishes ? 0.0f : behind;
                }
                if (__ballot(T > 0.0f) == 0ull) left = 1u;  // (the last round: every pixel has finished)
            }
            p.T = T;
#pragma unroll
            for (int q = 0; q < 4; ++q) p.sums = __builtin_amdgcn_mfma_f32_4x4x1f32(w[q], e[q].c, p.sums, 0, 0, 0);
        }
    };
    auto walk_lists_carefully = [&](uint32_t quads) {
#pragma unroll 1
        for (uint32_t i = 0; i < 4u * quads; ++i) {
            const Staged e = fetch(s_list[wave][group][i]);
            blend_one<true, false>(p, pxf, pyf, e.a, e.b, e.c);
        }
    };
    auto walk_all = [&](auto plain, int count) {
        for (int k = 0; k < count; ++k) {
            if (__ballot(p.T > 0.0f) == 0ull) break;
            const Staged e = fetch((uint32_t)k * 16u);
            blend_one<false, plain.value>(p, pxf, pyf, e.a, e.b, e.c);
        }
    };

    // this thread's Gaussian of the batch, requested one batch ahead
    uint32_t index = lo + tid < hi ? values[lo + tid] : 0u;
    for (uint32_t base = lo; base < hi; base += kBatch) {
        const uint64_t live = __ballot(p.T > 0.0f);  // lanes whose pixel is still accumulating
        const bool wave_done = live == 0ull;
        bool finite = true, is_definite = true;
        const uint32_t j = base + tid;
        if (tid < kBatch && j < hi) {
            const uint32_t g = index;
            if (j + kBatch < hi) index = values[j + kBatch];
            const float4* __restrict__ rec = reinterpret_cast<const float4*>(records + (size_t)g * kRecordFloats);
            const float4 r0 = rec[0], r1 = rec[1], r2 = rec[2];
            // a negative opacity gives a negative alpha, which every pixel rejects: log2(0) = -inf does the same
            const float log2o = __builtin_amdgcn_logf(r1.y < 0.0f ? 0.0f : r1.y);
            s_a[tid] = make_float4(r0.x, r0.y, -0.5f * r0.z, -r0.w);
            uint32_t mask = 0u;
            if (kCull) {
                const TileReach reach(r0.x, r0.y, r0.z, r0.w, r1.x, r2.z, r2.w, (float)(tile_x * kTile), (float)(tile_y * kTile));
#pragma unroll
                for (int b = 3; b >= 0; --b) mask = (mask << 4) | reach.row((float)b);
                mask = reach.unless_infinite(mask, 0xFFFFu);
                is_definite = definite(r0.z, reach.rho);
            }
            s_b[tid] = make_float4(-0.5f * r1.x, log2o, __uint_as_float(mask), 0.f);
            s_c[tid] = make_float4(r1.z, r1.w, r2.x, r2.y);
            // (the sum of the magnitudes overflows only where one of them is beyond 2^125: then the careful way is right too)
            finite = fabsf(r1.z) + fabsf(r1.w) + fabsf(r2.x) + fabsf(r2.y) < __builtin_inff();
        }
        const bool all_finite = __ballot(!finite) == 0ull, all_definite = __ballot(!is_definite) == 0ull;
        if (lane == 0) s_wave_state[wave] = (wave_done ? 1u : 0u) | (all_finite ? 0u : 2u) | (all_definite ? 0u : 4u);
        __syncthreads();
        const uint32_t w0 = s_wave_state[0], w1 = s_wave_state[1], w2 = s_wave_state[2], w3 = s_wave_state[3];
        if ((w0 & w1 & w2 & w3 & 1u) != 0u) break;
        const int unusual = __builtin_amdgcn_readfirstlane((int)((w0 | w1 | w2 | w3) & 6u));
        const int count = (int)min((uint32_t)kBatch, hi - base);
        if (!wave_done) {
            if (kCull) {
                // ---- lists: which staged Gaussians reach which 4x4 block (lane = Gaussian) ----
                uint32_t len[4] = {0u, 0u, 0u, 0u};  // uniform over the wavefront
                // A block's lane mask is the result register of one comparison, and a lane's rank among the mask's lanes
                // the hardware's masked bit count.
                for (int chunk = 0; chunk < count; chunk += 64) {
                    const int k = chunk + lane;
                    const uint32_t reached = k < count ? __float_as_uint(s_b[k].z) >> first_bit : 0u;
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        // a block whose 16 pixels have all finished gets no entries (its lane group idles through
                        // the null record while the other blocks of the wavefront are served)
                        if (((live >> (16 * b)) & 0xFFFFull) == 0ull) continue;
                        const uint64_t m = __ballot((reached & (1u << (4 * (b >> 1) + (b & 1)))) != 0u);
                        if (__builtin_amdgcn_inverse_ballot_w64(m))
                            s_list[wave][b][lanes_below_in(m, len[b])] = (ListEntry)(k * 16);
                        len[b] += (uint32_t)__popcll(m);
                    }
                }
                const uint32_t longest = (uint32_t)__builtin_amdgcn_readfirstlane(
                    (int)max(max(len[0], len[1]), max(len[2], len[3])));
                const uint32_t quads = (longest + 3u) / 4u;
                // every lane group pads its list with the null record up to the common length
                uint32_t mine = len[0];
                mine = group == 1 ? len[1] : mine;
                mine = group == 2 ? len[2] : mine;
                mine = group == 3 ? len[3] : mine;
                for (uint32_t at = mine + (uint32_t)sub; at < quads * 4u; at += 16u)
                    s_list[wave][group][at] = (ListEntry)kNullEntry;
                // a wavefront's LDS operations execute in order: its list writes precede the reads below
                wave_lds_sync();
                if ((unusual & 2) == 0) walk_lists(unusual == 0, quads);
                else walk_lists_carefully(quads);
            } else {
                if (unusual == 0) walk_all(std::true_type{}, count);
                else walk_all(std::false_type{}, count);
            }
        }
        __syncthreads();
    }

    // lane j of a quad holds channel j of the quad's four pixels
    const float T = p.limit > 0.0f ? p.T : p.last;
    const float quad_T[4] = {quad_lane<0>(T), quad_lane<1>(T), quad_lane<2>(T), quad_lane<3>(T)};
    const int j = lane & 3, x0 = px - j;
    const size_t plane = (size_t)f.W * f.H;
    float* const dst = j < 3 ? image + (size_t)j * plane : out_depth;
    const float bg = j < 3 ? f.bg[j] : 0.0f;
    const size_t o = (size_t)py * f.W + x0;
    f32x4 v;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = p.sums[i] + quad_T[i] * bg;
    if (py < f.H && dst) {
        // (rows of a multiple of four floats keep the 16-B alignment of their plane)
        if ((f.W & 3) == 0 && ((reinterpret_cast<uintptr_t>(image) | reinterpret_cast<uintptr_t>(out_depth)) & 15u) == 0u) {
            if (x0 < f.W) *reinterpret_cast<f32x4*>(dst + o) = v;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                if (x0 + i < f.W) dst[o + i] = v[i];
        }
    }
    if (inside && out_alpha) out_alpha[(size_t)py * f.W + px] = 1.0f - T;
}

}  // namespace

int launch_fill_u32(uint32_t* p, size_t n, uint32_t v, hipStream_t s)
{
    if (n == 0) return GS355_OK;
    hipLaunchKernelGGL(fill_u32_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n, v);
    GS355_CHECK_LAUNCH("fill");
    return GS355_OK;
}

int launch_ranges(const gs355_header* header, uint32_t n_cap, const uint64_t* keys, uint32_t* ranges, int tiles,
                  hipStream_t s)
{
    const int rc = launch_fill_u32(ranges, (size_t)tiles * 2, 0u, s);
    if (rc) return rc;
    if (n_cap == 0) return GS355_OK;
    hipLaunchKernelGGL(ranges_kernel, dim3((n_cap + 255) / 256), dim3(256), 0, s, header, keys, ranges,
                       (uint32_t)tiles);
    GS355_CHECK_LAUNCH("ranges");
    return GS355_OK;
}

int launch_blend(const FrameArgs& f, const gs355_header* header, const uint32_t* ranges, const uint4* order, const uint32_t* values,
                 const float* records, float* image, float* depth, float* alpha, bool cull, hipStream_t s)
{
    const int tiles = f.grid_x * f.grid_y;
    if (cull)
        hipLaunchKernelGGL(blend_kernel<true>, dim3(tiles), dim3(256), 0, s, f, header, ranges, order, values, records, image,
                           depth, alpha);
    else
        hipLaunchKernelGGL(blend_kernel<false>, dim3(tiles), dim3(256), 0, s, f, header, ranges, order, values, records, image,
                           depth, alpha);
    GS355_CHECK_LAUNCH("blend");
    return GS355_OK;
}

}  // namespace gs355
