// Per-Gaussian preprocess and key duplication for gfx950.
//
// Replaces the per-Gaussian stage of the rasterizer behind the reference's
// GaussianRasterizer.forward / .visible_filter (call sites:
// benchmarks/nerf/origin_gs/gs_model.py:211-220, 327-329).  The in-tree Python
// statements of two sub-steps are followed for layout and constants:
//   SH -> RGB            landmark/nerf_components/utils/sh_utils.py:24-94
//   scale/quat -> cov3D  landmark/nerf_components/utils/general_utils.py:64-102
//
// This translation unit is compiled with -ffp-contract=off: depth bits,
// radius and the tile rectangle feed the integer pipeline (keys, sort order,
// ranges), so every expression here is evaluated as unfused IEEE fp32 in the
// written order, with correctly rounded division and square root.
#include "gs355_internal.h"

namespace gs355 {

namespace {

constexpr float kShC0 = 0.28209479177387814f;
constexpr float kShC1 = 0.4886025119029199f;
constexpr float kShC2[5] = {1.0925484305920792f, -1.0925484305920792f, 0.31539156525252005f,
                            -1.0925484305920792f, 0.5462742152960396f};
constexpr float kShC3[7] = {-0.5900435899266435f, 2.890611442640554f, -0.4570457994644658f,
                            0.3731763325901154f, -0.4570457994644658f, 1.445305721320277f,
                            -0.5900435899266435f};

// 3D covariance, packed upper triangle, from scale and (r,x,y,z) quaternion.
__device__ __forceinline__ void covariance3d(const float* __restrict__ scale, float mod,
                                             const float* __restrict__ quat, float cov[6])
{
    const float sx = mod * scale[0], sy = mod * scale[1], sz = mod * scale[2];
    const float r = quat[0], x = quat[1], y = quat[2], z = quat[3];
    // rows of the rotation, each column scaled by its axis length
    const float l00 = (1.f - 2.f * (y * y + z * z)) * sx, l01 = (2.f * (x * y - r * z)) * sy,
                l02 = (2.f * (x * z + r * y)) * sz;
    const float l10 = (2.f * (x * y + r * z)) * sx, l11 = (1.f - 2.f * (x * x + z * z)) * sy,
                l12 = (2.f * (y * z - r * x)) * sz;
    const float l20 = (2.f * (x * z - r * y)) * sx, l21 = (2.f * (y * z + r * x)) * sy,
                l22 = (1.f - 2.f * (x * x + y * y)) * sz;
    cov[0] = (l00 * l00 + l01 * l01) + l02 * l02;
    cov[1] = (l00 * l10 + l01 * l11) + l02 * l12;
    cov[2] = (l00 * l20 + l01 * l21) + l02 * l22;
    cov[3] = (l10 * l10 + l11 * l11) + l12 * l12;
    cov[4] = (l10 * l20 + l11 * l21) + l12 * l22;
    cov[5] = (l20 * l20 + l21 * l21) + l22 * l22;
}

// Real SH basis of degree 0..3 at the unit direction (dx, dy, dz), with the
// sign of each term folded in, so that colour = sum_k basis[k] * sh[k].
// Each value is the product the closed-form expression multiplies the
// coefficient by, associated the same way ((C * a) * b).
__device__ __forceinline__ void sh_basis(int degree, float dx, float dy, float dz, float b[16])
{
    const float len = sqrtf((dx * dx + dy * dy) + dz * dz);
    dx = dx / len;
    dy = dy / len;
    dz = dz / len;
    b[0] = kShC0;
    if (degree > 0) {
        b[1] = -(kShC1 * dy);
        b[2] = kShC1 * dz;
        b[3] = -(kShC1 * dx);
        if (degree > 1) {
            const float xx = dx * dx, yy = dy * dy, zz = dz * dz;
            const float xy = dx * dy, yz = dy * dz, xz = dx * dz;
            b[4] = kShC2[0] * xy;
            b[5] = kShC2[1] * yz;
            b[6] = kShC2[2] * (2.0f * zz - xx - yy);
            b[7] = kShC2[3] * xz;
            b[8] = kShC2[4] * (xx - yy);
            if (degree > 2) {
                b[9] = kShC3[0] * dy * (3.0f * xx - yy);
                b[10] = kShC3[1] * xy * dz;
                b[11] = kShC3[2] * dy * (4.0f * zz - xx - yy);
                b[12] = kShC3[3] * dz * (2.0f * zz - 3.0f * xx - 3.0f * yy);
                b[13] = kShC3[4] * dx * (4.0f * zz - xx - yy);
                b[14] = kShC3[5] * dz * (xx - yy);
                b[15] = kShC3[6] * dx * (xx - 3.0f * yy);
            }
        }
    }
}

// res[c] += sum over coefficients k in [kFirst, kFirst + kCount) below
// `terms` of basis[k] * sh[3 * (k - kFirst) + c], added one by one in
// ascending k: `sh` points at coefficient kFirst of a [M,3] block
// (coefficient-major, RGB innermost) in global memory or in LDS.
template <int kFirst, int kCount>
__device__ __forceinline__ void sh_accumulate(int terms, const float* sh, const float b[16], float res[3])
{
#pragma unroll
    for (int k = 0; k < kCount; ++k) {
        if (kFirst + k < terms) {
#pragma unroll
            for (int c = 0; c < 3; ++c) res[c] = res[c] + b[kFirst + k] * sh[3 * k + c];
        }
    }
}

__device__ __forceinline__ void sh_finish(float res[3])
{
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const float v = res[c] + 0.5f;
        res[c] = v < 0.0f ? 0.0f : v;
    }
}

// One wavefront fetches the SH blocks of up to 64 Gaussians with coalesced 16-B loads (twelve lanes per block of sixteen
// coefficients) and each lane then evaluates the colour of its own entry from LDS.  `owner[e]` is the position of entry e's
// Gaussian within the workgroup's 256 (entries are the workgroup's surviving Gaussians, packed in order), so the
// loads touch survivors' blocks only, however few of the 256 survived.  A row of the staging area holds an
// entry's coefficients and, behind them, the Gaussian's position on the way in and its colour on the way out.
//
// kCoeffs: coefficients per Gaussian, 4, 9 or 16 (degrees 1 to 3).  kSplit: the split storage of the stored parameters (9 or 16),
// whose first coefficient (12 B per Gaussian) is read by the entry's own lane, and the others as a row of their own.
// Rows of a multiple of four floats are 16-B chunks as they are.  The others (27 floats of nine coefficients, 45 behind a
// first one) are dword-aligned and read with 16-B loads all the same: a Gaussian's row starts up to three floats
// behind a 16-B boundary, (row * kRow) & 3, and spans kChunks aligned chunks.  They land in the staging row as they are,
// so that the coefficients of entry e start at that float of its row.  `n_floats`: kRow P.  The last chunk of the last row
// may reach past the array: it is pulled back inside, and that row's last floats are fetched by its own lane.
//
// What it is for: a lane that reads its own block asks for a cache line per dword, and 64 lanes' blocks of 108 B are more
// lines than the L1 keeps until their next dword (staged_blocks).
//
// fetch() and colour() are apart so that the caller has work to do while the blocks travel.
template <bool kSplit, int kCoeffs>
struct ShEntries {
    static constexpr int kRow = 3 * (kSplit ? kCoeffs - 1 : kCoeffs);  // floats per Gaussian
    static constexpr bool kWhole = kRow % 4 == 0;
    static constexpr int kChunks = kWhole ? kRow / 4 : (kRow + 6) / 4;  // 16-B loads per row, and per lane for 64 rows
    static constexpr int kBeside = 4 * kChunks;  // floats before the position / colour
    // floats per row of the staging area: 4 modulo 8 keeps the 16-B reads of the 64 lanes on distinct banks
    static constexpr int kStride = 4 * (kChunks + 1 + kChunks % 2);

    typedef float f4v __attribute__((ext_vector_type(4)));
    f4v v[kChunks];
    float first_coeff[3];
    size_t row, last_chunk;

    // all loads are in flight together; slots past the last entry re-read that entry (same value, same address)
    __device__ __forceinline__ void fetch(const float* __restrict__ shs, const float* __restrict__ rest, size_t n_floats,
                                          size_t group_first, const uint8_t* __restrict__ owner, int first_entry, int count,
                                          int lane)
    {
        last_chunk = n_floats / 4 - 1;  // (one row alone is two chunks or more)
        const f4v* __restrict__ chunks = reinterpret_cast<const f4v*>(kSplit ? rest : shs);
#pragma unroll
        for (int it = 0; it < kChunks; ++it) {
            if (it * 64 >= kChunks * count) break;  // uniform: fewer survivors, fewer loads
            const int q4 = it * 64 + lane;
            const int e = min(q4 / kChunks, count - 1), m = q4 % kChunks;
            const size_t i = group_first + owner[first_entry + e];
            // (read once per frame: a streaming load, which leaves the cache to the records the blend gathers)
            if (kWhole)
                v[it] = __builtin_nontemporal_load(chunks + i * (kRow / 4) + m);
            else
                v[it] = __builtin_nontemporal_load(chunks + min(i * kRow / 4 + m, last_chunk));
        }
        row = group_first + owner[first_entry + min(lane, count - 1)];
        if (kSplit)
#pragma unroll
            for (int c = 0; c < 3; ++c) first_coeff[c] = __builtin_nontemporal_load(&shs[3 * row + c]);
    }

    __device__ __forceinline__ void colour(float4* __restrict__ mine, const float* __restrict__ shs, const float* __restrict__ rest,
                                           int count, int lane, int degree, const float* campos)
    {
#pragma unroll
        for (int it = 0; it < kChunks; ++it) {
            if (it * 64 >= kChunks * count) break;
            const int q4 = it * 64 + lane;
            mine[min(q4 / kChunks, count - 1) * (kStride / 4) + q4 % kChunks] = make_float4(v[it].x, v[it].y, v[it].z, v[it].w);
        }
        wave_lds_sync();
        if (lane >= count) return;
        float* __restrict__ slot = reinterpret_cast<float*>(mine) + lane * kStride;
        float* __restrict__ coeffs = slot + (kWhole ? 0 : (int)((uint32_t)row * (uint32_t)kRow & 3u));
        if (!kWhole && (row + 1) * kRow > 4 * (last_chunk + 1))  // the array's last row, where its length is no multiple of four
            for (int k = (int)(4 * (last_chunk + 1) - row * kRow); k < kRow; ++k) coeffs[k] = (kSplit ? rest : shs)[row * kRow + k];
        float b[16], rgb[3] = {0.f, 0.f, 0.f};
        sh_basis(degree, slot[kBeside] - campos[0], slot[kBeside + 1] - campos[1], slot[kBeside + 2] - campos[2], b);
        const int terms = (degree + 1) * (degree + 1);
        if (kSplit) {
            sh_accumulate<0, 1>(terms, first_coeff, b, rgb);
            sh_accumulate<1, kCoeffs - 1>(terms, coeffs, b, rgb);
        } else {
            sh_accumulate<0, kCoeffs>(terms, coeffs, b, rgb);
        }
        sh_finish(rgb);
#pragma unroll
        for (int c = 0; c < 3; ++c) slot[kBeside + c] = rgb[c];
    }
};

// Octree-GS level-of-detail test of one anchor, in the reference's order of fp32 operations
// (octreegs_encoding.py:251-264).
__device__ __forceinline__ bool lod_keeps(const gs355_anchor_lod& l, float log2_fork, int i, float x, float y, float z,
                                          const float* campos)
{
    const float level = l.level[i];
    const float shift = (0.5f * l.voxel_size) / powf(l.fork, level);
    const float dx = (x + shift) - campos[0], dy = (y + shift) - campos[1], dz = (z + shift) - campos[2];
    const float dist = sqrtf((dx * dx + dy * dy) + dz * dz) * l.resolution_scale;
    const float pred = log2f(l.standard_dist / dist) / log2_fork + l.extra_level[i];
    float r = l.rounding == 0 ? floorf(pred) : l.rounding == 1 ? rintf(pred) : ceilf(pred);
    r = fminf(fmaxf(r, 0.0f), (float)l.max_level);  // NaN -> 0
    return level <= r;
}

// The word of the tiles a splat is blended in (TileRegion), from its tile rectangle and its reach.  Rows of a masked region
// are evaluated here, once per Gaussian, so that the kernels that count and place the pairs only walk bits; larger regions
// leave that to the wavefronts that expand them.  A row costs some 30 vector instructions and splats of small scenes have
// one to three of them, in a kernel that waits for memory: 6M Gaussians at 1080p 304 -> 306 us while the SH blocks are on
// their way (317 ahead of them), 1M large splats 57 -> 59.  What it saves (6M / 1M / 20M Gaussians, the last at 4K):
// scatter 123 -> 97 / 102 -> 73 / 322 -> 260 us, sort 117 -> 83 / 115 -> 63 / 197 -> 160, blend 323 -> 292 / 164 -> 145 /
// 785 -> 706, blend backward 1025 -> 870 (6M).
__device__ __forceinline__ uint64_t tile_region(const Rect q, float px, float py, float qx, float qy, float qz, float ex, float ey)
{
    const uint64_t whole = whole_region(q);
    if (!(ex < INFINITY)) return whole;
    if (ex < 0.0f) return 0;
    const float x = px - (float)(q.x0 * kTile), y = py - (float)(q.y0 * kTile);
    int c0, c1, r0, r1;
    TileSpans::tiles_of(x - ex, x + ex, q.x1 - q.x0, c0, c1);
    TileSpans::tiles_of(y - ey, y + ey, q.y1 - q.y0, r0, r1);
    const int w = c1 - c0, h = r1 - r0;
    if (w <= 0 || h <= 0) return 0;
    const int x0 = q.x0 + c0, y0 = q.y0 + r0;
    const uint64_t corner = (uint64_t)x0 | ((uint64_t)y0 << 16);
    if (w > kMaskWidth || w * h > kMaskTiles)
        return corner | ((uint64_t)((x0 + w) | 0x8000) << 32) | ((uint64_t)(y0 + h) << 48);
    const TileSpans spans(px, py, qx, qy, qz, ex, ey, x0, y0);
    uint32_t mask = 0u;
    for (int r = 0; r < h; ++r) {
        int first, end;
        spans.columns(r, w, first, end);
        mask |= (((1u << end) - 1u) & ~((1u << first) - 1u)) << (r * w);
    }
    if (mask == 0u) return 0;
    return corner | ((uint64_t)(mask | ((uint32_t)(w - 1) << 28) | 0x80000000u) << 32);
}

// Scenes from which on a wavefront's records leave as whole lines: at half a million the way through LDS costs what it saves
// (colours given: 500k 14.8 us by lane, 15.0 by line; 1M 25.8 and 23.4; 130k 7.1 and 7.3).
constexpr int kRecordLinesFrom = 1 << 19;
// Scenes from which on those lines are streamed: 100 MB of records, of which the L2 keeps little for the blend whatever this kernel
// does, while what the binning reads next stays.  Preprocess within frames: 6M 299 -> 285 us, 20M at 4K 819 -> 764, stored
// parameters 311 -> 285, and the count and scatter of 20M 89 + 204 -> 82 + 196; frames of 4.5M Gaussians 2.4 % (a slab), 6.5 (a
// ball) and 0.7 (a part of a scene) quicker, of 3.3M 1.7, 3.6 and 0.4, of 2M 0.4, 0.2 and -0.1, of 1M 0.5, 0.1 and 0.
constexpr int kRecordsStreamedFrom = 1 << 21;

// kStored: g holds the vanilla model's stored parameters, activated here (the activated copies would cost a pass over
// memory each, and joining the SH coefficients one over 192 B per Gaussian: at 6M Gaussians 1.3 ms of such passes in
// front of a kernel of 0.3 ms).
// kPacked: coefficients of SH blocks that are fetched by way of LDS (ShEntries), 0: none.  The 20 to 53 KB of that leave seven to
// three wavefronts per SIMD, so calls whose blocks go by lane (staged_blocks), and those with colours given, run a kernel without it, at
// eight: 1.5M decoded Gaussians 100 -> 76 us, 600k 32.5 -> 24.5, 160k 13.8 -> 12.4.
template <bool kRadiiOnly, bool kStored, int kPacked>
__global__ __launch_bounds__(256) void preprocess_kernel(FrameArgs f, gs355_gaussians g, ParameterArgs par, FilterArgs fx,
                                                         float* __restrict__ records,
                                                         uint32_t* __restrict__ tiles_touched,
                                                         uint64_t* __restrict__ rects,
                                                         uint32_t* __restrict__ depth_bits,
                                                         uint2* __restrict__ wave_totals, uint8_t* __restrict__ lit,
                                                         int32_t* __restrict__ radii)
{
    typedef ShEntries<kStored, kPacked ? kPacked : 16> Entries;
    // staging area for the SH blocks of each wavefront's 64 Gaussians
    __shared__ float4 s_sh[kPacked ? 4 * 64 * Entries::kStride / 4 : 1];
    // the records of each wavefront on their way out, where there are no rows to take their place
    __shared__ float4 s_records[kRadiiOnly || kPacked ? 1 : 4 * 64 * 3];
    // the workgroup's surviving Gaussians, packed in order: position within the workgroup; survivors per wavefront
    __shared__ uint8_t s_owner[kPacked ? 256 : 1];
    __shared__ int s_alive[4];

    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int P = effective_count(f, g.P);
    if ((int)(blockIdx.x * blockDim.x) >= P) return;  // (uniform; the capacity behind a device-side count)
    const bool valid = i < P;
    const float* __restrict__ V = f.viewmatrix;
    const float* __restrict__ M = f.projmatrix;
    // Read here, ahead of the kernel's stores, so that it goes through the scalar cache: behind them the compiler reads it
    // with vector loads, one more latency between the SH blocks and the colours (6M Gaussians 304 -> 316 us).
    float campos[3] = {0.f, 0.f, 0.f};
    if (kPacked) {
#pragma unroll
        for (int k = 0; k < 3; ++k) campos[k] = f.campos[k];
    }

    // ---- geometry: cull, covariance, EWA projection, conic, radius, tile rectangle ----
    int radius = 0;
    uint32_t touched = 0;
    Rect rect = {0, 0, 0, 0};
    float x = 0.f, y = 0.f, z = 0.f, vz = 0.f, px = 0.f, py = 0.f, ca = 0.f, cc = 0.f, qx = 0.f, qy = 0.f, qz = 0.f;
    // Every per-Gaussian geometry input is requested before the cull decides
    // whether it is needed, instead of a chain of dependent latencies (culled
    // Gaussians cost 28 to 32 B of extra reads).  With the branch for given
    // covariances the mean arrives before the others are requested; compiled
    // apart, without that wait, the frame of 6M Gaussians stays as it is and the
    // radii-only kernel goes from 57.8 to 61 us.
    float cov[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, scale[3] = {0.f, 0.f, 0.f}, quat[4] = {0.f, 0.f, 0.f, 0.f};
    float opacity = 0.f;
    bool gated = false;  // anchor outside the level-of-detail mask (anchor prefilter only)
// (the per-Gaussian inputs are read once per frame: streaming loads)
#define GEO_LOAD(p) __builtin_nontemporal_load(&(p))
    if (valid) {
        x = GEO_LOAD(g.means3D[3 * (size_t)i]);
        y = GEO_LOAD(g.means3D[3 * (size_t)i + 1]);
        z = GEO_LOAD(g.means3D[3 * (size_t)i + 2]);
        if (kRadiiOnly && fx.use_lod) {
            gated = !lod_keeps(fx.lod, fx.log2_fork, i, x, y, z, f.campos);
            if (fx.lod_mask) fx.lod_mask[i] = gated ? 0 : 1;
        }
        if (!kStored && g.cov3D_precomp) {
#pragma unroll
            for (int k = 0; k < 6; ++k) cov[k] = g.cov3D_precomp[6 * (size_t)i + k];
        } else {
#pragma unroll
            for (int k = 0; k < 3; ++k) scale[k] = GEO_LOAD(g.scales[(kRadiiOnly ? fx.scale_stride : 3) * (size_t)i + k]);
#pragma unroll
            for (int k = 0; k < 4; ++k) quat[k] = GEO_LOAD(g.rotations[4 * (size_t)i + k]);
        }
        if (!kRadiiOnly) opacity = GEO_LOAD(g.opacities[i]);
    }
    if (valid && !gated) do {
        const float vx = ((V[0] * x + V[4] * y) + V[8] * z) + V[12];
        const float vy = ((V[1] * x + V[5] * y) + V[9] * z) + V[13];
        vz = ((V[2] * x + V[6] * y) + V[10] * z) + V[14];
        if (vz <= 0.2f) break;  // behind or too close to the camera plane

        const float hx = ((M[0] * x + M[4] * y) + M[8] * z) + M[12];
        const float hy = ((M[1] * x + M[5] * y) + M[9] * z) + M[13];
        const float hw = ((M[3] * x + M[7] * y) + M[11] * z) + M[15];
        const float inv_w = 1.0f / (hw + 0.0000001f);
        const float ndc_x = hx * inv_w, ndc_y = hy * inv_w;

        if (kStored) {
#pragma unroll
            for (int k = 0; k < 3; ++k) scale[k] = expf(scale[k]);
            const float norm = quaternion_norm(quat);
#pragma unroll
            for (int k = 0; k < 4; ++k) quat[k] = quat[k] / norm;
        }
        if (kStored || !g.cov3D_precomp) covariance3d(scale, f.scale_modifier, quat, cov);

        // EWA splatting: Jacobian of the perspective projection at the
        // (frustum-clamped) view-space mean, times the world->view rotation.
        const float lim_x = 1.3f * f.tanfovx, lim_y = 1.3f * f.tanfovy;
        const float tz = vz;
        const float tx = fminf(lim_x, fmaxf(-lim_x, vx / tz)) * tz;
        const float ty = fminf(lim_y, fmaxf(-lim_y, vy / tz)) * tz;
        const float j00 = f.focal_x / tz, j02 = -(f.focal_x * tx) / (tz * tz);
        const float j11 = f.focal_y / tz, j12 = -(f.focal_y * ty) / (tz * tz);
        // a[r][k] = sum_i J[r][i] * Rwv[i][k], Rwv[i][k] = V[4k+i]
        const float a00 = j00 * V[0] + j02 * V[2], a01 = j00 * V[4] + j02 * V[6], a02 = j00 * V[8] + j02 * V[10];
        const float a10 = j11 * V[1] + j12 * V[2], a11 = j11 * V[5] + j12 * V[6], a12 = j11 * V[9] + j12 * V[10];
        // b = a * Sigma
        const float b00 = (a00 * cov[0] + a01 * cov[1]) + a02 * cov[2];
        const float b01 = (a00 * cov[1] + a01 * cov[3]) + a02 * cov[4];
        const float b02 = (a00 * cov[2] + a01 * cov[4]) + a02 * cov[5];
        const float b10 = (a10 * cov[0] + a11 * cov[1]) + a12 * cov[2];
        const float b11 = (a10 * cov[1] + a11 * cov[3]) + a12 * cov[4];
        const float b12 = (a10 * cov[2] + a11 * cov[4]) + a12 * cov[5];
        // 2D covariance b * a^T with the 0.3 px low-pass on the diagonal
        ca = ((b00 * a00 + b01 * a01) + b02 * a02) + 0.3f;
        const float cb = (b00 * a10 + b01 * a11) + b02 * a12;
        cc = ((b10 * a10 + b11 * a11) + b12 * a12) + 0.3f;

        const float det = ca * cc - cb * cb;
        if (det == 0.0f) break;
        const float det_inv = 1.0f / det;
        const float mid = 0.5f * (ca + cc);
        const float disc = sqrtf(fmaxf(0.1f, mid * mid - det));
        const float lambda1 = mid + disc, lambda2 = mid - disc;
        const float rf = ceilf(3.0f * sqrtf(fmaxf(lambda1, lambda2)));
        if (!(rf < 1073741824.0f)) break;  // non-finite or absurd footprint
        const int rad = (int)rf;

        px = ((ndc_x + 1.0f) * (float)f.W - 1.0f) * 0.5f;
        py = ((ndc_y + 1.0f) * (float)f.H - 1.0f) * 0.5f;
        const Rect q = tile_rect(px, py, rad, f.grid_x, f.grid_y);
        const int area = (q.x1 - q.x0) * (q.y1 - q.y0);
        if (area == 0) break;

        radius = rad;
        touched = (uint32_t)area;
        rect = q;
        qx = cc * det_inv;
        qy = -cb * det_inv;
        qz = ca * det_inv;
    } while (false);

    if (valid && radii) __builtin_nontemporal_store(radius, &radii[i]);  // (no later stage reads radii)
    if (kRadiiOnly) {
        if (valid && fx.visible) fx.visible[i] = radius > 0 ? 1 : 0;
        return;
    }
    const bool alive = radius > 0;
    if (kStored && alive) opacity = logistic(opacity);
    {  // the wavefront's keys and survivors: what the frame's key count is made of
        const uint32_t keys = wave_sum(touched);
        const uint32_t visible = (uint32_t)__popcll(__ballot(alive));
        if ((threadIdx.x & 63) == 0 && valid) {
            wave_totals[i >> 6] = make_uint2(keys, visible);
            if (i == 0) *f.parts = (uint32_t)f.tile_reach;
        }
    }

    // Reach of the splat, for the culling of tiles (below) and of the blend's pixel blocks: half-extents
    // (ex, ey) of the axis-aligned box around the region where alpha can reach
    // 1/255, i.e. where 0.5 d^T Q d <= ln(255 * opacity).  The box is enlarged
    // by more than the rounding error of the blend's fp32 evaluation of the
    // exponent (bounded below by `noise`), so a pixel block outside the box is
    // certain to take the blend's `alpha < 1/255` branch on all of its pixels.
    // +inf = never cull (large or ill-conditioned splats; conics that are not
    // positive definite, to which a caller's covariances can lead: those have
    // no such box), -inf = never visible.
    float ex = 0.f, ey = 0.f;
    auto reach_and_region = [&]() {
        uint64_t region = 0;
        if (alive) {
            const float reach = (float)radius + 24.0f;  // |d| over every pixel of every touched tile
            const float noise = 2.4e-7f * (fabsf(qx) + fabsf(qy) + fabsf(qz)) * reach * reach;
            if (opacity != opacity || !(noise < 0.02f) || !(qx > 0.0f && qz > 0.0f)) {
                ex = ey = INFINITY;
            } else if (!(opacity * 255.0f * 1.0001f >= 1.0f)) {
                ex = ey = -INFINITY;
            } else {
                const float tau = fmaxf(__logf(opacity * 255.0f), 0.0f) * 1.001f + 0.05f;
                ex = sqrtf(2.0f * tau * ca) * 1.001f + 0.01f;
                ey = sqrtf(2.0f * tau * cc) * 1.001f + 0.01f;
            }
            region = tile_region(rect, px, py, qx, qy, qz, f.tile_reach ? ex : INFINITY, ey);
        }
        if (valid) {
            // (the classic scan's input, which that makes by itself where it was left out: 4 of 16 B per Gaussian)
            if (!f.tile_reach) __builtin_nontemporal_store(touched, &tiles_touched[i]);
            rects[i] = region;
        }
    };

    // ---- colour ----
    float rgb[3] = {0.f, 0.f, 0.f};
    const uint64_t alive_lanes = __ballot(alive);
    // LDS of this wavefront alone, for its records: where there are rows, of what those leave, or over those that have been read
    float4* out_rows = kPacked ? s_sh : s_records + (threadIdx.x >> 6) * 64 * 3;
    bool room = P >= kRecordLinesFrom;
    const bool given = !kStored && !kPacked && g.colors_precomp != nullptr;
    if (given) {
        if (alive) {
            rgb[0] = g.colors_precomp[3 * (size_t)i];
            rgb[1] = g.colors_precomp[3 * (size_t)i + 1];
            rgb[2] = g.colors_precomp[3 * (size_t)i + 2];
        }
        reach_and_region();
    } else {
        // kPacked: the survivors of the workgroup are packed (in order) and each wavefront fetches the SH blocks of 64 of
        // them with coalesced loads through LDS, so the memory system sees dense wavefronts however many Gaussians were
        // culled.  Else every survivor fetches its own block.  Same values and the same order of additions either way.
        if constexpr (kPacked) {
            const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
            const uint64_t m = alive_lanes;
            if (lane == 0) s_alive[wave] = __popcll(m);
            __syncthreads();
            int before = 0, total = 0;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                before += w < wave ? s_alive[w] : 0;
                total += s_alive[w];
            }
            // packed entry e lives in row e of the staging area
            float* __restrict__ my_row = reinterpret_cast<float*>(s_sh) +
                                         (before + __popcll(m & ((1ull << lane) - 1ull))) * Entries::kStride;
            if (alive) {
                s_owner[before + __popcll(m & ((1ull << lane) - 1ull))] = (uint8_t)threadIdx.x;
                my_row[Entries::kBeside] = x;
                my_row[Entries::kBeside + 1] = y;
                my_row[Entries::kBeside + 2] = z;
            }
            __syncthreads();
            // each wavefront takes a quarter of the packed survivors (entry e sits in row e of the staging area), and finds
            // its own Gaussians' tiles while their blocks are on the way
            const int share = (total + 3) / 4, first_entry = wave * share, count = min(share, total - first_entry);
            float4* __restrict__ rows = s_sh + first_entry * (Entries::kStride / 4);
            // The opacity has to be there before the blocks are requested: the number of loads behind it then depends on the
            // number of survivors, so that waiting for it would be waiting for all of them, ahead of the work that is to hide
            // them (6M Gaussians 304 -> 326 us).
            if (!kStored) asm volatile("" : "+v"(opacity));
            Entries entries;
            if (count > 0)
                entries.fetch(g.shs, par.rest, (size_t)g.P * Entries::kRow, (size_t)blockIdx.x * blockDim.x, s_owner, first_entry, count, lane);
            reach_and_region();
            if (count > 0) entries.colour(rows, g.shs, par.rest, count, lane, f.sh_degree, campos);
            __syncthreads();
            if (alive) {
#pragma unroll
                for (int c = 0; c < 3; ++c) rgb[c] = my_row[Entries::kBeside + c];
            }
            // (behind all survivors' rows, or over this wavefront's own)
            constexpr int kRow4 = Entries::kStride / 4, kOutRows = (64 * 3 + kRow4 - 1) / kRow4;
            const bool behind = total + 4 * kOutRows <= 256;
            out_rows = s_sh + (behind ? total + wave * kOutRows : before) * kRow4;
            room = room && (behind || __popcll(m) >= kOutRows);
        } else {
            reach_and_region();
            if (alive) {
                float b[16];
                sh_basis(f.sh_degree, x - f.campos[0], y - f.campos[1], z - f.campos[2], b);
                const int terms = (f.sh_degree + 1) * (f.sh_degree + 1);
                if (kStored) {
                    sh_accumulate<0, 1>(terms, g.shs + (size_t)i * 3, b, rgb);
                    sh_accumulate<1, 15>(terms, par.rest + (size_t)i * (f.sh_coeffs - 1) * 3, b, rgb);
                } else {
                    sh_accumulate<0, 16>(terms, g.shs + (size_t)i * f.sh_coeffs * 3, b, rgb);
                }
                sh_finish(rgb);
            }
        }
    }
    // Which channels are above zero is all that the backward pass wants of a colour (zero: clamped, no gradient): a byte
    // instead of 12 of the record's 48, whose cache lines it would read from end to end (preprocess backward of 6M
    // Gaussians 780 -> 723 us, for 2 us here, which the tile counts left out above give back).
    if (valid && !given) lit[i] = (uint8_t)((rgb[0] > 0.0f) | ((rgb[1] > 0.0f) << 1) | ((rgb[2] > 0.0f) << 2));
    const float4 r0 = make_float4(px, py, qx, qy), r1 = make_float4(qz, opacity, rgb[0], rgb[1]), r2 = make_float4(rgb[2], vz, ex, ey);
    if (valid) depth_bits[i] = __float_as_uint(vz);
    if (room) {
        // A wavefront's records leave as whole lines, those of 64 B that hold some of a survivor's record: what else is in
        // them is nobody's.  A lane that stores its own record makes three requests of 16 B, each of which takes a CU's path
        // to the L2 as long as one of 64, and where neighbours were culled, lines that are written in parts.  20M Gaussians of
        // which 57 / 44 / 24 % survive: 1184 / 1039 / 751 -> 1031 / 910 / 715 us (degree 0, 44 %: 666 -> 488), 6M of which
        // 88 % do 380 -> 328, their stored parameters 393 -> 347 (the kernel by itself, again and again; within frames 305 ->
        // 287 and 356 -> 301), 3.9M decoded Gaussians 78 -> 62.
        const int lane = threadIdx.x & 63;
        wave_lds_sync();
        out_rows[3 * lane] = r0;
        out_rows[3 * lane + 1] = r1;
        out_rows[3 * lane + 2] = r2;
        wave_lds_sync();
        float4* __restrict__ dst = reinterpret_cast<float4*>(records + (size_t)(i - lane) * kRecordFloats);
        const int end = 3 * min(64, P - (i - lane));
        const bool streamed = P >= kRecordsStreamedFrom;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const int at = 64 * k + lane;
            if (at < end && ((alive_lanes >> ((at & ~3) / 3)) & 3ull) != 0ull) {
                typedef float f32x4 __attribute__((ext_vector_type(4)));
                const float4 v = out_rows[at];
                if (streamed) __builtin_nontemporal_store((f32x4){v.x, v.y, v.z, v.w}, reinterpret_cast<f32x4*>(dst + at));
                else dst[at] = v;
            }
        }
    } else if (alive) {
        float4* __restrict__ rec = reinterpret_cast<float4*>(records + (size_t)i * kRecordFloats);
        rec[0] = r0;
        rec[1] = r1;
        rec[2] = r2;
    }
}

// One workgroup expands the keys of 256 consecutive Gaussians.  Output slots
// are walked by consecutive lanes (coalesced stores); each slot finds its
// source Gaussian by binary search over the group's offsets held in LDS.
__global__ __launch_bounds__(256) void duplicate_kernel(FrameArgs f, int32_t P, const float* __restrict__ records,
                                                        const int32_t* __restrict__ radii,
                                                        const uint32_t* __restrict__ offsets,
                                                        const gs355_header* __restrict__ header,
                                                        uint64_t* __restrict__ keys, uint32_t* __restrict__ values)
{
    __shared__ uint32_t s_end[256];    // inclusive offset of each Gaussian of the group
    __shared__ uint32_t s_depth[256];  // depth bits
    __shared__ int s_x0[256], s_y0[256], s_w[256];

    if (header->overflow) return;  // capacity too small: the caller redoes the frame
    P = effective_count(f, P);
    const int t = threadIdx.x;
    const int g0 = blockIdx.x * 256;
    if (g0 >= P) return;  // uniform
    const int i = g0 + t;
    const uint32_t begin = g0 == 0 ? 0u : offsets[g0 - 1];
    uint32_t end_i = begin;
    if (i < P) {
        end_i = offsets[i];
        const int rad = radii[i];
        if (rad > 0) {
            const float* rec = records + (size_t)i * kRecordFloats;
            const Rect q = tile_rect(rec[0], rec[1], rad, f.grid_x, f.grid_y);
            s_x0[t] = q.x0;
            s_y0[t] = q.y0;
            s_w[t] = q.x1 - q.x0;
            s_depth[t] = __float_as_uint(rec[9]);
        }
    }
    s_end[t] = end_i;  // threads past P repeat `begin`, harmless: never selected
    __syncthreads();
    const int last = min(255, P - 1 - g0);
    const uint32_t end = s_end[last];

    for (uint32_t j = begin + t; j < end; j += 256) {
        // smallest k with s_end[k] > j
        int lo = 0, hi = last;
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (s_end[mid] > j) hi = mid;
            else lo = mid + 1;
        }
        const uint32_t first = lo == 0 ? begin : s_end[lo - 1];
        const uint32_t local = j - first;
        const int w = s_w[lo];
        const int ty = s_y0[lo] + (int)(local / (uint32_t)w);
        const int tx = s_x0[lo] + (int)(local % (uint32_t)w);
        keys[j] = ((uint64_t)(uint32_t)(ty * f.grid_x + tx) << 32) | (uint64_t)s_depth[lo];
        values[j] = (uint32_t)(g0 + lo);
    }
}

// Whether SH blocks travel through LDS (ShEntries) or each lane reads its own.  Staged, a block is fetched whole, by three to seven
// wavefronts per SIMD; a lane fetches what the active degree needs, at eight.  So it takes a degree that needs all or most of
// the block, and a scene whose blocks the caches do not keep between a lane's dwords.  By way of LDS and by lane, us at 1080p
// with 88 % of the Gaussians on the screen:
//   16 coefficients, degree 3   131k 11.2 14.7, 800k 46 154, 6M 288 879         degree 2   131k 11.1 10.9, 300k 21 26, 6M 280 458
//   9, degree 2                 131k 10.0 9.4, 200k 13.2 14.5, 6M 215 391       stored     200k 14.5 13.6, 300k 17.4 17.7, 6M 210 340
//   4, degree 1                 524k 20.3 18.1, 800k 26.6 26.8, 6M 151 169      stored     524k 23.0 19.5, 2M 61 55, 6M 171 165
//   16, degree 1                800k 45 34, 6M 278 267                          stored     800k 49 35, 6M 292 289
//   16, degree 0                800k 45 29, 6M 279 233                          stored     800k 49 26, 6M 292 136
//   9, degree 1                 300k 17.5 14.6, 1.2M 48 46, 6M 211 250          stored     300k 17.0 14.9, 1.2M 47 42, 6M 208 227
//   9, degree 0                 300k 17.0 12.7, 1.2M 47 39, 6M 207 212          stored     300k 16.5 13.2, 1.2M 46 33, 6M 207 139
// (with 16 % on the screen nine coefficients at degree 1, 4M and 12M: 108 80 and 310 246)
bool staged_blocks(int coeffs, int degree, bool stored, int32_t P)
{
    if (coeffs == 16) return degree >= 2;
    if (coeffs == 9) return degree >= 2 && P >= (stored ? 4 << 16 : 3 << 16);
    return coeffs == 4 && degree >= 1 && !stored && P >= 3 << 18;
}

}  // namespace

int launch_preprocess(const FrameArgs& f, const gs355_gaussians& g, const ParameterArgs* par, bool radii_only, float* records,
                      uint32_t* tiles_touched, uint64_t* rects, uint32_t* depth_bits, uint2* wave_totals, uint8_t* lit,
                      int32_t* radii, hipStream_t s)
{
    if (g.P == 0) return GS355_OK;
    const dim3 block(256), grid((g.P + 255) / 256);
    const FilterArgs none;
    // (any other number of coefficients, and blocks off the 16-byte boundaries of ordinary allocations: a lane per block)
    const bool aligned = (par || !g.colors_precomp) && (reinterpret_cast<uintptr_t>(par ? par->rest : g.shs) & 15u) == 0;
    const int packed = aligned && staged_blocks(f.sh_coeffs, f.sh_degree, par != nullptr, g.P) ? f.sh_coeffs : 0;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, block, 0, s, f, g, par ? *par : ParameterArgs(), none, records, tiles_touched, rects,
                           depth_bits, wave_totals, lit, radii);
    };
    if (radii_only) launch(preprocess_kernel<true, false, 0>);
    else if (packed == 16) launch(par ? preprocess_kernel<false, true, 16> : preprocess_kernel<false, false, 16>);
    else if (packed == 9) launch(par ? preprocess_kernel<false, true, 9> : preprocess_kernel<false, false, 9>);
    else if (packed == 4) launch(preprocess_kernel<false, false, 4>);
    else launch(par ? preprocess_kernel<false, true, 0> : preprocess_kernel<false, false, 0>);
    GS355_CHECK_LAUNCH("preprocess");
    return GS355_OK;
}

int launch_anchor_filter(const FrameArgs& f, const gs355_gaussians& g, const FilterArgs& x, int32_t* radii, hipStream_t s)
{
    if (g.P == 0) return GS355_OK;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3((g.P + 255) / 256), dim3(256), 0, s, f, g, ParameterArgs(), x, (float*)nullptr,
                           (uint32_t*)nullptr, (uint64_t*)nullptr, (uint32_t*)nullptr, (uint2*)nullptr, (uint8_t*)nullptr, radii);
    };
    if (x.stored)
        launch(preprocess_kernel<true, true, 0>);
    else
        launch(preprocess_kernel<true, false, 0>);
    GS355_CHECK_LAUNCH("anchor filter");
    return GS355_OK;
}

int launch_duplicate(const FrameArgs& f, int32_t P, const float* records, const int32_t* radii,
                     const uint32_t* offsets, const gs355_header* header, uint64_t* keys, uint32_t* values,
                     hipStream_t s)
{
    if (P == 0) return GS355_OK;
    hipLaunchKernelGGL(duplicate_kernel, dim3((P + 255) / 256), dim3(256), 0, s, f, P, records, radii, offsets,
                       header, keys, values);
    GS355_CHECK_LAUNCH("duplicate");
    return GS355_OK;
}

}  // namespace gs355
