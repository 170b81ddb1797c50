// Internal declarations shared by the gs355 translation units (host side).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "gs355.h"

namespace gs355 {

constexpr int kTile = GS355_TILE;
constexpr int kRecordFloats = 12;  // px, py, conic xyz, opacity, r, g, b, depth, pad, pad

// radix sort geometry: 256 threads x kSortItems keys per workgroup, 8-bit digits
constexpr int kSortThreads = 256;
constexpr int kSortItems = 16;
constexpr int kSortTile = kSortThreads * kSortItems;
constexpr int kRadixBits = 8;
constexpr int kRadix = 1 << kRadixBits;

// tile-bucketed sort: buckets up to kTileSortCap[3] pairs are sorted in LDS; larger ones are split into such pieces first
constexpr int kTileSortCap[4] = {1024, 2048, 5120, 10240};  // in-LDS sorter size classes (pairs per bucket)

// scan geometry: 256 threads x 16 items per workgroup
constexpr int kScanThreads = 256;
constexpr int kScanItems = 16;
constexpr int kScanTile = kScanThreads * kScanItems;

struct FrameArgs {  // by-value kernel argument
    int32_t W, H, grid_x, grid_y;
    float tanfovx, tanfovy, focal_x, focal_y, scale_modifier;
    int32_t sh_degree, sh_coeffs;
    const float* viewmatrix;
    const float* projmatrix;
    const float* campos;
    const float* bg;
    const uint32_t* p_device;  // optional device-side number of Gaussians (gs355_gaussians.P_device)
    int32_t plain_regions;  // the grid is too large for flags in the tile regions' words (TileRegion)
    int32_t tile_reach;     // preprocess: a Gaussian's region is the tiles its alpha >= 1/255 ellipse reaches
    uint32_t* parts;        // preprocess: the workspace header's word for that
};

// Number of Gaussians a kernel processes: the host's P, or the device-side count when there is one.
__device__ __forceinline__ int effective_count(const FrameArgs& f, int P)
{
    if (!f.p_device) return P;
    const uint32_t n = *f.p_device;
    return n < (uint32_t)P ? (int)n : P;
}

// The stored parameters of the vanilla model in place of activated values (gs355_run_parameters): g.scales holds
// logarithms, g.rotations unnormalised quaternions, g.opacities logits, g.shs the first SH coefficient [P,1,3].
struct ParameterArgs {
    const float* rest = nullptr;  // [P, M - 1, 3]
    float* d_rest = nullptr;      // its gradient (backward pass)
};

// Extras of the radii-only preprocess when it serves the anchor prefilter (by-value kernel argument).
struct FilterArgs {
    int32_t scale_stride = 3;   // floats between the scale rows
    int32_t stored = 0;         // scales are logarithms, rotations unnormalised quaternions
    int32_t use_lod = 0;
    gs355_anchor_lod lod = {};
    float log2_fork = 1.0f;     // (float)log2((double)fork), as the reference's host-side math.log2(fork)
    uint8_t* lod_mask = nullptr;  // optional
    uint8_t* visible = nullptr;   // optional: radius > 0
};

int set_error(int code, const char* fmt, ...);

// Tile rectangle of a splat.  Only subtractions, additions and divisions by 16:
// nothing a compiler could contract, so every translation unit gets the same
// rectangle from the same (px, py, radius).
struct Rect {
    int x0, y0, x1, y1;
};

// min(grid, max(0, (int)v)) with truncation toward zero, defined for any v.
__device__ __forceinline__ int tile_clamp(float v, int grid)
{
    if (!(v > 0.0f)) return 0;
    if (v >= (float)grid) return grid;
    return (int)v;
}

__device__ __forceinline__ Rect tile_rect(float px, float py, int radius, int grid_x, int grid_y)
{
    const float r = (float)radius;
    Rect q;
    q.x0 = tile_clamp((px - r) / 16.0f, grid_x);
    q.y0 = tile_clamp((py - r) / 16.0f, grid_y);
    q.x1 = tile_clamp((px + r + 15.0f) / 16.0f, grid_x);
    q.y1 = tile_clamp((py + r + 15.0f) / 16.0f, grid_y);
    return q;
}

// the rectangle as a Gaussian's tiles (TileRegion)
__device__ __forceinline__ uint64_t whole_region(const Rect q)
{
    return (uint64_t)q.x0 | ((uint64_t)q.y0 << 16) | ((uint64_t)q.x1 << 32) | ((uint64_t)q.y1 << 48);
}

// Exponent of one (pixel, Gaussian) pair,  hx dx^2 + ny dx dy + hz dy^2  with hx = -conic_x / 2, ny = -conic_y,
// hz = -conic_z / 2 and (dx, dy) = centre - pixel, as two nested multiply-adds: five instructions.  The forward
// blend and the backward blend both call this, so the two passes see the same value and decide alike.
__device__ __forceinline__ float pair_exponent(float dx, float dy, float hx, float ny, float hz)
{
#pragma clang fp contract(off)
    const float u = hx * dx;
    const float v = __builtin_fmaf(ny, dy, u);
    const float w = hz * dy;
    const float z = w * dy;
    return __builtin_fmaf(dx, v, z);
}

// Which of a tile's sixteen 4x4 blocks the splat's alpha >= 1/255 ellipse can reach, a row of four at a time (bit = column).
// The record's reach is the half-extent (Rx, Ry) of the ellipse's bounding box; with rho = -conic_y / sqrt(conic_x conic_z)
// the ellipse's span at dy = Ry t is Rx (rho t +- sqrt((1 - rho^2)(1 - t^2))).  Over a row of blocks, t in [t0, t1], the
// upper end is largest at t = rho pulled into the interval, the lower end smallest at -rho: two spans per block row instead
// of the bounding box for all of them.  (A row beyond the ellipse gives sqrt(negative) = NaN, and no blocks.)
// The reach contains the rounding of the exponent (gs355_preprocess.hip); `slack` covers that its margin was added to Rx
// and Ry separately, which bends t by up to 0.002 + 0.02 / Ry, and the rounding here.
// With the bounding box alone 36 % of the blend's list entries reached no pixel in a scene of large splats, 21 % in one of
// small ones.  About 115 vector instructions per 64 records and tile, against some 20 per list entry left out (65 in the
// backward blend): blend 198 -> 161 us (1M large splats, 1080p), 361 -> 334 us (6M), 969 -> 903 us (20M, 4K), 304 -> 290 us
// (500k anchors).
struct TileReach {
    float rho, across, scale, left, right, t_first, t_step, t_span, reach;

    __device__ __forceinline__ TileReach(float px, float py, float conic_x, float conic_y, float conic_z, float reach_x,
                                         float reach_y, float tile_x0, float tile_y0)
    {
        const float inv_y = __builtin_amdgcn_rcpf(reach_y);
        rho = fmaxf(-1.0f, fminf(1.0f, -conic_y * __builtin_amdgcn_rsqf(conic_x * conic_z)));
        across = __builtin_amdgcn_sqrtf(fmaxf(0.0f, __builtin_fmaf(-rho, rho, 1.0f)) + 1e-5f);
        const float slack = __builtin_fmaf(reach_x, __builtin_fmaf(0.02f, inv_y, 0.002f), 0.01f);
        const float x = px - tile_x0;
        t_first = (tile_y0 - py) * inv_y;
        t_step = 4.0f * inv_y;
        t_span = 3.0f * inv_y;
        // block columns below trunc(right end + 1) and from trunc(left end + almost 1) on are reached
        right = __builtin_fmaf(0.25f, x + slack, 1.0f);
        left = __builtin_fmaf(0.25f, x - slack, 0.2499f);
        scale = 0.25f * reach_x;
        reach = reach_x;
    }

    // Rows as they come from row(), for a reach that is a number; +inf reaches `all`, -inf nothing.
    __device__ __forceinline__ uint32_t unless_infinite(uint32_t mask, uint32_t all) const
    {
        return reach < 0.0f ? 0u : reach < __builtin_inff() ? mask : all;
    }

    __device__ __forceinline__ uint32_t row(float b) const
    {
        const float t0 = __builtin_fmaf(b, t_step, t_first), t1 = t0 + t_span;
        const float up = __builtin_amdgcn_fmed3f(rho, t0, t1), down = __builtin_amdgcn_fmed3f(-rho, t0, t1);
        const float half_up = __builtin_amdgcn_sqrtf(__builtin_fmaf(-up, up, 1.0f));
        const float half_down = __builtin_amdgcn_sqrtf(__builtin_fmaf(-down, down, 1.0f));
        const float hi = __builtin_fmaf(scale, __builtin_fmaf(rho, up, across * half_up), right);
        const float lo = __builtin_fmaf(scale, __builtin_fmaf(rho, down, -(across * half_down)), left);
        const uint32_t n1 = (uint32_t)__builtin_amdgcn_fmed3f(hi, 0.0f, 4.0f), n0 = (uint32_t)__builtin_amdgcn_fmed3f(lo, 0.0f, 4.0f);
        return ((1u << n1) - 1u) & ~((1u << n0) - 1u);
    }
};

// A splat whose conic is positive and whose |rho| is below kDefinite has no pixel with an exponent above zero.  The two square
// terms of the exponent outweigh the mixed one by at least 1 - |rho| of their sum, and pair_exponent's five roundings are off
// by less than 2^-21 = 4.8e-7 of it (rho itself by 4e-7): the exponent comes out negative, or zero at the splat's centre.
// rho alone does not tell: it is that of a negative definite conic as well, which a caller's covariance can lead to (minus 0.3
// to 0.6 square pixels, before the low-pass) and whose exponents are above zero everywhere else.  Conics of mixed signs give
// |rho| = 1, as do products of the diagonal that are zero or not a number; finite conics of accepted splats stay below 2^50
// (entries of a 2D covariance that are not zero are 2^-25 or more), so that the product does not overflow.  The forward blend tests for exponents
// above zero only in batches with a record that is not definite (axes of more than 400:1 on the screen, most often).
constexpr float kDefinite = 0.99999f;
__device__ __forceinline__ bool definite(float conic_x, float rho) { return conic_x > 0.0f && fabsf(rho) < kDefinite; }

// The columns of tiles that the splat's alpha >= 1/255 ellipse can reach, for one row of tiles at a time: TileReach's span
// with tiles in the place of blocks (the same formula, and the same slack).  Rows and columns count from tile (x0, y0).
// Contraction is off: the kernels that count, place and sum the pairs of large splats each evaluate this and have to agree.
struct TileSpans {
    float rho = 0.f, across = 0.f, slack = 0.f, rx = 0.f, x = 0.f, y = 0.f, inv_y = 0.f;

    TileSpans() = default;
    __device__ __forceinline__ TileSpans(float px, float py, float conic_x, float conic_y, float conic_z, float reach_x,
                                         float reach_y, int x0, int y0)
    {
#pragma clang fp contract(off)
        inv_y = __builtin_amdgcn_rcpf(reach_y);
        rho = fmaxf(-1.0f, fminf(1.0f, -conic_y * __builtin_amdgcn_rsqf(conic_x * conic_z)));
        across = __builtin_amdgcn_sqrtf(fmaxf(0.0f, 1.0f - rho * rho) + 1e-5f);
        slack = reach_x * (0.02f * inv_y + 0.002f) + 0.01f;
        rx = reach_x;
        x = px - (float)(x0 * kTile);
        y = py - (float)(y0 * kTile);
    }
    // from a Gaussian's record
    __device__ __forceinline__ TileSpans(const float* __restrict__ record, int x0, int y0)
        : TileSpans(record[0], record[1], record[2], record[3], record[4], record[10], record[11], x0, y0)
    {
    }

    // Integers in [0, n] around the pixel interval [lo, hi] from the corner: first tile that ends at or behind lo, one
    // past the last that begins before or at hi (pixel centres are integers, a tile's last one is its first plus 15).
    static __device__ __forceinline__ void tiles_of(float lo, float hi, int n, int& first, int& end)
    {
#pragma clang fp contract(off)
        first = (int)__builtin_amdgcn_fmed3f(lo * 0.0625f + 0.0624f, 0.0f, (float)n);
        end = (int)__builtin_amdgcn_fmed3f(hi * 0.0625f + 1.0f, 0.0f, (float)n);
    }

    // columns [first, end) of the `width` tiles of row `row` (first >= end: none)
    __device__ __forceinline__ void columns(int row, int width, int& first, int& end) const
    {
#pragma clang fp contract(off)
        const float top = (float)(row * kTile) - y;
        const float t0 = __builtin_amdgcn_fmed3f(top * inv_y, -1.0f, 1.0f);
        const float t1 = __builtin_amdgcn_fmed3f((top + (float)(kTile - 1)) * inv_y, -1.0f, 1.0f);
        const float up = __builtin_amdgcn_fmed3f(rho, t0, t1), down = __builtin_amdgcn_fmed3f(-rho, t0, t1);
        const float half_up = __builtin_amdgcn_sqrtf(fmaxf(0.0f, 1.0f - up * up));
        const float half_down = __builtin_amdgcn_sqrtf(fmaxf(0.0f, 1.0f - down * down));
        const float hi = x + (rx * (rho * up + across * half_up) + slack);
        const float lo = x + (rx * (rho * down - across * half_down) - slack);
        tiles_of(lo, hi, width, first, end);
    }
};

// The tiles a Gaussian is blended in, as the word that the preprocess leaves per Gaussian (zero: none):
//   whole     x0 | y0 << 16 | x1 << 32 | y1 << 48       every tile of the rectangle
//   spans     the same with bit 47 set                  of the rectangle's tiles those inside the ellipse (TileSpans)
//   masked    x0 | y0 << 16 | mask << 32 | (width - 1) << 60 | 1 << 63
//                                                       of at most 28 tiles, at most 8 side by side, those in the mask
// Tiles of a region are numbered row by row over its rectangle, from its first row with a tile to its last.  A grid of more
// than 32767 tiles along an axis needs the flags' bits for coordinates: its regions are whole (`plain`).
// 6M Gaussians at 1080p reach 73 % of their rectangles' tiles and nearly all of their regions are masked; of 1M large
// splats 48 %, in spans a fifth.
constexpr int kMaskTiles = 28, kMaskWidth = 8;
struct TileRegion {
    int x0, y0, width, area;  // area: tile numbers in use (of a masked region up to its last tile)
    uint32_t mask;
    bool masked, spans;

    __device__ __forceinline__ TileRegion(uint64_t word, bool plain)
    {
        const uint32_t low = (uint32_t)word, high = (uint32_t)(word >> 32);
        x0 = (int)(low & 0xFFFFu);
        y0 = (int)(low >> 16);
        masked = !plain && (high >> 31) != 0u;
        spans = !plain && !masked && (high & 0x8000u) != 0u;
        mask = masked ? high & ((1u << kMaskTiles) - 1u) : 0u;
        const int x1 = (int)(high & (spans ? 0x7FFFu : 0xFFFFu)), y1 = (int)(high >> 16);
        width = masked ? (int)((high >> 28) & 7u) + 1 : x1 - x0;
        area = masked ? 32 - __clz((int)mask) : width * (y1 - y0);
    }
    // row and column of tile number e (the quotient by the reciprocal is off by one at most)
    __device__ __forceinline__ void place(int e, int& row, int& col) const
    {
        row = (int)(((float)e + 0.5f) * __builtin_amdgcn_rcpf((float)width));
        col = e - row * width;
        if (col < 0) { --row; col += width; }
        else if (col >= width) { ++row; col -= width; }
    }
    __device__ __forceinline__ int tile(int row, int col, int grid_x) const { return (y0 + row) * grid_x + x0 + col; }
    // whether tile number e is one of the region's (`s`: of a region with spans)
    __device__ __forceinline__ bool holds(int e, int row, int col, const TileSpans& s) const
    {
        if (masked) return ((mask >> e) & 1u) != 0u;
        if (!spans) return true;
        int first, end;
        s.columns(row, width, first, end);
        return col >= first && col < end;
    }
};

// The hardware exp2 is monotone, so exp2(t) < 1/255 exactly when t < kAlphaCut, the smallest float whose exp2 reaches
// 1/255 (found by running v_exp_f32 over every float between -8.2 and -7.8).  The blend (forward and backward) decides
// on t = power * log2(e) + log2(opacity) and leaves the exp2 (a quarter-rate instruction) to the pairs that pass; the
// forward blend's verification variant decides on the exponential itself, and the tests hold the two to identical
// images on scenes full of opacities around 1/255.
constexpr float kAlphaCut = -7.99435329f;  // bits 0xc0ffd1be

// stage launchers (each returns a gs355_status)
// `par` (may be NULL): g holds stored parameters
int launch_preprocess(const FrameArgs& f, const gs355_gaussians& g, const ParameterArgs* par, bool radii_only, float* records,
                      uint32_t* tiles_touched, uint64_t* rects, uint32_t* depth_bits, uint2* wave_totals, uint8_t* lit,
                      int32_t* radii, hipStream_t s);
int launch_scan_offsets(const FrameArgs& f, int32_t P, const float* records, const int32_t* radii, uint32_t* tiles_touched,
                        uint64_t* rects, uint32_t* offsets, uint32_t* scan_tmp, gs355_header* header, gs355_header* header_copy,
                        uint32_t n_cap, hipStream_t s);
int launch_anchor_filter(const FrameArgs& f, const gs355_gaussians& g, const FilterArgs& x, int32_t* radii, hipStream_t s);
int launch_duplicate(const FrameArgs& f, int32_t P, const float* records, const int32_t* radii,
                     const uint32_t* offsets, const gs355_header* header, uint64_t* keys, uint32_t* values,
                     hipStream_t s);
int launch_sort(const gs355_header* header, uint32_t n_cap, int passes, uint64_t* keys0, uint64_t* keys1,
                uint32_t* vals0, uint32_t* vals1, uint32_t* hist, uint32_t* scan_tmp, hipStream_t s);
int launch_ranges(const gs355_header* header, uint32_t n_cap, const uint64_t* keys, uint32_t* ranges, int tiles,
                  hipStream_t s);
// `order`: the tiles in the tile sort's order where header->ordered says so
int launch_blend(const FrameArgs& f, const gs355_header* header, const uint32_t* ranges, const uint4* order, const uint32_t* values,
                 const float* records, float* image, float* depth, float* alpha, bool cull, hipStream_t s);

int launch_render_backward(const FrameArgs& f, const gs355_gaussians& g, const gs355_header* header,
                           const uint32_t* ranges, const uint4* order, const uint32_t* values, const float* records,
                           const uint64_t* rects, const uint8_t* lit, const gs355_backward_inputs& in, uint2* record_slots, uint32_t* next_slot,
                           float* key_grads, const gs355_gradients& out, const ParameterArgs* par, hipStream_t s);

// Activations of the stored parameters, each with the framework's own elementwise rounding (the caller is compiled
// without contraction): the normalisation's sum of squares is taken pairwise, as its row reduction takes it.
__device__ __forceinline__ float logistic(float x) { return 1.0f / (1.0f + expf(-x)); }

__device__ __forceinline__ float quaternion_norm(const float q[4])
{
#pragma clang fp contract(off)
    const float n = sqrtf((q[0] * q[0] + q[1] * q[1]) + (q[2] * q[2] + q[3] * q[3]));
    return n < 1e-12f ? 1e-12f : n;  // (NaN stays NaN)
}

// `first` plus the number of lanes below this one that `mask` (uniform over the wavefront) holds: the hardware's masked
// bit count.
__device__ __forceinline__ uint32_t lanes_below_in(uint64_t mask, uint32_t first = 0u)
{
    return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, first));
}

// Lane exchanges inside the vector unit (no LDS): sums, minima and maxima over a wavefront.
template <int kCtrl, int kRows>
__device__ __forceinline__ uint32_t dpp(uint32_t absent, uint32_t v)
{
    return (uint32_t)__builtin_amdgcn_update_dpp((int)absent, (int)v, kCtrl, kRows, 0xf, false);
}
template <typename Op>
__device__ __forceinline__ uint32_t row_scan(uint32_t v, uint32_t neutral, Op op)  // inclusive, over each row of sixteen lanes
{
    v = op(v, dpp<0x111, 0xf>(neutral, v));  // row_shr 1, 2, 4, 8
    v = op(v, dpp<0x112, 0xf>(neutral, v));
    v = op(v, dpp<0x114, 0xf>(neutral, v));
    return op(v, dpp<0x118, 0xf>(neutral, v));
}
template <typename Op>
__device__ __forceinline__ uint32_t wave_scan(uint32_t v, uint32_t neutral, Op op)  // inclusive
{
    v = row_scan(v, neutral, op);
    v = op(v, dpp<0x142, 0xa>(neutral, v));  // row_bcast 15 into rows 1 and 3, 31 into rows 2 and 3
    return op(v, dpp<0x143, 0xc>(neutral, v));
}
__device__ __forceinline__ uint32_t wave_sum_scan(uint32_t v)
{
    return wave_scan(v, 0u, [](uint32_t a, uint32_t b) { return a + b; });
}
// The sum in every lane, and that of values below 2^50.  (Six exchanges through LDS, one behind the other, are 0.3 us where one
// wavefront has nothing else to do.)
__device__ __forceinline__ uint32_t wave_sum(uint32_t v) { return (uint32_t)__builtin_amdgcn_readlane((int)wave_sum_scan(v), 63); }
__device__ __forceinline__ uint64_t wave_sum(uint64_t v)
{
    return ((uint64_t)wave_sum((uint32_t)(v >> 24)) << 24) + (uint64_t)wave_sum((uint32_t)v & 0xFFFFFFu);
}

// Orders one wavefront's LDS writes before its later LDS reads (and the reverse).  The hardware executes a
// wavefront's LDS instructions in order; the fences (wavefront scope: no instructions) and the scheduling
// barrier keep the compiler from moving the accesses across this point.
__device__ __forceinline__ void wave_lds_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

int launch_fill_u32(uint32_t* p, size_t n, uint32_t v, hipStream_t s);

// Marks a header copy as complete (it may be host memory that a host thread watches): everything stored in it before is
// visible to whoever sees the mark.
__device__ __forceinline__ void mark_ready(gs355_header* copy)
{
    __hip_atomic_store(&copy->ready, 1u, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// tile-bucketed path
constexpr int kBinThreads = 1024;       // threads per binning workgroup
constexpr int kBinMaxGroups = 256;      // binning workgroups (each owns a contiguous slice of the Gaussians)
constexpr int kBinMaxTiles = 36000;     // counters of one workgroup that fit in LDS (4 B each)
constexpr int kCoarseShift = 4;         // the scatter's first level: bins of 16 consecutive tiles
constexpr int kCoarseTiles = 1 << kCoarseShift;
// up to kBinMaxTiles tiles a slice counts per tile; beyond, per coarse bin (tile totals counted from the bins)
constexpr int kBinMaxTilesWide = kBinMaxTiles * kCoarseTiles;
constexpr int kCoarseMaxGaussians = 1 << (32 - kCoarseShift);  // a coarse pair's index shares its word with the tile bits
int bin_groups(int32_t P, int* per_group);
// words of the slice matrix: [slices][tiles], or [slices][coarse bins] beyond kBinMaxTiles tiles
inline size_t bin_matrix_words(size_t tiles)
{
    const size_t columns = tiles <= (size_t)kBinMaxTiles ? tiles : (tiles + kCoarseTiles - 1) >> kCoarseShift;
    return (size_t)kBinMaxGroups * columns;
}
// tile_base: u32[2][tiles] (bases, then the scatter's cursors), then u64[ceil(tiles / 64)] (bases of blocks of 64 tiles),
// then u32[coarse bins + 1] (chunks of the second scatter level before each bin), u32[ceil(tiles / 64)] (buckets per larger
// sorter size class) and u32[tiles] (pairs per tile).  Beyond kBinMaxTiles tiles launch_tile_layout
// publishes the header and the coarse bins' bases only; ranges, lists and tile bases follow in launch_tile_scatter.
// per slice, and before it per 64 Gaussians (the preprocess's wavefronts): keys of the whole rectangles, Gaussians with a
// radius.  The frame's key count and its overflow go by the whole rectangles, so that a capacity that suffices for them
// suffices whatever the regions leave out.
struct SliceTotals {
    uint64_t keys;
    uint32_t visible, unused;
};
inline size_t wave_totals_count(int32_t P) { return ((size_t)P + 63) / 64; }
int launch_tile_count(const FrameArgs& f, int32_t P, const uint64_t* rects, const float* records, const uint2* wave_totals,
                      uint32_t* matrix, SliceTotals* slice_totals, hipStream_t s);
int launch_tile_layout(int32_t P, uint32_t* matrix, const SliceTotals* slice_totals, int tiles, uint32_t n_cap,
                       gs355_header* header, gs355_header* header_copy, uint32_t* tile_base, uint32_t* ranges, uint32_t* lists,
                       bool in_scatter, hipStream_t s);
// What a scatter that makes the layout itself (after launch_tile_layout with `in_scatter`) needs besides its own arguments.
struct ScatterLayout {
    const SliceTotals* slice_totals;
    gs355_header* header_copy;
};
// Pairs from which a frame scatters in two levels.  What decides is the order that the Gaussians are stored in, which the call does
// not say.  Whole frames at 1080p, two levels against one: slabs in random order 0.96 of the time at 3.7 to 5.7 Mi pairs, 0.94 at 7.6,
// 0.93 at 9.5; in Morton order, whose runs of neighbours the L2 merges by itself, 1.04 at all of these, in blocks of 20 m 1.03.  The
// line lies between.  Decoded Gaussians follow their anchors: 1.05 at 1.7 Mi pairs, 1.03 at 7.0, 1.02 at 9.4 (more not measured);
// where the caller has read their number they arrive as given ones.
inline uint32_t two_level_from(bool decoded) { return (decoded ? 12u : 6u) << 20; }
// `coarse`: a second buffer of the buckets' size (first level of the two-level scatter).  `levels`: 1 or 2 = that
// scatter whatever the frame holds, 0 = chosen on the device by the key count against `two_from` (both variants are launched); images
// beyond kBinMaxTiles tiles always take two levels.  `make`: NULL, or the layout is made on the way (up to kBinMaxTiles tiles)
int launch_tile_scatter(const FrameArgs& f, int32_t P, const uint64_t* rects, const float* records, const uint32_t* depth_bits,
                        gs355_header* header, const uint32_t* matrix, uint32_t n_cap,
                        uint32_t* tile_base, uint32_t* ranges, uint32_t* lists, uint64_t* buckets, uint64_t* coarse,
                        int levels, uint32_t two_from, const ScatterLayout* make, hipStream_t s);
// lists: u32[kListHeader + 8 * tiles]: the four class counts, four spare words, the four lists, then {u32 tile, first, last, 0}
// [tiles], the tiles by the length of their lists
constexpr int kListHeader = 8;
inline uint4* tile_order(uint32_t* lists, int tiles) { return reinterpret_cast<uint4*>(lists + kListHeader + 4 * (size_t)tiles); }
inline const uint4* tile_order(const uint32_t* lists, int tiles) { return tile_order(const_cast<uint32_t*>(lists), tiles); }
// The tile of a blend's workgroup and its list.
struct BlendTile {
    uint32_t tile, lo, hi;
    __device__ __forceinline__ BlendTile(const gs355_header* __restrict__ header, const uint32_t* __restrict__ ranges,
                                         const uint4* __restrict__ order)
    {
        // (all three requested together: one latency)
        const uint32_t b = blockIdx.x;
        const uint4 o = order[b];
        const uint2 r = reinterpret_cast<const uint2*>(ranges)[b];
        const bool ordered = header->ordered != 0u;
        tile = ordered ? o.x : b;
        lo = ordered ? o.y : r.x;
        hi = ordered ? o.z : r.y;
    }
};
int launch_tile_sort(gs355_header* header, int tiles, const uint32_t* ranges, uint32_t* lists,
                     uint64_t* buckets, uint64_t* out_keys, uint32_t* out_vals, bool keys_too, uint32_t skip_classes, hipStream_t s);

// anchor decode: argument checks, and the exclusive prefix of per-run (kept offsets, visible anchors) with the totals
int check_decoder(const gs355_decoder* dec, const gs355_anchors* an);
int launch_run_scan(const uint2* totals, uint2* base, uint32_t runs, uint32_t* num_emitted, uint32_t* num_visible,
                    hipStream_t s);

// row compaction by a byte mask (gs355_gather_rows); scratch: gather_scratch_words(P) words
size_t gather_scratch_words(int32_t P);
int launch_gather_rows(int32_t P, const uint8_t* mask, int32_t n_arrays, const gs355_gather_array* arrays,
                       uint32_t* count_out, uint32_t* scratch, hipStream_t s);

// generic exclusive scan of u32 (n <= 2^32-1); tmp needs scan_tmp_words(n) words
size_t scan_tmp_words(size_t n);
int launch_exclusive_scan(const uint32_t* in, uint32_t* out, size_t n, uint32_t* tmp, hipStream_t s);

#define GS355_CHECK_LAUNCH(what)                                                        \
    do {                                                                                \
        hipError_t e__ = hipGetLastError();                                             \
        if (e__ != hipSuccess) return set_error(GS355_EHIP, "%s: %s", what, hipGetErrorString(e__)); \
    } while (0)

}  // namespace gs355
