// Tile-bucketed sort for gfx950: the fast equivalent of "duplicate keys ->
// radix sort -> tile ranges" of the rasterizer behind
// GaussianRasterizer.forward (benchmarks/nerf/origin_gs/gs_model.py:211-220).
//
// The 64-bit key is (tile_id << 32 | depth bits).  Its high word is known when
// a pair is generated, so the most significant digit is resolved by counting:
// pairs are counted per tile, an exclusive scan of the counts gives every tile
// its slot range (these ARE the per-tile ranges), and pairs are scattered into
// their tile's bucket (in one level, or through coarse bins of 16 tiles when
// the frame holds many pairs).  What remains is an independent sort of each
// bucket by its low word, done by one workgroup per tile entirely in LDS (up
// to 10240 pairs in the 160 KB of a CU; larger buckets are split into such
// pieces first).  Bucket order after the scatter is arbitrary, so
// pairs are ordered by (depth bits, Gaussian index): exactly the order a
// stable sort of the emission-ordered keys produces.
//
// No workgroup waits on another; persistent loops run over fixed lists, or
// take entries from a counter until it passes the list's length.
#include <atomic>

#include "gs355_internal.h"

namespace gs355 {

namespace {

// whole rectangles of more tiles than this, and all regions with spans, are queued and expanded by a wavefront each (8 and 16
// measured slower, 64 and 128 the same)
constexpr int kInlineTiles = 32;
constexpr int kBinItems = 4;      // Gaussians per thread and round of the binning walk

// Gaussians per slice: at most kBinMaxGroups slices, in whole rounds of a workgroup for large frames, in whole wavefronts
// for small ones, so that a frame of a few thousand Gaussians is still spread over the chip.
__host__ __device__ __forceinline__ int slice_size(int P, int groups)
{
    const int per = (P + groups - 1) / groups, unit = per > kBinThreads / 2 ? kBinThreads : 64;
    const int whole = (per + unit - 1) / unit * unit;
    return whole < 64 ? 64 : whole;
}

// A slice of at most half a workgroup's threads gives each of its Gaussians 2, 4, 8 or 16 lanes, which take the tiles of
// its rectangle in turn: with a lane per Gaussian a slice of large splats is a chain of LDS requests as long as its
// largest rectangle, on the few compute units that a small frame's slices occupy.  10k Gaussians at 256x256 (26 tiles
// each): count 13.4 -> 4.7 us, scatter 29.0 -> 7.0 us.
__device__ __forceinline__ int lanes_per_gaussian(int per_group)
{
    int lanes = 1;
    while (lanes < 16 && 2 * lanes * per_group <= kBinThreads) lanes *= 2;
    return lanes;
}

// A share of a region's tiles for each of `lanes` lanes (a power of two), this one the `sub`-th; `record`: the Gaussian's.
// Of a region with spans a lane takes whole rows, or several lanes one where there are more lanes than rows: a row's span
// costs some 30 instructions, too many to evaluate for every tile (100k large splats: count 24.3, scatter 27.0 us by tile,
// 12.2 and 18.0 by row).
template <typename Visit>
__device__ __forceinline__ void walk_region(const TileRegion& q, const float* __restrict__ record, int sub, int lanes, int grid_x,
                                            Visit visit)
{
    if (q.spans) {
        const TileSpans s(record, q.x0, q.y0);
        const int rows = q.area / q.width;
        int share = lanes;  // lanes per row
        while (share > 1 && lanes < rows * share) share >>= 1;
        for (int row = sub / share; row < rows; row += lanes / share) {
            int first, end;
            s.columns(row, q.width, first, end);
            const int t = q.tile(row, 0, grid_x);
            for (int col = first + sub % share; col < end; col += share) visit(t + col);
        }
    } else {
        for (int e = sub; e < q.area; e += lanes) {
            int row, col;
            q.place(e, row, col);
            if (!q.masked || ((q.mask >> e) & 1u) != 0u) visit(q.tile(row, col, grid_x));
        }
    }
}

// The runs [ta, tb) of consecutive tiles of a masked or whole region, a row at a time (a row of a mask is one run: the
// ellipse is convex).
template <typename Visit>
__device__ __forceinline__ void walk_rows(const TileRegion& q, int grid_x, Visit visit)
{
    int t = q.y0 * grid_x + q.x0;
    if (q.masked) {
        const uint32_t row_bits = (1u << q.width) - 1u;
        for (uint32_t m = q.mask; m != 0u; m >>= q.width, t += grid_x) {
            const uint32_t row = m & row_bits;
            if (row != 0u) {
                const int first = t + __builtin_ctz(row);
                visit(first, first + __popc(row));
            }
        }
    } else {
        for (int e = 0; e < q.area; e += q.width, t += grid_x) visit(t, t + q.width);
    }
}

// ---------------------------------------------------------------------------
// Counting.  Workgroup c owns Gaussians [c * per_group, (c+1) * per_group) and a private array of counters in LDS.
//   up to kBinMaxTiles tiles:  one counter per tile; matrix[c][t] = pairs of this slice that fall in tile t.  No
//                              global atomic is issued anywhere on this path.
//   more tiles (kWide):        one counter per coarse bin of kCoarseTiles consecutive tiles, matrix[c][b]; the
//                              tiles' own totals are counted later, from the pairs of each bin (fine_count_kernel).
// A thread walks the tile rectangle of its own Gaussian; rectangles of more than kInlineTiles tiles are queued and
// walked by the wavefronts, one rectangle each at a time.
template <bool kWide>
__global__ __launch_bounds__(kBinThreads) void tile_count_kernel(FrameArgs f, int32_t P, int per_group,
                                                                 const uint64_t* __restrict__ rects,
                                                                 const float* __restrict__ records,
                                                                 const uint2* __restrict__ wave_totals, int n_totals,
                                                                 uint32_t* __restrict__ matrix,
                                                                 SliceTotals* __restrict__ slice_totals)
{
    extern __shared__ uint32_t s_count[];  // [tiles], or [coarse bins] when kWide
    __shared__ uint32_t s_queue[kBinItems * kBinThreads];
    __shared__ uint32_t s_nqueue, s_visible;
    __shared__ unsigned long long s_keys;

    if (f.p_device) {  // the slices follow the device-side count
        P = effective_count(f, P);
        per_group = slice_size(P, (int)gridDim.x);
        n_totals = (P + 63) / 64;
    }
    const int T = f.grid_x * f.grid_y;
    const int counters = kWide ? (T + kCoarseTiles - 1) >> kCoarseShift : T;
    const int tid = threadIdx.x, c = blockIdx.x;
    for (int t = tid; t < counters; t += kBinThreads) s_count[t] = 0u;
    if (tid == 0) {
        s_visible = 0;
        s_keys = 0;
        s_nqueue = 0;
    }
    // the workgroup's share of the preprocess's totals (any split serves: the layout adds the shares up), requested here and
    // added up behind the tiles
    const int share = (n_totals + (int)gridDim.x - 1) / (int)gridDim.x, share_end = min(n_totals, (c + 1) * share);
    const int share_first = c * share + tid;
    const uint2 total = share_first < share_end ? wave_totals[share_first] : make_uint2(0u, 0u);
    const int g_begin = min(P, c * per_group);
    const int g_end = min(P, g_begin + per_group);
    // a slice of few Gaussians: several lanes each, and a single round
    const int lanes = lanes_per_gaussian(per_group), only = g_begin + tid / lanes;
    const uint64_t only_rect = lanes > 1 && only < g_end ? rects[only] : 0ull;
    __syncthreads();
    auto add = [&](int t) { atomicAdd(&s_count[kWide ? t >> kCoarseShift : t], 1u); };
    // large rectangles: one per wavefront at a time, 64 tiles per step (the sixteen wavefronts work on sixteen
    // rectangles side by side; the whole workgroup on one rectangle left most of its threads idle)
    auto walk_queue = [&]() {
        const uint32_t nq = s_nqueue;
        uint32_t k = (uint32_t)tid >> 6;
        uint32_t gi = k < nq ? s_queue[k] : 0u;
        uint64_t next = k < nq ? rects[gi] : 0ull;
        while (k < nq) {
            const TileRegion q(next, f.plain_regions);
            const float* __restrict__ record = records + (size_t)gi * kRecordFloats;
            k += kBinThreads / 64;
            if (k < nq) {
                gi = s_queue[k];
                next = rects[gi];
            }
            walk_region(q, record, tid & 63, 64, f.grid_x, add);
        }
    };

    if (lanes > 1) {  // (uniform)
        const int sub = tid % lanes;
        if (only < g_end) {
            const TileRegion q(only_rect, f.plain_regions);
            if (q.area > kInlineTiles * lanes) {
                if (sub == 0) s_queue[atomicAdd(&s_nqueue, 1u)] = (uint32_t)only;
            } else {
                walk_region(q, records + (size_t)only * kRecordFloats, sub, lanes, f.grid_x, add);
            }
        }
        __syncthreads();
        walk_queue();
    } else {
        // a thread's Gaussians of a round: their rectangles are requested together, and those of the next round before
        // this round's are walked (a slice is a dozen rounds or more, each otherwise a memory latency plus its walk)
        uint64_t ahead[kBinItems];
#pragma unroll
        for (int u = 0; u < kBinItems; ++u) ahead[u] = g_begin < g_end ? rects[min(g_begin + u * kBinThreads + tid, g_end - 1)] : 0ull;
        for (int base = g_begin; base < g_end; base += kBinItems * kBinThreads) {
            if (tid == 0) s_nqueue = 0;
            __syncthreads();
            uint64_t rr[kBinItems];
#pragma unroll
            for (int u = 0; u < kBinItems; ++u) rr[u] = ahead[u];
            if (base + kBinItems * kBinThreads < g_end) {  // uniform
#pragma unroll
                for (int u = 0; u < kBinItems; ++u)
                    ahead[u] = rects[min(base + (kBinItems + u) * kBinThreads + tid, g_end - 1)];
            }
#pragma unroll
            for (int u = 0; u < kBinItems; ++u) {
                const int i = base + u * kBinThreads + tid;
                if (i < g_end) {
                    const TileRegion q(rr[u], f.plain_regions);
                    if (q.area > (q.spans ? 0 : kInlineTiles)) {
                        s_queue[atomicAdd(&s_nqueue, 1u)] = (uint32_t)i;
                    } else {
                        walk_rows(q, f.grid_x, [&](int ta, int tb) {
                            if (kWide) {  // one request per coarse bin the run crosses
                                while (ta < tb) {
                                    const int stop = min(tb, ((ta >> kCoarseShift) + 1) << kCoarseShift);
                                    atomicAdd(&s_count[ta >> kCoarseShift], (uint32_t)(stop - ta));
                                    ta = stop;
                                }
                            } else {
                                for (; ta < tb; ++ta) add(ta);
                            }
                        });
                    }
                }
            }
            __syncthreads();
            walk_queue();
            __syncthreads();
        }
    }
    if (share_first - (tid & 63) < share_end) {  // (uniform)
        uint64_t keys = total.x;
        uint32_t visible = total.y;
        for (int k = share_first + kBinThreads; k < share_end; k += kBinThreads) {
            const uint2 v = wave_totals[k];
            keys += v.x;
            visible += v.y;
        }
        keys = wave_sum(keys);
        visible = wave_sum(visible);
        if ((tid & 63) == 0) {
            atomicAdd(&s_keys, (unsigned long long)keys);
            atomicAdd(&s_visible, visible);
        }
    }
    __syncthreads();
    uint32_t* __restrict__ row = matrix + (size_t)c * counters;
    for (int t = tid; t < counters; t += kBinThreads) row[t] = s_count[t];
    if (tid == 0) slice_totals[c] = {(uint64_t)s_keys, s_visible, 0u};
}

// ---------------------------------------------------------------------------
// Scatter.  Writing every pair straight into its tile's bucket spreads a
// workgroup's stores over thousands of buckets: each 8-byte store then costs a
// whole 32-byte sector of memory traffic.  Frames of many pairs therefore take
// two levels: the pairs go first into coarse bins of kCoarseTiles consecutive
// tiles (a workgroup keeps a few hundred write streams going, which the L2
// merges into full lines), then workgroups read each bin back (contiguous)
// and spread it over the bin's 16 buckets in line-sized runs.  The coarse bin of
// tiles [16 b, 16 b + 16) is the concatenation of their buckets, so the same
// slot arithmetic serves both levels: a slice's pairs of bin b start at
// tile_base[16 b] plus the sum of the slice prefixes of the bin's tiles.  A
// coarse pair carries the tile's position within its bin in the low four bits
// of the index word.  The two launches of the second level cost some 40 us
// whatever the frame holds, so frames of few pairs (two_level_from) scatter
// in one level; the key count is only known on the device, so both variants
// are launched and each returns at once when the other one applies.

// Layout of the buckets inside the scatter (frames whose scatter follows the slice prefix in one call; tile_publish_kernel
// does the same in a launch of its own).  Every workgroup needs all tile bases anyway, and has them from the tiles' totals
// for two scans of a wavefront per 64 tiles; a block of 64 tiles is published (cursors, ranges, size-class lists) by one
// workgroup, the header by the first and the second level's work list by the last.  A launch of 256 threads for 256 tiles
// takes 4.4 us, most of it start and end.  Frames of 10k Gaussians at 256x256 47.5 -> 45.3 us, 130k 89.3 -> 85.4, 1M large
// splats 336 -> 329 and 6M 782 -> 773 at 1080p, 20M at 4K 1610 -> 1584 (with the first rectangles requested ahead of it, which is
// 2 us of the 130k frame).
struct LayoutArgs {
    const uint32_t* totals;       // [tiles]; NULL: the layout is there already
    const uint64_t* block_sums;   // [ceil(tiles / 64)]
    const uint32_t* block_classes;
    const SliceTotals* slice_totals;
    uint32_t n_cap;
    gs355_header* header;
    gs355_header* header_copy;
    uint32_t* ranges;
    uint32_t* lists;
    uint32_t* chunk_base;  // pairs per coarse bin, turned into chunks before each bin (for a second level in a later call too)
};

// The frame's header from sums over all blocks and slices (one thread).  `in_class`: buckets on the lists of the larger size
// classes, or NULL; `beyond`: those of the last that are larger than the LDS.
__device__ __forceinline__ void write_header(gs355_header* header, gs355_header* header_copy, uint64_t keys, uint32_t total,
                                             bool overflow, uint32_t n_cap, uint32_t visible, const uint32_t* in_class,
                                             uint32_t beyond)
{
    for (int k = 0; k < (header_copy ? 2 : 1); ++k) {
        gs355_header* const h = k ? header_copy : header;
        h->num_keys_total = keys;
        h->num_keys = overflow ? n_cap : total;
        h->overflow = overflow ? 1u : 0u;
        h->num_visible = visible;
        for (int c = 0; c < 3; ++c) h->sort_class_count[c] = in_class ? in_class[c] - (c == 2 ? beyond : 0u) : 0xFFFFFFFFu;
        h->sort_beyond_count = in_class ? beyond : 0xFFFFFFFFu;
        h->ordered = 0u;  // (until the tile sort has made the order)
    }
    if (header_copy) mark_ready(header_copy);
}

// A bucket's larger size class, or -1 (too small for the lists).
__device__ __forceinline__ int size_class(uint32_t n)
{
    if (n > (uint32_t)kTileSortCap[2]) return 2;  // (and what is larger than the LDS)
    if (n > (uint32_t)kTileSortCap[1]) return 1;
    return n > (uint32_t)kTileSortCap[0] ? 0 : -1;
}

constexpr uint32_t chunks_of(uint32_t pairs);

// Fills s_bin with this slice's first slot in each column and publishes the layout; returns the number of pairs, or
// 0xFFFFFFFF for a frame that overflowed.  `scratch`: kLayoutWords words of LDS, free again behind the next barrier.  `row`:
// what earlier slices put into each tile.
constexpr int kLayoutWords = 4 * kBinThreads;

template <int kShift>
__device__ __forceinline__ uint32_t lay_out(const LayoutArgs& a, int T, uint32_t* __restrict__ tile_base,
                                            const uint32_t* __restrict__ row, uint32_t* __restrict__ s_bin,
                                            uint32_t* __restrict__ scratch)
{
    static_assert((kBinMaxTiles + 63) / 64 <= kBinThreads && kBinMaxTiles < (1 << 16), "a block per thread, 16 bits a class");
    static_assert(kBinMaxGroups <= kBinThreads, "a slice per thread");
    constexpr int kWavesHere = kBinThreads / 64;
    uint32_t* const s_block = scratch;                    // pairs before each block of 64 tiles
    uint32_t* const s_classes = scratch + kBinThreads;    // buckets of classes 0 and 1 before it (16 bits each)
    uint32_t* const s_class2 = scratch + 2 * kBinThreads;
    uint32_t* const s_waves = scratch + 3 * kBinThreads;  // per wavefront: these three, visible Gaussians, keys
    constexpr int kSums = 6;
    static_assert(3 * kBinThreads + (kSums + 1) * kWavesHere <= kLayoutWords, "and the chunks' sums");
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int n_blocks = (T + 63) / 64;
    // (the first block's values are under way while the sums are made)
    const int t_first = wave * 64 + lane;
    uint32_t next_total = t_first < T ? a.totals[t_first] : 0u, next_before = t_first < T ? row[t_first] : 0u;
    const int bins = (T + kCoarseTiles - 1) >> kCoarseShift;
    constexpr int kBinsEach = ((kBinMaxTiles >> kCoarseShift) + kBinThreads) / kBinThreads;  // coarse bins per thread of the last workgroup
    const bool last = blockIdx.x == gridDim.x - 1;
    uint32_t bin_chunks[kBinsEach] = {};
    if (last)
#pragma unroll
        for (int k = 0; k < kBinsEach; ++k)
            if (kBinsEach * tid + k < bins) bin_chunks[k] = chunks_of(a.chunk_base[kBinsEach * tid + k]);
    const uint32_t pairs = tid < n_blocks ? (uint32_t)a.block_sums[tid] : 0u;  // (beyond 2^32 pairs the frame overflows)
    const uint32_t word = tid < n_blocks ? a.block_classes[tid] : 0u;
    SliceTotals slice = {0ull, 0u, 0u};
    if (tid < (int)gridDim.x) slice = a.slice_totals[tid];
    // (16 bits each: classes 0 and 1; class 2 and those of it beyond the LDS)
    const uint32_t two = (word & 0xFFu) | ((word & 0xFF00u) << 8), third = ((word >> 16) & 0xFFu) | ((word >> 24) << 16);
    const uint32_t pairs_inc = wave_sum_scan(pairs), two_inc = wave_sum_scan(two), third_inc = wave_sum_scan(third);
    // (keys below 2^50, as two sums: 24 bits and the rest)
    const uint32_t sums[kSums] = {pairs_inc, two_inc, third_inc, wave_sum_scan(slice.visible),
                                  wave_sum_scan((uint32_t)slice.keys & 0xFFFFFFu), wave_sum_scan((uint32_t)(slice.keys >> 24))};
    if (lane == 63) {
#pragma unroll
        for (int k = 0; k < kSums; ++k) s_waves[kWavesHere * k + wave] = sums[k];
    }
    __syncthreads();
    uint32_t before[3], all[kSums];  // over the wavefronts, a lane each
#pragma unroll
    for (int k = 0; k < kSums; ++k) {
        static_assert(kWavesHere == 16, "a row of lanes");
        const uint32_t inc = row_scan(s_waves[kWavesHere * k + (lane & 15)], 0u, [](uint32_t x, uint32_t y) { return x + y; });
        all[k] = (uint32_t)__builtin_amdgcn_readlane((int)inc, 15);
        if (k < 3) before[k] = wave ? (uint32_t)__builtin_amdgcn_readlane((int)inc, wave - 1) : 0u;
    }
    const uint64_t keys = ((uint64_t)all[5] << 24) + all[4];  // of whole rectangles: at least the pairs
    if (tid < n_blocks) {
        s_block[tid] = before[0] + pairs_inc - pairs;
        s_classes[tid] = before[1] + two_inc - two;
        s_class2[tid] = (before[2] + third_inc - third) & 0xFFFFu;
    }
    const bool overflow = keys > (uint64_t)a.n_cap;
    if (blockIdx.x == 0 && tid == 0) {
        const uint32_t in_class[3] = {all[1] & 0xFFFFu, all[1] >> 16, all[2] & 0xFFFFu};
        write_header(a.header, a.header_copy, keys, all[0], overflow, a.n_cap, all[3], in_class, all[2] >> 16);
        for (int c = 0; c < 3; ++c) a.lists[c] = in_class[c];
    }
    if (overflow) return 0xFFFFFFFFu;  // later stages do nothing either
    __syncthreads();
    for (int b = wave; b < n_blocks; b += kWavesHere) {  // (uniform per wavefront)
        const int t = b * 64 + lane, t_next = t + kBinThreads;
        const uint32_t v = next_total, earlier = next_before;
        if (b + kWavesHere < n_blocks) {
            next_total = t_next < T ? a.totals[t_next] : 0u;
            next_before = t_next < T ? row[t_next] : 0u;
        }
        const uint32_t end = s_block[b] + wave_sum_scan(v), first = end - v;
        if (kShift == 0) {
            if (t < T) s_bin[t] = first + earlier;
        } else {  // a column is a row of sixteen lanes
            static_assert(kShift == 0 || kCoarseTiles == 16, "a row of lanes");
            auto add = [](uint32_t x, uint32_t y) { return x + y; };
            const uint32_t start = end - row_scan(v, 0u, add), sum = row_scan(earlier, 0u, add);  // (in the row's last lane)
            if ((lane & 15) == 15 && (t & ~15) < T) s_bin[t >> kCoarseShift] = start + sum;
        }
        if ((uint32_t)b % gridDim.x != blockIdx.x) continue;
        if (t < T) {
            tile_base[t] = first;
            tile_base[T + t] = first;  // the bucket's next free slot during the second level
            a.ranges[2 * t] = v ? first : 0u;
            a.ranges[2 * t + 1] = v ? end : 0u;
        }
        const int cls = size_class(v);
        const uint32_t at[3] = {s_classes[b] & 0xFFFFu, s_classes[b] >> 16, s_class2[b]};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            const uint64_t m = __ballot(cls == c);
            if (cls == c) a.lists[kListHeader + (size_t)c * T + lanes_below_in(m, at[c])] = (uint32_t)t;
        }
    }
    if (last) {  // (each element was read by the thread that overwrites it)
        uint32_t chunks = 0;
#pragma unroll
        for (int k = 0; k < kBinsEach; ++k) chunks += bin_chunks[k];
        const uint32_t inc = wave_sum_scan(chunks);
        if (lane == 63) s_waves[kSums * kWavesHere + wave] = inc;
        __syncthreads();
        uint32_t run = inc - chunks;
        for (int w = 0; w < wave; ++w) run += s_waves[kSums * kWavesHere + w];
#pragma unroll
        for (int k = 0; k < kBinsEach; ++k) {
            if (kBinsEach * tid + k < bins) a.chunk_base[kBinsEach * tid + k] = run;
            run += bin_chunks[k];
        }
        if (tid == kBinThreads - 1) a.chunk_base[bins] = run;
    }
    return all[0];
}

// The walk of the counting kernel with one cursor per column: a coarse bin (kShift = kCoarseShift) or a tile
// (kShift = 0, straight into the buckets).  The tiles of one rectangle row are consecutive, so a row takes one slot
// request per coarse bin it crosses instead of one per tile.  Runs only when min_keys <= pairs of the frame <
// max_keys.  (Two variants were measured slower: staging each round in LDS ordered by bin, so that consecutive
// lanes store consecutive pairs, walks the rectangles twice; walking a thread's rectangles side by side to keep
// several slot requests in flight costs more in bookkeeping than the latency it hides.)
template <int kShift, bool kWide>
__global__ __launch_bounds__(kBinThreads) void scatter_kernel(FrameArgs f, int32_t P, int per_group,
                                                              const uint64_t* __restrict__ rects,
                                                              const float* __restrict__ records,
                                                              const uint32_t* __restrict__ depth_bits,
                                                              const gs355_header* header,
                                                              uint32_t min_keys, uint32_t max_keys,
                                                              const uint32_t* __restrict__ matrix,
                                                              uint32_t* bases,
                                                              uint64_t* __restrict__ dst, LayoutArgs layout)
{
    static_assert(!kWide || kShift > 0, "beyond kBinMaxTiles tiles only coarse bins fit in LDS");
    extern __shared__ uint32_t s_bin[];  // [columns] next free slot of this slice in each column
    __shared__ uint32_t s_queue[kBinItems * kBinThreads];
    static_assert(kBinItems * kBinThreads >= kLayoutWords, "the layout is made in the queue's memory");
    __shared__ uint32_t s_nqueue;

    constexpr int kSpan = 1 << kShift;
    const int T = f.grid_x * f.grid_y, bins = (T + kSpan - 1) >> kShift;
    const int tid = threadIdx.x, c = blockIdx.x, wave = tid >> 6, lane = tid & 63;
    // a column's first slot for this slice: the column's base (kWide: bases[b]; else the base of its first tile)
    // plus what the earlier slices put into it (the matrix holds that per bin when kWide, else per tile)
    const uint32_t* __restrict__ row = matrix + (size_t)c * (kWide ? bins : T);
    if (f.p_device) {
        P = effective_count(f, P);
        per_group = slice_size(P, (int)gridDim.x);
    }
    const int g_begin = min(P, c * per_group);
    const int g_end = min(P, g_begin + per_group);
    // the first round's rectangles and depths, under way while the layout is made
    const int lanes = lanes_per_gaussian(per_group);
    uint64_t rr[kBinItems] = {};
    uint32_t depths[kBinItems] = {};
    auto request = [&](int first) {
#pragma unroll
        for (int u = 0; u < kBinItems; ++u) {
            const int i = min(first + u * kBinThreads + tid, g_end - 1);
            rr[u] = rects[i];
            depths[u] = depth_bits[i];
        }
    };
    if (g_begin < g_end) {  // (uniform)
        if (lanes > 1) {
            const int i = min(g_begin + tid / lanes, g_end - 1);
            rr[0] = rects[i];
            depths[0] = depth_bits[i];
        } else {
            request(g_begin);
        }
    }
    if (!kWide && layout.totals) {  // (uniform)
        const uint32_t keys = lay_out<kShift>(layout, T, bases, row, s_bin, s_queue);
        if (keys == 0xFFFFFFFFu || keys < min_keys || keys >= max_keys) return;
    } else {
        if (header->overflow || header->num_keys < min_keys || header->num_keys >= max_keys) return;
        for (int b = tid; b < bins; b += kBinThreads)
            s_bin[b] = kWide ? bases[b] + row[b] : kShift ? bases[b << kShift] : bases[b] + row[b];
        if (!kWide && kShift) {
            __syncthreads();
            for (int t = tid; t < T; t += kBinThreads) {
                const uint32_t before = row[t];
                if (before) atomicAdd(&s_bin[t >> kShift], before);
            }
        }
    }
    // the tiles [ta, tb) of one rectangle row, cut where they cross into the next column
    auto emit_row = [&](int ta, int tb, uint64_t payload) {
        while (ta < tb) {
            const int stop = min(tb, ((ta >> kShift) + 1) << kShift);
            uint32_t slot = atomicAdd(&s_bin[ta >> kShift], (uint32_t)(stop - ta));
            // the segment's slots are consecutive: two pairs per 16-byte store where the slot is even (every store
            // is a 64-byte request on the way to the L2, however few bytes it carries)
            if ((slot & 1u) && ta < stop) dst[slot++] = payload | (uint64_t)(ta++ & (kSpan - 1));
            for (; ta + 1 < stop; ta += 2, slot += 2) {
                ulonglong2 two;
                two.x = payload | (uint64_t)(ta & (kSpan - 1));
                two.y = payload | (uint64_t)((ta + 1) & (kSpan - 1));
                *reinterpret_cast<ulonglong2*>(dst + slot) = two;
            }
            if (ta < stop) dst[slot] = payload | (uint64_t)(ta++ & (kSpan - 1));
        }
    };

    auto emit_tile = [&](int t, uint64_t payload) {
        dst[atomicAdd(&s_bin[t >> kShift], 1u)] = payload | (uint64_t)(t & (kSpan - 1));
    };
    auto payload_of = [&](uint32_t depth, uint32_t i) { return ((uint64_t)depth << 32) | ((uint64_t)i << kShift); };
    // large rectangles: one per wavefront at a time, 64 tiles per step
    auto walk_queue = [&]() {
        const uint32_t nq = s_nqueue;
        uint32_t k = wave, gi = k < nq ? s_queue[k] : 0u, depth = k < nq ? depth_bits[gi] : 0u;
        uint64_t next = k < nq ? rects[gi] : 0ull;
        while (k < nq) {
            const TileRegion q(next, f.plain_regions);
            const float* __restrict__ record = records + (size_t)gi * kRecordFloats;
            const uint64_t payload = payload_of(depth, gi);
            k += kBinThreads / 64;
            if (k < nq) {
                gi = s_queue[k];
                next = rects[gi];
                depth = depth_bits[gi];
            }
            walk_region(q, record, lane, 64, f.grid_x, [&](int t) { emit_tile(t, payload); });
        }
    };
    if (lanes > 1) {  // (uniform; a single round, as in the count)
        if (tid == 0) s_nqueue = 0;
        __syncthreads();
        const int i = g_begin + tid / lanes, sub = tid % lanes;
        if (i < g_end) {
            const TileRegion q(rr[0], f.plain_regions);
            const uint64_t payload = payload_of(depths[0], (uint32_t)i);
            if (q.area > kInlineTiles * lanes) {
                if (sub == 0) s_queue[atomicAdd(&s_nqueue, 1u)] = (uint32_t)i;
            } else {
                walk_region(q, records + (size_t)i * kRecordFloats, sub, lanes, f.grid_x,
                            [&](int t) { emit_tile(t, payload); });
            }
        }
        __syncthreads();
        walk_queue();
        return;
    }

    for (int first = g_begin; first < g_end; first += kBinItems * kBinThreads) {
        if (tid == 0) s_nqueue = 0;
        __syncthreads();
        // (requested a round ahead, as in the count, they are awaited together with the stores in between: 6M Gaussians +6 us)
        if (first != g_begin) request(first);
#pragma unroll
        for (int u = 0; u < kBinItems; ++u) {
            const int i = first + u * kBinThreads + tid;
            if (i < g_end) {
                const TileRegion q(rr[u], f.plain_regions);
                if (q.area > (q.spans ? 0 : kInlineTiles)) {
                    s_queue[atomicAdd(&s_nqueue, 1u)] = (uint32_t)i;
                } else {
                    const uint64_t payload = payload_of(depths[u], (uint32_t)i);
                    walk_rows(q, f.grid_x, [&](int ta, int tb) { emit_row(ta, tb, payload); });
                }
            }
        }
        __syncthreads();
        walk_queue();
        __syncthreads();
    }
}

// Second level: the pairs of a coarse bin (contiguous) go to the buckets of the bin's tiles, a chunk of kFineChunk pairs
// at a time.  Chunks never cross a bin; chunk_base[b] = chunks of the bins before b, chunk_base[bins] = all of them
// (made with the layout).  The kFineGrid workgroups take equal, contiguous runs of chunks, so every workgroup has work
// however the pairs are spread over the bins, and a bin of many pairs is shared by many workgroups.  A chunk is split
// by tile inside LDS first (wave-level ranking by the four tile bits, a scan over the per-wave counts), the
// workgroup reserves a run of slots per bucket with one global atomic each, and consecutive lanes then store
// consecutive pairs of one bucket: full-line writes instead of one memory transaction per pair.  Order inside a
// bucket is arbitrary, as the sort expects.
constexpr int kFineThreads = 256;
constexpr int kFineWaves = kFineThreads / 64;
constexpr int kFineItems = 8;                             // pairs per thread and chunk
constexpr int kFineChunk = kFineThreads * kFineItems;  // 2048 pairs = 16 KB of LDS
constexpr uint32_t chunks_of(uint32_t pairs) { return (pairs + (uint32_t)kFineChunk - 1u) / (uint32_t)kFineChunk; }
constexpr int kFineGrid = 8192;                          // a chunk per workgroup at 6M Gaussians / 1080p, a few each at 4K

// A workgroup's run of chunks.  next() gives the following chunk's bin, first pair and pair count.
struct ChunkRun {
    const uint32_t* chunk_base;
    uint32_t c, c_end;  // next chunk, end of the run
    int b, bins;        // bin of chunk c (once begun)

    __device__ ChunkRun(const uint32_t* __restrict__ base, int n_bins) : chunk_base(base), b(0), bins(n_bins)
    {
        const uint32_t total = base[n_bins], per = (total + gridDim.x - 1) / gridDim.x;
        c = min(total, blockIdx.x * per);
        c_end = min(total, c + per);
        if (c < c_end) {  // the bin that holds chunk c: the last one whose base is <= c
            int lo = 0, hi = n_bins;  // base[lo] <= c < base[hi]
            while (hi - lo > 1) {
                const int mid = (lo + hi) >> 1;
                if (base[mid] <= c) lo = mid;
                else hi = mid;
            }
            b = lo;
        }
    }
    // `first_pair(bin)`: where the bin's pairs start in the coarse buffer
    template <typename First>
    __device__ bool next(First first_pair, uint32_t num_keys, int& bin, uint32_t& j0, uint32_t& n, uint32_t& bin_begin,
                         uint32_t& bin_end)
    {
        if (c >= c_end) return false;
        while (chunk_base[b + 1] <= c) ++b;  // (bins without pairs have no chunks)
        bin = b;
        bin_begin = first_pair(b);
        bin_end = b + 1 < bins ? first_pair(b + 1) : num_keys;
        j0 = bin_begin + (c - chunk_base[b]) * (uint32_t)kFineChunk;
        n = min((uint32_t)kFineChunk, bin_end - j0);
        ++c;
        return true;
    }
};

// A chunk is a chain of steps with a barrier between each two: the tiles' totals, their prefix and the request for slots are
// one of them (the prefix by exchanges through LDS in a step of its own, the slots awaited before the staging: 26.6 -> 25.0 us
// at 1M large splats, 34.5 -> 33.2 at 6M, 62.8 -> 59.9 at 20M and 4K).
__global__ __launch_bounds__(kFineThreads) void fine_scatter_kernel(const gs355_header* __restrict__ header,
                                                                    uint32_t min_keys,
                                                                    const uint32_t* __restrict__ tile_base,
                                                                    uint32_t* __restrict__ cursor, int T,
                                                                    const uint32_t* __restrict__ chunk_base,
                                                                    const uint64_t* __restrict__ coarse,
                                                                    uint64_t* __restrict__ buckets)
{
    __shared__ uint64_t s_stage[kFineChunk];
    __shared__ uint32_t s_count[kFineWaves][kCoarseTiles];  // pairs per (wavefront, tile) of the chunk, then their offsets
    __shared__ uint32_t s_start[kCoarseTiles + 1];          // first staged position of each tile's pairs
    __shared__ uint32_t s_slot[kCoarseTiles];               // first reserved slot of each bucket for this chunk
    if (header->overflow || header->num_keys < min_keys) return;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const uint64_t lanes_below = (1ull << lane) - 1ull;
    const uint32_t num_keys = header->num_keys;
    ChunkRun run(chunk_base, (T + kCoarseTiles - 1) >> kCoarseShift);
    int bin;
    uint32_t j0, n, begin, end;
    while (run.next([&](int b) { return tile_base[b << kCoarseShift]; }, num_keys, bin, j0, n, begin, end)) {
        const int t0 = bin << kCoarseShift;
        for (int k = tid; k < kFineWaves * kCoarseTiles; k += kFineThreads) (&s_count[0][0])[k] = 0;
        __syncthreads();
        // a wavefront owns kFineItems x 64 consecutive pairs of the chunk
        uint64_t v[kFineItems];
        uint32_t rank[kFineItems];
#pragma unroll
        for (int u = 0; u < kFineItems; ++u) {
            const uint32_t p = (uint32_t)(wave * kFineItems + u) * 64u + lane;
            v[u] = p < n ? coarse[j0 + p] : 0ull;
        }
#pragma unroll
        for (int u = 0; u < kFineItems; ++u) {
            const uint32_t p = (uint32_t)(wave * kFineItems + u) * 64u + lane;
            const bool valid = p < n;
            const uint32_t d = (uint32_t)v[u] & (kCoarseTiles - 1);
            uint64_t peers = __ballot(valid);
#pragma unroll
            for (int bit = 0; bit < kCoarseShift; ++bit) {
                const bool one = (d >> bit) & 1u;
                const uint64_t m = __ballot(one);
                peers &= one ? m : ~m;
            }
            uint32_t before = 0;
            if (valid) {
                const int leader = __ffsll((unsigned long long)peers) - 1;
                if (lane == leader) before = atomicAdd(&s_count[wave][d], (uint32_t)__popcll(peers));
                before = __shfl(before, leader, 64);
            }
            rank[u] = before + (uint32_t)__popcll(peers & lanes_below);
        }
        __syncthreads();
        uint32_t slot = 0;
        if (tid < kCoarseTiles) {  // per tile: its total in the chunk, where its pairs are staged, and the slots it gets in its bucket
            uint32_t total = 0;
#pragma unroll
            for (int w = 0; w < kFineWaves; ++w) {
                const uint32_t c = s_count[w][tid];
                s_count[w][tid] = total;  // pairs of this tile in earlier wavefronts
                total += c;
            }
            static_assert(kCoarseTiles == 16, "a row of lanes");
            const uint32_t inc = row_scan(total, 0u, [](uint32_t x, uint32_t y) { return x + y; });
            s_start[tid] = inc - total;
            if (tid == kCoarseTiles - 1) s_start[kCoarseTiles] = inc;
            if (total && t0 + tid < T) slot = atomicAdd(&cursor[t0 + tid], total);  // (under way while the pairs are staged)
        }
        __syncthreads();
#pragma unroll
        for (int u = 0; u < kFineItems; ++u) {
            const uint32_t p = (uint32_t)(wave * kFineItems + u) * 64u + lane;
            if (p < n) {
                const uint32_t d = (uint32_t)v[u] & (kCoarseTiles - 1);
                s_stage[s_start[d] + s_count[wave][d] + rank[u]] = v[u];
            }
        }
        if (tid < kCoarseTiles) s_slot[tid] = slot;
        __syncthreads();
        for (uint32_t p = tid; p < n; p += kFineThreads) {
            const uint64_t pair = s_stage[p];
            const uint32_t low = (uint32_t)pair, d = low & (kCoarseTiles - 1);
            const uint32_t slot = s_slot[d] + (p - s_start[d]);
            // (a slot outside the bin cannot happen with pairs the coarse level wrote; the test keeps corrupted input
            // from reaching other memory)
            if (slot >= begin && slot < end) buckets[slot] = (pair & 0xFFFFFFFF00000000ull) | (uint64_t)(low >> kCoarseShift);
        }
        __syncthreads();
    }
}

// Pairs per tile, counted from the coarse bins (images of more tiles than a slice can count in LDS): the chunks of
// the fine scatter, a wavefront-level count by the four tile bits, one global atomic per tile and chunk.
// `bin_base` [bins]: first pair of each bin; `totals` [T] and `block_sums` [T / 64] (pairs per 64 tiles) cleared
// beforehand.
__global__ __launch_bounds__(kFineThreads) void fine_count_kernel(const gs355_header* __restrict__ header,
                                                                  const uint32_t* __restrict__ bin_base, int bins,
                                                                  int T, const uint32_t* __restrict__ chunk_base,
                                                                  const uint64_t* __restrict__ coarse,
                                                                  uint32_t* __restrict__ totals,
                                                                  uint64_t* __restrict__ block_sums,
                                                                  uint32_t* __restrict__ list_counts)
{
    __shared__ uint32_t s_count[kCoarseTiles];
    if (blockIdx.x == 0 && threadIdx.x < 4) list_counts[threadIdx.x] = 0u;  // filled with the layout
    if (header->overflow) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const uint32_t num_keys = header->num_keys;
    ChunkRun run(chunk_base, bins);
    int bin;
    uint32_t j0, n, begin, end;
    while (run.next([&](int b) { return bin_base[b]; }, num_keys, bin, j0, n, begin, end)) {
        const int t0 = bin << kCoarseShift;
        if (tid < kCoarseTiles) s_count[tid] = 0;
        __syncthreads();
        uint64_t v[kFineItems];
#pragma unroll
        for (int u = 0; u < kFineItems; ++u) {
            const uint32_t p = (uint32_t)(u * kFineThreads + tid);
            v[u] = p < n ? coarse[j0 + p] : 0ull;
        }
#pragma unroll
        for (int u = 0; u < kFineItems; ++u) {
            const bool valid = (uint32_t)(u * kFineThreads + tid) < n;
            const uint32_t d = (uint32_t)v[u] & (kCoarseTiles - 1);
            uint64_t peers = __ballot(valid);
#pragma unroll
            for (int bit = 0; bit < kCoarseShift; ++bit) {
                const bool one = (d >> bit) & 1u;
                const uint64_t m = __ballot(one);
                peers &= one ? m : ~m;
            }
            if (valid && lane == __ffsll((unsigned long long)peers) - 1) atomicAdd(&s_count[d], (uint32_t)__popcll(peers));
        }
        __syncthreads();
        if (tid < kCoarseTiles && t0 + tid < T && s_count[tid]) {
            atomicAdd(&totals[t0 + tid], s_count[tid]);
            atomicAdd(reinterpret_cast<unsigned long long*>(&block_sums[(t0 + tid) >> 6]), (unsigned long long)s_count[tid]);
        }
        __syncthreads();
    }
}

// Exclusive prefix of every tile's counts over the slices (in place), the
// tile's total and the total of the workgroup's tiles.  A workgroup covers 64 tiles; its sixteen wavefronts take a
// sixteenth of the slices each, all requested at once and kept in registers, exchange their sums through LDS and write the
// prefixes shifted by the wavefronts' before them.  (Four wavefronts that read their quarter twice, sixteen slices at a
// time, were a chain of eight memory latencies: 9.7 us for 1700 tiles, as many as for 8160.)
constexpr int kPrefixParts = 16;
constexpr int kPrefixRows = kBinMaxGroups / kPrefixParts;
__global__ __launch_bounds__(64 * kPrefixParts) void slice_prefix_kernel(uint32_t* __restrict__ matrix, int groups, int tiles,
                                                                         uint32_t* __restrict__ totals,
                                                                         uint64_t* __restrict__ block_sums,
                                                                         uint32_t* __restrict__ bin_sums,
                                                                         uint32_t* __restrict__ block_classes,
                                                                         uint32_t* __restrict__ list_counts)
{
    __shared__ uint32_t s_part[kPrefixParts][64];
    if (blockIdx.x == 0 && threadIdx.x < 4) list_counts[threadIdx.x] = 0u;  // filled with the layout
    const int lane = threadIdx.x & 63, part = threadIdx.x >> 6;
    const int t = blockIdx.x * 64 + lane;
    const int per = (groups + kPrefixParts - 1) / kPrefixParts;  // <= kPrefixRows
    const int c0 = min(part * per, groups), rows = min(per, groups - c0);
    const bool live = t < tiles;
    uint32_t* __restrict__ column = matrix + (size_t)c0 * tiles + t;
    uint32_t v[kPrefixRows], sum = 0;
#pragma unroll
    for (int k = 0; k < kPrefixRows; ++k) v[k] = live && k < rows ? column[(size_t)k * tiles] : 0u;
#pragma unroll
    for (int k = 0; k < kPrefixRows; ++k) sum += v[k];
    s_part[part][lane] = sum;
    __syncthreads();
    uint32_t run = 0, total = 0;
#pragma unroll
    for (int p = 0; p < kPrefixParts; ++p) {
        const uint32_t n = s_part[p][lane];
        if (p < part) run += n;
        total += n;
    }
#pragma unroll
    for (int k = 0; k < kPrefixRows; ++k) {
        if (live && k < rows) column[(size_t)k * tiles] = run;
        run += v[k];
    }
    if (part == 0) {
        if (live) totals[t] = total;
        const uint64_t sum64 = wave_sum((uint64_t)(live ? total : 0u));  // the 64 tiles of this workgroup are one block of the layout's scan
        if (lane == 0) block_sums[blockIdx.x] = sum64;
        if (block_classes) {  // columns are tiles: how many of the 64 fall in each larger sorter size class, a byte each
            const uint32_t v = live ? total : 0u;
            const uint32_t n1 = (uint32_t)__popcll(__ballot(v > (uint32_t)kTileSortCap[0] && v <= (uint32_t)kTileSortCap[1]));
            const uint32_t n2 = (uint32_t)__popcll(__ballot(v > (uint32_t)kTileSortCap[1] && v <= (uint32_t)kTileSortCap[2]));
            const uint32_t n3 = (uint32_t)__popcll(__ballot(v > (uint32_t)kTileSortCap[2]));
            const uint32_t beyond = (uint32_t)__popcll(__ballot(v > (uint32_t)kTileSortCap[3]));  // (of them)
            if (lane == 0) block_classes[blockIdx.x] = n1 | (n2 << 8) | (n3 << 16) | (beyond << 24);
        }
        if (bin_sums) {  // columns are tiles: the pairs of each coarse bin (kCoarseTiles consecutive tiles)
            uint32_t bin = live ? total : 0u;
#pragma unroll
            for (int d = 1; d < kCoarseTiles; d <<= 1) bin += __shfl_xor(bin, d, 64);
            if ((lane & (kCoarseTiles - 1)) == 0 && live) bin_sums[t >> kCoarseShift] = bin;
        }
    }
}

// Layout of the buckets from the tiles' totals: one wavefront per block of 64 tiles, four per workgroup.  Every
// workgroup adds up the block totals itself (a few hundred words, at most 9000): those before its own blocks give its
// first slot, all of them the number of pairs; the slices' totals are the frame's key count, which decides overflow before
// anything is published — so no workgroup waits for another and no separate scan pass is launched.  Workgroup 0 also
// writes the frame header and the work list of the scatter's second level: chunk_base[b] = chunks of kFineChunk pairs in
// the coarse bins before b, chunk_base[bins] = all (`bin_pairs`, the pairs per bin, may be the same array).  With
// kTiles the wavefronts publish tile bases, the scatter's cursors, the ranges and the lists of buckets too large for the
// small sorter; without, the columns are coarse bins and only their bases are written.  Where the buckets per size class were counted
// by block (`block_classes`, a byte per class), a block's places in the lists follow from the blocks before it, as its
// slots do; else they are requested from the lists' counters (`lists[0..3]` cleared by an earlier kernel), which costs
// three dependent round trips to memory (9.1 us at 1080p against 5.1).  `totals` and `tile_base` may be the same array.
// `header_known`: second layout of a frame (by tile, after the one by coarse bin): the header stands, and nothing is done
// on overflow.
template <bool kTiles>
__global__ __launch_bounds__(256) void tile_publish_kernel(const uint32_t* totals, uint32_t tiles,
                                                           const uint64_t* __restrict__ block_sums, uint32_t n_blocks,
                                                           const SliceTotals* __restrict__ slice_totals, int groups,
                                                           uint32_t n_cap, gs355_header* __restrict__ header,
                                                           gs355_header* __restrict__ header_copy, bool header_known,
                                                           uint32_t* tile_base,
                                                           uint32_t* __restrict__ ranges, uint32_t* __restrict__ lists,
                                                           const uint32_t* bin_pairs, int bins, uint32_t* chunk_base,
                                                           const uint32_t* __restrict__ block_classes)
{
    __shared__ uint64_t s_before[4], s_total[4], s_class_before[4], s_class_total[4], s_keys[4];
    __shared__ uint32_t s_vis[4], s_chunks[4];
    if (header_known && header->overflow) return;
    // counts of the three classes and of what is beyond the LDS, 16 bits each
    static_assert(kBinMaxTiles < (1 << 16), "(columns that are tiles)");
    auto classes_of = [&](uint32_t b) {
        const uint32_t w = block_classes[b];
        return (uint64_t)((w & 0xFFu) | ((w & 0xFF00u) << 8)) | ((uint64_t)(((w >> 16) & 0xFFu) | ((w >> 24) << 16)) << 32);
    };
    auto class_count = [](uint64_t packed, int c) { return (uint32_t)(packed >> (16 * c)) & 0xFFFFu; };
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const uint32_t first_block = blockIdx.x * 4u, block = first_block + (uint32_t)wave;
    {
        uint64_t before = 0, total = 0, class_before = 0, class_total = 0;
        for (uint32_t b = threadIdx.x; b < n_blocks; b += 256u) {
            const uint64_t v = block_sums[b];
            total += v;
            before += b < first_block ? v : 0ull;
            if (block_classes) {
                const uint64_t w = classes_of(b);
                class_total += w;
                class_before += b < first_block ? w : 0ull;
            }
        }
        uint32_t vis = 0;
        uint64_t keys = 0;
        if (!header_known) {
            for (int c = threadIdx.x; c < groups; c += 256) {
                const SliceTotals v = slice_totals[c];
                vis += v.visible;
                keys += v.keys;
            }
        }
        before = wave_sum(before);
        total = wave_sum(total);
        vis = wave_sum(vis);
        keys = wave_sum(keys);
        auto sum_classes = [](uint64_t v) { return ((uint64_t)wave_sum((uint32_t)(v >> 32)) << 32) | wave_sum((uint32_t)v); };
        class_before = sum_classes(class_before);
        class_total = sum_classes(class_total);
        if (lane == 0) {
            s_before[wave] = before;
            s_total[wave] = total;
            s_vis[wave] = vis;
            s_keys[wave] = keys;
            s_class_before[wave] = class_before;
            s_class_total[wave] = class_total;
        }
    }
    __syncthreads();
    const uint64_t total = (s_total[0] + s_total[1]) + (s_total[2] + s_total[3]);
    const uint64_t keys = (s_keys[0] + s_keys[1]) + (s_keys[2] + s_keys[3]);  // of whole rectangles: at least `total`
    const bool overflow = keys > (uint64_t)n_cap;
    if (blockIdx.x == 0 && threadIdx.x == 0 && !header_known) {
        const uint64_t packed = (s_class_total[0] + s_class_total[1]) + (s_class_total[2] + s_class_total[3]);
        const uint32_t in_class[3] = {class_count(packed, 0), class_count(packed, 1), class_count(packed, 2)};
        write_header(header, header_copy, keys, (uint32_t)total, overflow, n_cap, (s_vis[0] + s_vis[1]) + (s_vis[2] + s_vis[3]),
                     block_classes ? in_class : nullptr, class_count(packed, 3));
        if (block_classes && kTiles)
            for (int c = 0; c < 3; ++c) lists[c] = in_class[c];
    }
    if (overflow) return;  // later stages do nothing either

    if (blockIdx.x == 0 && bins > 0) {
        const int per_thread = (bins + 255) / 256;
        const int q0 = min((int)threadIdx.x * per_thread, bins), q1 = min(q0 + per_thread, bins);
        uint32_t chunks = 0;
        for (int q = q0; q < q1; ++q) chunks += chunks_of(bin_pairs[q]);
        uint32_t cinc = chunks;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t up = __shfl_up(cinc, d, 64);
            if (lane >= d) cinc += up;
        }
        if (lane == 63) s_chunks[wave] = cinc;
        __syncthreads();
        uint32_t run = cinc - chunks;
        for (int w = 0; w < wave; ++w) run += s_chunks[w];
        for (int q = q0; q < q1; ++q) {  // (each element is read before it is overwritten, by its own thread)
            const uint32_t n = chunks_of(bin_pairs[q]);
            chunk_base[q] = run;
            run += n;
        }
        if (threadIdx.x == 255) chunk_base[bins] = run;
    }

    uint64_t base = (s_before[0] + s_before[1]) + (s_before[2] + s_before[3]);  // first slot of the workgroup's blocks
    for (int w = 0; w < wave; ++w) base += first_block + (uint32_t)w < n_blocks ? block_sums[first_block + w] : 0ull;
    const uint32_t t = block * 64u + (uint32_t)lane;
    const bool live = t < tiles;
    const uint32_t v = live ? totals[t] : 0u;
    if (block * 64u >= tiles) return;  // (uniform per wavefront)
    const uint32_t inc = wave_sum_scan(v);
    const uint32_t first = (uint32_t)base + inc - v;
    if (live) tile_base[t] = first;
    if (!kTiles) return;
    if (live) {
        ranges[2 * t] = v ? first : 0u;
        ranges[2 * t + 1] = v ? first + v : 0u;
        tile_base[tiles + t] = first;  // the bucket's next free slot during the scatter
    }
    // buckets beyond the smallest sorter's capacity go on the list of their size class (order within a list is free;
    // without counts by block, one request per wavefront and class)
    const int cls = size_class(v);
    uint64_t class_first = 0;
    if (block_classes) {
        class_first = (s_class_before[0] + s_class_before[1]) + (s_class_before[2] + s_class_before[3]);
        for (int w = 0; w < wave; ++w) class_first += classes_of(first_block + (uint32_t)w);  // (earlier blocks exist)
    }
#pragma unroll
    for (int c = 0; c < 3; ++c) {
        const uint64_t m = __ballot(cls == c);
        if (m == 0ull) continue;
        uint32_t at = class_count(class_first, c);
        if (!block_classes) {
            const int leader = __ffsll((unsigned long long)m) - 1;
            if (lane == leader) at = atomicAdd(&lists[c], (uint32_t)__popcll(m));
            at = __shfl(at, leader, 64);
        }
        if (cls == c) lists[kListHeader + (size_t)c * tiles + lanes_below_in(m, at)] = t;
    }
}

constexpr int kRounds = 4;  // 64-key rounds per wavefront and step of a radix pass

// ---------------------------------------------------------------------------
// Storage of a bucket during sorting: two words per pair.
struct LdsPairs {
    uint32_t* d;  // depth bits
    uint32_t* i;  // Gaussian index
    __device__ __forceinline__ void load(uint32_t j, uint32_t& kd, uint32_t& ki) const
    {
        kd = d[j];
        ki = i[j];
    }
    __device__ __forceinline__ void store(uint32_t j, uint32_t kd, uint32_t ki) const
    {
        d[j] = kd;
        i[j] = ki;
    }
};

struct GlobalPairs {
    uint64_t* p;  // depth bits << 32 | Gaussian index
    __device__ __forceinline__ void load(uint32_t j, uint32_t& kd, uint32_t& ki) const
    {
        const uint64_t v = p[j];
        kd = (uint32_t)(v >> 32);
        ki = (uint32_t)v;
    }
    __device__ __forceinline__ void store(uint32_t j, uint32_t kd, uint32_t ki) const
    {
        p[j] = ((uint64_t)kd << 32) | (uint64_t)ki;
    }
};

struct SortScratch {
    uint32_t* hist;           // [256] digit totals, then running digit bases
    uint32_t (*cnt)[256];     // [kT / 64][256] per-wave digit counts of the current chunk
    uint32_t* flags;          // [8] small flags / partial sums
};

// One stable 8-bit LSD pass over n pairs, digit taken from the depth word
// (by_depth) or the index word.  Returns false (and moves nothing) when every
// pair has the same digit.
template <int kT, typename Src, typename Dst>
__device__ __forceinline__ bool radix_pass(const Src src, const Dst dst, uint32_t n, int shift, bool by_depth, const SortScratch sc)
{
    constexpr int kWaves = kT / 64, kChunk = kWaves * kRounds * 64;
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    const bool digit = kT == 256 || tid < 256;  // (uniform per wavefront) a thread per digit
    if (digit) sc.hist[tid] = 0;
    if (tid < 8) sc.flags[tid] = 0;
    __syncthreads();
    for (uint32_t j = tid; j < n; j += kT) {
        uint32_t kd, ki;
        src.load(j, kd, ki);
        atomicAdd(&sc.hist[((by_depth ? kd : ki) >> shift) & 255u], 1u);
    }
    __syncthreads();
    {
        // exclusive scan of the 256 digit totals; detect the single-digit case
        const uint32_t h = digit ? sc.hist[tid] : 0u;
        uint32_t inc = h;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t up = __shfl_up(inc, d, 64);
            if (lane >= d) inc += up;
        }
        if (digit && lane == 63) sc.flags[wave] = inc;
        if (h == n) sc.flags[4] = 1;
        __syncthreads();
        if (digit) {
            uint32_t off = 0;
            for (int w = 0; w < wave; ++w) off += sc.flags[w];
            sc.hist[tid] = off + inc - h;
        }
        const bool single = sc.flags[4] != 0;
        __syncthreads();
        if (single) return false;
    }
    const uint64_t lanes_below = (1ull << lane) - 1ull;
    for (uint32_t c0 = 0; c0 < n; c0 += kChunk) {
#pragma unroll
        for (int w = 0; w < kWaves; w += kT / 256) (&sc.cnt[w][0])[tid] = 0;
        __syncthreads();
        uint32_t kd[kRounds], ki[kRounds], rank[kRounds];
#pragma unroll
        for (int r = 0; r < kRounds; ++r) {
            const uint32_t j = c0 + (uint32_t)(wave * kRounds + r) * 64u + lane;
            const bool valid = j < n;
            kd[r] = 0;
            ki[r] = 0;
            if (valid) src.load(j, kd[r], ki[r]);
            const uint32_t dgt = ((by_depth ? kd[r] : ki[r]) >> shift) & 255u;
            uint64_t peers = __ballot(valid);
#pragma unroll
            for (int bit = 0; bit < 8; ++bit) {
                const bool one = (dgt >> bit) & 1u;
                const uint64_t m = __ballot(one);
                peers &= one ? m : ~m;
            }
            uint32_t pre = 0;
            const uint32_t below = (uint32_t)__popcll(peers & lanes_below);
            if (valid) {
                const int leader = __ffsll((unsigned long long)peers) - 1;
                if (lane == leader) pre = atomicAdd(&sc.cnt[wave][dgt], (uint32_t)__popcll(peers));
                pre = __shfl(pre, leader, 64);
            }
            rank[r] = pre + below;
        }
        __syncthreads();
        if (digit) {
            uint32_t run = sc.hist[tid];
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                const uint32_t c = sc.cnt[w][tid];
                sc.cnt[w][tid] = run;
                run += c;
            }
            sc.hist[tid] = run;
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kRounds; ++r) {
            const uint32_t j = c0 + (uint32_t)(wave * kRounds + r) * 64u + lane;
            if (j < n) {
                const uint32_t dgt = ((by_depth ? kd[r] : ki[r]) >> shift) & 255u;
                dst.store(sc.cnt[wave][dgt] + rank[r], kd[r], ki[r]);
            }
        }
        __syncthreads();
    }
    return true;
}

// Sort n pairs held in buffer A (B is scratch of the same size) by
// (depth bits, index).  Returns true if the result is in B.
template <int kT, typename Buf>
__device__ __forceinline__ bool sort_pairs(const Buf A, const Buf B, uint32_t n, const SortScratch sc)
{
    bool in_b = false;
    // depth passes; pairs of one tile rarely share depth bits, so the index
    // word is only brought in when a tie is actually present
    for (int pass = 0; pass < 4; ++pass) {
        const bool moved = in_b ? radix_pass<kT>(B, A, n, pass * 8, true, sc) : radix_pass<kT>(A, B, n, pass * 8, true, sc);
        if (moved) in_b = !in_b;
    }
    {
        const Buf cur = in_b ? B : A;
        if (threadIdx.x == 0) sc.flags[5] = 0;
        __syncthreads();
        bool tie = false;
        for (uint32_t j = threadIdx.x; j + 1 < n; j += kT) {
            uint32_t d0, i0, d1, i1;
            cur.load(j, d0, i0);
            cur.load(j + 1, d1, i1);
            tie |= (d0 == d1) && (i0 > i1);
        }
        if (tie) sc.flags[5] = 1;
        __syncthreads();
        const bool any = sc.flags[5] != 0;
        __syncthreads();
        if (!any) return in_b;
    }
    // equal depth bits out of index order: full (index, then depth) stable sort
    for (int pass = 0; pass < 8; ++pass) {
        const bool by_depth = pass >= 4;
        const int shift = (pass & 3) * 8;
        const bool moved = in_b ? radix_pass<kT>(B, A, n, shift, by_depth, sc) : radix_pass<kT>(A, B, n, shift, by_depth, sc);
        if (moved) in_b = !in_b;
    }
    return in_b;
}

template <int kT, typename Buf>
__device__ __forceinline__ void write_sorted(const Buf cur, uint32_t n, uint32_t tile, bool keys_too, uint64_t* out_keys,
                                             uint32_t* out_vals)
{
    for (uint32_t j = threadIdx.x; j < n; j += kT) {
        uint32_t kd, ki;
        cur.load(j, kd, ki);
        if (keys_too) out_keys[j] = ((uint64_t)tile << 32) | (uint64_t)kd;
        out_vals[j] = ki;
    }
}

// ---------------------------------------------------------------------------
// In-LDS bucket sorter: kT threads, up to kT * kR pairs, kR of them held in each thread's registers.
// The counting sort keeps the bucket in LDS once, as 64-bit pairs.  The radix passes it falls back to keep it as depth bits
// and index (8 B per pair) plus two 16-bit permutations that ping-pong between passes (4 B per pair), every pass ranking
// the whole bucket at once (each wavefront owns kR * 64 consecutive positions).
template <int kT, int kR>
struct LdsSorter {
    static constexpr int kW = kT / 64;
    static constexpr int kCap = kT * kR;
    // fine bins per thread of the counting pass: one 16-byte access
    static constexpr int kBinsPer = 4;
    static constexpr int kB = kBinsPer * kT;                      // fine bins
    // counters: [kW][256] words for the radix passes, or the fine bins and 512 coarse words of the counting pass
    static constexpr int kCounterWords = kB + 512 > kW * 256 ? kB + 512 : kW * 256;
    static constexpr size_t kBytes = (size_t)kCap * 12 + (size_t)kCounterWords * 4 + 192;

    uint32_t* depth;     // [kCap]
    uint32_t* index;     // [kCap]
    uint16_t* perm0;     // two permutations of [kCap] each, back to back
    uint32_t (*cnt)[256];  // [kW][256]
    uint32_t* flags;     // [48]

    __device__ explicit LdsSorter(uint32_t* lds)
    {
        depth = lds;
        index = lds + kCap;
        perm0 = reinterpret_cast<uint16_t*>(lds + 2 * kCap);
        cnt = reinterpret_cast<uint32_t(*)[256]>(lds + 3 * kCap);
        flags = lds + 3 * kCap + kCounterWords;
    }

    __device__ __forceinline__ uint16_t* perm(int which) const { return perm0 + which * kCap; }

    // One stable pass.  `src` < 0: the input order is the identity.  Returns the
    // buffer holding the output order (unchanged when all digits are equal).
    __device__ __forceinline__ int pass(uint32_t n, int shift, bool by_depth, int src) const
    {
        const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
        for (int k = tid; k < kW * 256; k += kT) (&cnt[0][0])[k] = 0;
        if (tid == 0) flags[8] = 0;
        __syncthreads();
        const int dst = src == 0 ? 1 : 0;
        const uint64_t lanes_below = (1ull << lane) - 1ull;
        uint32_t ent[kR];  // entry | digit << 16
        uint32_t rank[kR];
#pragma unroll
        for (int r = 0; r < kR; ++r) {
            ent[r] = 0;
            rank[r] = 0;
            if ((uint32_t)(wave * kR + r) * 64u >= n) continue;  // whole round past the end (uniform per wavefront)
            const uint32_t j = (uint32_t)(wave * kR + r) * 64u + lane;
            const bool valid = j < n;
            const uint32_t e = valid ? (src < 0 ? j : (uint32_t)perm(src)[j]) : 0u;
            const uint32_t key = valid ? (by_depth ? depth[e] : index[e]) : 0u;
            const uint32_t dgt = (key >> shift) & 255u;
            uint64_t peers = __ballot(valid);
#pragma unroll
            for (int bit = 0; bit < 8; ++bit) {
                const bool one = (dgt >> bit) & 1u;
                const uint64_t m = __ballot(one);
                peers &= one ? m : ~m;
            }
            uint32_t pre = 0;
            const uint32_t below = (uint32_t)__popcll(peers & lanes_below);
            if (valid) {
                const int leader = __ffsll((unsigned long long)peers) - 1;
                if (lane == leader) pre = atomicAdd(&cnt[wave][dgt], (uint32_t)__popcll(peers));
                pre = __shfl(pre, leader, 64);
            }
            rank[r] = pre + below;
            ent[r] = e | (dgt << 16);
        }
        __syncthreads();
        // digit totals, exclusive scan over the 256 digits (wavefronts 0..3), per-wave bases
        uint32_t total = 0, inc = 0;
        if (tid < 256) {
#pragma unroll
            for (int w = 0; w < kW; ++w) total += cnt[w][tid];
            if (total == n) flags[8] = 1;  // every pair has this digit: nothing to move
            inc = total;
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const uint32_t up = __shfl_up(inc, d, 64);
                if (lane >= d) inc += up;
            }
            if (lane == 63) flags[wave] = inc;
        }
        __syncthreads();
        if (tid < 256) {
            uint32_t base = inc - total;
            for (int w = 0; w < wave; ++w) base += flags[w];
#pragma unroll
            for (int w = 0; w < kW; ++w) {
                const uint32_t c = cnt[w][tid];
                cnt[w][tid] = base;
                base += c;
            }
        }
        __syncthreads();
        const bool single = flags[8] != 0;
        if (!single) {
#pragma unroll
            for (int r = 0; r < kR; ++r) {
                const uint32_t j = (uint32_t)(wave * kR + r) * 64u + lane;
                if (j < n) perm(dst)[cnt[wave][ent[r] >> 16] + rank[r]] = (uint16_t)ent[r];
            }
        }
        __syncthreads();
        return single ? src : dst;
    }

    // Sort the n loaded pairs by (depth bits, index); returns the buffer with
    // the final order.
    __device__ __forceinline__ int sort(uint32_t n, uint32_t varying) const
    {
        int cur = -1;
        // bytes of the depth word that are identical in every pair need no pass
        // (inside one tile the exponent byte of the depths usually is)
        for (int p = 0; p < 4; ++p)
            if ((varying >> (p * 8)) & 255u) cur = pass(n, p * 8, true, cur);
        if (cur < 0) {  // no pass moved anything (all depth bits equal, or n == 1): start from the identity
            for (uint32_t j = threadIdx.x; j < n; j += kT) perm(0)[j] = (uint16_t)j;
            cur = 0;
            __syncthreads();
        }
        // Bucket order before the sort is arbitrary, so pairs with equal depth
        // bits may be out of index order.  Such runs are rare and short: a few
        // rounds of odd-even transposition inside runs settle them; only if a
        // round still swaps after that is the full (index, depth) sort run.
        uint16_t* const P = perm(cur);
        bool unsettled = true;
        for (int round = 0; round < 4 && unsettled; ++round) {
            if (threadIdx.x == 0) flags[10] = 0;
            __syncthreads();
            bool swapped = false;
            for (int phase = 0; phase < 2; ++phase) {
                for (uint32_t j = 2u * threadIdx.x + phase; j + 1 < n; j += 2u * kT) {
                    const uint32_t e0 = P[j], e1 = P[j + 1];
                    if (depth[e0] == depth[e1] && index[e0] > index[e1]) {
                        P[j] = (uint16_t)e1;
                        P[j + 1] = (uint16_t)e0;
                        swapped = true;
                    }
                }
                __syncthreads();
            }
            if (swapped) flags[10] = 1;
            __syncthreads();
            unsettled = flags[10] != 0;
            __syncthreads();
        }
        if (!unsettled) return cur;
        for (int p = 0; p < 8; ++p) cur = pass(n, (p & 3) * 8, p >= 4, cur);
        return cur;
    }

    // Fast path: one counting pass over a monotone map of the depth onto kB bins leaves a pair or two per bin; every pair
    // then ranks itself among the members of its bin.  Bins are ordered and each bin is fully ordered, so the result is
    // the exact total order by (depth bits, index) whatever order the LDS atomics ran in.
    // Depths along the rays of a tile cluster (most splats sit near the ground), so the map is adaptive: a
    // 256-bin histogram over [dmin, dmax] gives a piecewise-linear estimate of each pair's final position, and
    // the bin is that position scaled to kB.  Positions are floats: conversion, multiplication and multiply-add round
    // monotonically and a coarse bin's end is a whole number, so the map stays monotone.
    // The pairs wait in registers, and pass through LDS three times as they are (to their bin, to its ranking readers, to
    // their place): ten LDS accesses per pair.  Kept in LDS as separate words behind a permutation they took twenty (6M
    // Gaussians, 1080p, 13.4M pairs: the four classes 17 + 51 + 80 + 20 us, so 15 + 36 + 61 + 11).
    // Returns false when some bin is too full for this to pay (nothing but the counters has then been written): the caller
    // runs the radix passes.
    static constexpr uint32_t kMaxBin = 256;

    // `keys_too`: leaves the sorted pairs in the place of `depth`, else their indices.  (Values alone: 6M Gaussians 84 -> 79 us
    // for all classes, 1M large splats 63 -> 60, 20M at 4K 161 -> 155.)
    __device__ __forceinline__ bool counting_sort(const uint64_t (&v)[kR], uint32_t n, uint32_t dmin, uint32_t dmax, bool keys_too) const
    {
        const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
        uint32_t* const count = &cnt[0][0];                              // [kB] pairs per bin, then the bin's first slot
        uint32_t* const coarse = count + kB;                             // [256] pairs per coarse bin
        float2* const line = reinterpret_cast<float2*>(coarse);          // [256] pairs before it and in it (same words)
        uint64_t* const pairs = reinterpret_cast<uint64_t*>(depth);      // [kCap]
        const uint32_t range = dmax - dmin;
        const float scale = 256.0f / ((float)range + 1.0f);
        const float to_bin = n > (uint32_t)kB ? (float)kB / (float)n : 1.0f;
        // (the counters were cleared by the caller, before the barrier that made dmin and dmax known)
        float at[kR];
#pragma unroll
        for (int r = 0; r < kR; ++r) {
            at[r] = fminf((float)((uint32_t)(v[r] >> 32) - dmin) * scale, 255.99998f);
            if ((uint32_t)r * kT + tid < n) atomicAdd(&coarse[(uint32_t)at[r]], 1u);
        }
        __syncthreads();
        uint32_t own = 0, inc = 0;
        if (tid < 256) {  // exclusive scan of the coarse counts (wavefronts 0..3)
            own = coarse[tid];
            inc = wave_sum_scan(own);
            if (lane == 63) flags[16 + wave] = inc;
        }
        __syncthreads();
        if (tid < 256) {
            uint32_t before = inc - own;
            for (int w = 0; w < wave; ++w) before += flags[16 + w];
            line[tid] = make_float2((float)before, (float)own);
        }
        __syncthreads();
        uint32_t bin[kR], slot[kR];
#pragma unroll
        for (int r = 0; r < kR; ++r) {
            bin[r] = slot[r] = 0;
            if ((uint32_t)r * kT + tid < n) {
                const float2 l = line[(uint32_t)at[r]];
                const float pos = __builtin_fmaf(__builtin_amdgcn_fractf(at[r]), l.y, l.x);  // in [0, n]
                bin[r] = min((uint32_t)(pos * to_bin), (uint32_t)kB - 1u);
                slot[r] = atomicAdd(&count[bin[r]], 1u);
            }
        }
        __syncthreads();
        // exclusive scan of the kB bin counts (a thread owns four consecutive bins)
        uint4 mine = reinterpret_cast<const uint4*>(count)[tid];
        const uint32_t c = (mine.x + mine.y) + (mine.z + mine.w);
        inc = wave_sum_scan(c);
        if (lane == 63) flags[16 + wave] = inc;
        if (max(max(mine.x, mine.y), max(mine.z, mine.w)) > kMaxBin) flags[8] = 1;
        __syncthreads();
        if (flags[8] != 0) {
            __syncthreads();
            return false;
        }
        uint32_t first = inc - c;
        for (int w = 0; w < wave; ++w) first += flags[16 + w];
        const uint32_t f1 = first + mine.x, f2 = f1 + mine.y;
        reinterpret_cast<uint4*>(count)[tid] = make_uint4(first, f1, f2, f2 + mine.z);
        if (tid == 0) count[kB] = n;  // (over the coarse bins, which are done with)
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kR; ++r)
            if ((uint32_t)r * kT + tid < n) pairs[count[bin[r]] + slot[r]] = v[r];
        if (tid < 4) pairs[n + tid] = ~0ull;  // (the permutations' area follows)
        __syncthreads();
        // A pair's rank among the members of its bin, four at a time: what follows the bin is larger than all of them, so
        // a bin of up to four needs no further test.
#pragma unroll
        for (int r = 0; r < kR; ++r) {
            if ((uint32_t)r * kT + tid < n) {
                const uint32_t lo = count[bin[r]], hi = count[bin[r] + 1];
                uint32_t rank = lo;
                for (uint32_t q = lo; q < hi; q += 4) {
#pragma unroll
                    for (uint32_t k = 0; k < 4; ++k) rank += pairs[q + k] < v[r] ? 1u : 0u;
                }
                slot[r] = rank;
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kR; ++r)
            if ((uint32_t)r * kT + tid < n) {
                if (keys_too) pairs[slot[r]] = v[r];
                else depth[slot[r]] = (uint32_t)v[r];
            }
        __syncthreads();
        return true;
    }

    // A bucket on its way from memory: where it lies and this thread's pairs of it (requested, not yet used).
    struct Fetched {
        uint32_t tile, lo, n;
        uint64_t v[kR];
    };

    __device__ __forceinline__ void fetch_range(Fetched& f, uint32_t tile, const uint32_t* __restrict__ ranges) const
    {
        f.tile = tile;
        f.lo = ranges[2 * tile];
        f.n = ranges[2 * tile + 1] - f.lo;
    }

    // the whole bucket is requested before the first pair is used: one memory latency, not one per round
    __device__ __forceinline__ void fetch_pairs(Fetched& f, const uint64_t* __restrict__ buckets) const
    {
        const bool mine = f.n != 0 && f.n <= (uint32_t)kCap;
#pragma unroll
        for (int r = 0; r < kR; ++r) {
            const uint32_t j = (uint32_t)r * kT + threadIdx.x;
            f.v[r] = mine && j < f.n ? __builtin_nontemporal_load(&buckets[f.lo + j]) : 0ull;  // (read once)
        }
    }

    // Sorts the fetched bucket and writes it out; ends with a barrier.
    __device__ __forceinline__ void sort_fetched(const Fetched& f, bool keys_too, uint64_t* __restrict__ out_keys,
                                                 uint32_t* __restrict__ out_vals) const
    {
        const uint32_t lo = f.lo, n = f.n, tile = f.tile;
        if (n == 0 || n > (uint32_t)kCap) return;  // uniform over the workgroup
        uint32_t dmin = 0xFFFFFFFFu, dmax = 0;
#pragma unroll
        for (int r = 0; r < kR; ++r) {
            if ((uint32_t)r * kT + threadIdx.x < n) {
                const uint32_t dj = (uint32_t)(f.v[r] >> 32);
                dmin = min(dmin, dj);
                dmax = max(dmax, dj);
            }
        }
        dmin = wave_scan(dmin, 0xFFFFFFFFu, [](uint32_t a, uint32_t b) { return min(a, b); });
        dmax = wave_scan(dmax, 0u, [](uint32_t a, uint32_t b) { return max(a, b); });
        const int wave = threadIdx.x >> 6;
        if ((threadIdx.x & 63) == 63) {
            flags[16 + wave] = dmin;
            flags[32 + wave] = dmax;
        }
        {  // the counting sort's counters, cleared here so that it needs no barrier of its own for it
            uint4* const count = reinterpret_cast<uint4*>(&cnt[0][0]);
            count[threadIdx.x] = make_uint4(0u, 0u, 0u, 0u);
            if (threadIdx.x < 128) count[kT + threadIdx.x] = make_uint4(0u, 0u, 0u, 0u);
            if (threadIdx.x == 0) flags[8] = 0;
        }
        __syncthreads();
        dmin = 0xFFFFFFFFu;
        dmax = 0;
#pragma unroll
        for (int w = 0; w < kW; ++w) {
            dmin = min(dmin, flags[16 + w]);
            dmax = max(dmax, flags[32 + w]);
        }
        if (counting_sort(f.v, n, dmin, dmax, keys_too)) {
            if (keys_too) {
                const uint64_t* const pairs = reinterpret_cast<const uint64_t*>(depth);
                for (uint32_t j = threadIdx.x; j < n; j += kT) {
                    const uint64_t v = pairs[j];
                    // (no later stage reads the sorted keys: a streaming store, which leaves the cache to the records the
                    // blend is about to gather)
                    __builtin_nontemporal_store(((uint64_t)tile << 32) | (v >> 32), &out_keys[lo + j]);
                    out_vals[lo + j] = (uint32_t)v;
                }
            } else {
                for (uint32_t j = threadIdx.x; j < n; j += kT) out_vals[lo + j] = depth[j];
            }
        } else {
            // depth bits that differ somewhere in the bucket: (OR of all) ^ (AND of all)
            uint32_t any = 0, all = 0xFFFFFFFFu;
            if (threadIdx.x == 0) {
                flags[11] = 0;
                flags[14] = 0xFFFFFFFFu;
            }
            __syncthreads();
#pragma unroll
            for (int r = 0; r < kR; ++r) {
                const uint32_t j = (uint32_t)r * kT + threadIdx.x;
                if (j < n) {
                    const uint32_t dj = (uint32_t)(f.v[r] >> 32);
                    depth[j] = dj;
                    index[j] = (uint32_t)f.v[r];
                    any |= dj;
                    all &= dj;
                }
            }
            atomicOr(&flags[11], any);
            atomicAnd(&flags[14], all);
            __syncthreads();
            const int cur = sort(n, flags[11] ^ flags[14]);
            for (uint32_t j = threadIdx.x; j < n; j += kT) {
                const uint32_t e = cur < 0 ? j : (uint32_t)perm(cur)[j];
                if (keys_too) __builtin_nontemporal_store(((uint64_t)tile << 32) | (uint64_t)depth[e], &out_keys[lo + j]);
                out_vals[lo + j] = index[e];
            }
        }
        __syncthreads();
    }

    __device__ __forceinline__ void run(uint32_t tile, const uint32_t* __restrict__ ranges, const uint64_t* __restrict__ buckets,
                        bool keys_too, uint64_t* __restrict__ out_keys, uint32_t* __restrict__ out_vals) const
    {
        Fetched f;
        fetch_range(f, tile, ranges);
        fetch_pairs(f, buckets);
        sort_fetched(f, keys_too, out_keys, out_vals);
    }
};

// The counting sort of LdsSorter by one wavefront, for buckets of up to 256 pairs: no barriers, and four times as many buckets
// side by side.  (A workgroup of four wavefronts per bucket waits at ten barriers however few pairs there are.)  It has no
// radix passes to fall back to: depths that share a bin rank themselves among all of it, which for 256 equal depths are 64
// steps.  8160 tiles of 145 pairs: 18.8 -> 13.8 us, 4056 of 93: 10.8 -> 9.4, 2170 of 243: 9.7 -> 8.6; frames of larger buckets
// unchanged.  For up to 512 pairs (eight per lane): 16.3, 11.1 and 10.0, and 500k anchors' tiles 24.8 -> 29.1.  Sorted by the
// wavefronts of the workgroups that the larger buckets have, one of four: slower than without (octree frame 206 -> 212).
struct WaveSorter {
    static constexpr int kR = 4, kCap = 64 * kR, kB = kCap;  // pairs per lane, pairs, fine bins
    static constexpr int kCoarse = 64;
    static constexpr int kWords = 2 * (kCap + 4) + kB + 4 + 2 * kCoarse;

    uint64_t* pairs;  // [kCap + 4]
    uint32_t* count;  // [kB + 4]
    uint32_t* coarse;  // [kCoarse]; float2 [kCoarse] over the same words

    __device__ explicit WaveSorter(uint32_t* lds)
        : pairs(reinterpret_cast<uint64_t*>(lds)), count(lds + 2 * (kCap + 4)), coarse(lds + 2 * (kCap + 4) + kB + 4)
    {
    }

    __device__ __forceinline__ void run(uint32_t tile, uint32_t lo, uint32_t n, const uint64_t* __restrict__ buckets, bool keys_too,
                                        uint64_t* __restrict__ out_keys, uint32_t* __restrict__ out_vals) const
    {
        const uint32_t lane = threadIdx.x & 63u;
        if (n == 0u || n > (uint32_t)kCap) return;  // (uniform)
        uint64_t v[kR];
#pragma unroll
        for (uint32_t r = 0; r < kR; ++r) v[r] = r * 64u + lane < n ? __builtin_nontemporal_load(&buckets[lo + r * 64u + lane]) : 0ull;  // (read once)
        reinterpret_cast<uint4*>(count)[lane] = make_uint4(0u, 0u, 0u, 0u);
        coarse[lane] = 0u;
        uint32_t dmin = 0xFFFFFFFFu, dmax = 0;
#pragma unroll
        for (uint32_t r = 0; r < kR; ++r) {
            if (r * 64u + lane < n) {
                dmin = min(dmin, (uint32_t)(v[r] >> 32));
                dmax = max(dmax, (uint32_t)(v[r] >> 32));
            }
        }
        dmin = (uint32_t)__builtin_amdgcn_readlane((int)wave_scan(dmin, 0xFFFFFFFFu, [](uint32_t a, uint32_t b) { return min(a, b); }), 63);
        dmax = (uint32_t)__builtin_amdgcn_readlane((int)wave_scan(dmax, 0u, [](uint32_t a, uint32_t b) { return max(a, b); }), 63);
        wave_lds_sync();
        const float scale = (float)kCoarse / ((float)(dmax - dmin) + 1.0f);
        float at[kR];
#pragma unroll
        for (uint32_t r = 0; r < kR; ++r) {
            at[r] = fminf((float)((uint32_t)(v[r] >> 32) - dmin) * scale, (float)kCoarse - 0.00001f);
            if (r * 64u + lane < n) atomicAdd(&coarse[(uint32_t)at[r]], 1u);
        }
        wave_lds_sync();
        const uint32_t own = coarse[lane], inc = wave_sum_scan(own);
        wave_lds_sync();
        float2* const line = reinterpret_cast<float2*>(coarse);
        line[lane] = make_float2((float)(inc - own), (float)own);
        wave_lds_sync();
        uint32_t bin[kR], slot[kR];
#pragma unroll
        for (uint32_t r = 0; r < kR; ++r) {
            bin[r] = slot[r] = 0;
            if (r * 64u + lane < n) {
                const float2 l = line[(uint32_t)at[r]];
                const float pos = __builtin_fmaf(__builtin_amdgcn_fractf(at[r]), l.y, l.x);  // in [0, n]
                bin[r] = min((uint32_t)pos, (uint32_t)kB - 1u);
                slot[r] = atomicAdd(&count[bin[r]], 1u);
            }
        }
        wave_lds_sync();
        const uint4 mine = reinterpret_cast<const uint4*>(count)[lane];  // (a lane owns four consecutive bins)
        const uint32_t c = (mine.x + mine.y) + (mine.z + mine.w);
        const uint32_t first = wave_sum_scan(c) - c, f1 = first + mine.x, f2 = f1 + mine.y;
        wave_lds_sync();
        reinterpret_cast<uint4*>(count)[lane] = make_uint4(first, f1, f2, f2 + mine.z);
        if (lane == 0) count[kB] = n;
        if (lane < 4) pairs[n + lane] = ~0ull;
        wave_lds_sync();
#pragma unroll
        for (uint32_t r = 0; r < kR; ++r)
            if (r * 64u + lane < n) pairs[count[bin[r]] + slot[r]] = v[r];
        wave_lds_sync();
        // (as LdsSorter: what follows the bin is larger than all of its members)
#pragma unroll
        for (uint32_t r = 0; r < kR; ++r) {
            if (r * 64u + lane < n) {
                const uint32_t begin = count[bin[r]], end = count[bin[r] + 1];
                uint32_t rank = begin;
                for (uint32_t q = begin; q < end; q += 4) {
#pragma unroll
                    for (uint32_t k = 0; k < 4; ++k) rank += pairs[q + k] < v[r] ? 1u : 0u;
                }
                slot[r] = rank;
            }
        }
        wave_lds_sync();
#pragma unroll
        for (uint32_t r = 0; r < kR; ++r)
            if (r * 64u + lane < n) pairs[slot[r]] = v[r];
        wave_lds_sync();
#pragma unroll
        for (uint32_t r = 0; r < kR; ++r) {
            const uint32_t j = r * 64u + lane;
            if (j < n) {
                const uint64_t p = pairs[j];
                if (keys_too) __builtin_nontemporal_store(((uint64_t)tile << 32) | (p >> 32), &out_keys[lo + j]);
                out_vals[lo + j] = (uint32_t)p;
            }
        }
    }
};

// Tiles in the order of their lists' lengths, longest first, as (tile, first, last, 0).  The blends' workgroups nearly all start at
// once in frames of a few thousand tiles, and the compute unit with the longest lists decides; in larger frames the last ones to
// start do.  2170 tiles: blend 47.1 -> 44.7 us, 1734: backward blend 100.5 -> 96.1; 8160 tiles, 6M Gaussians: 276.9 -> 272.6 and
// 844.7 -> 830.1, although neighbouring tiles no longer find each other's records in the L2.  One workgroup beside the sorts
// makes it, in 9 us for 8160 tiles, 16 for 14400 and 32 for 32400 (nearly all empty: 58, they share a bin), so it is made where
// the sorts take as long, from kOrderMinPairs pairs per tile on average (the sorts of 2170 tiles 9.1 -> 9.5 us with it).  With fewer it was the
// launch's length and the blends gained nothing: at 3840x2160 frames of 17, 14k, 582k and 2.2M pairs 126, 120, 155 and 249 us with it, 84,
// 94, 143 and 237 without; at 1920x1080 of 19, 30k and 500k pairs 48, 51 and 76, and 39, 48 and 73.
// Lengths are taken to a sixteenth of a power of two; the order within one of those steps is free.
constexpr int kOrderBins = 512;        // sixteen steps for each of 32 powers of two
constexpr int kOrderMinTiles = 257;    // up to a tile per compute unit there is nothing to order
constexpr int kOrderMaxTiles = kBinMaxTiles;
constexpr uint32_t kOrderMinPairs = 128;  // per tile

template <int kT>
__device__ __forceinline__ void order_tiles(const uint32_t* __restrict__ ranges, uint32_t tiles, uint4* __restrict__ order,
                                            uint32_t* __restrict__ lds)
{
    static_assert(kOrderBins % kT == 0 || kT % kOrderBins == 0, "bins per thread");
    constexpr int kAhead = 8, kPer = kOrderBins > kT ? kOrderBins / kT : 1;
    uint32_t* const bins = lds;
    uint32_t* const sums = lds + kOrderBins;  // per wavefront
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint2* __restrict__ range = reinterpret_cast<const uint2*>(ranges);
    auto bin_of = [](uint32_t n) {  // the longest first; exponents of (float)n: 127 to 159
        constexpr uint32_t last = kOrderBins - 1;
        return n == 0u ? last : last - 1u - min((__float_as_uint((float)n) >> 19) - (127u << 4), last - 1u);
    };
    for (uint32_t b = tid; b < (uint32_t)kOrderBins; b += kT) bins[b] = 0u;
    __syncthreads();
    auto each = [&](auto visit) {
        for (uint32_t t0 = tid; t0 < tiles; t0 += kAhead * kT) {
            uint2 r[kAhead];
#pragma unroll
            for (uint32_t u = 0; u < kAhead; ++u) r[u] = range[min(t0 + u * kT, tiles - 1u)];
#pragma unroll
            for (uint32_t u = 0; u < kAhead; ++u)
                if (t0 + u * kT < tiles) visit(t0 + u * kT, r[u]);
        }
    };
    each([&](uint32_t, uint2 r) { atomicAdd(&bins[bin_of(r.y - r.x)], 1u); });
    __syncthreads();
    uint32_t own[kPer], sum = 0;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        own[k] = kPer * tid + k < (uint32_t)kOrderBins ? bins[kPer * tid + k] : 0u;
        sum += own[k];
    }
    const uint32_t inc = wave_sum_scan(sum);
    if (lane == 63u) sums[wave] = inc;
    __syncthreads();
    uint32_t at = inc - sum;
    for (uint32_t w = 0; w < wave; ++w) at += sums[w];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        if (kPer * tid + k < (uint32_t)kOrderBins) bins[kPer * tid + k] = at;
        at += own[k];
    }
    __syncthreads();
    each([&](uint32_t t, uint2 r) { order[atomicAdd(&bins[bin_of(r.y - r.x)], 1u)] = make_uint4(t, r.x, r.y, 0u); });
}

// Smallest size class: one workgroup per tile; tiles with larger buckets leave at once.  `skip_classes` (bit c: the sorter of
// larger class c is not launched for this frame, the caller expecting no bucket of that size): such a bucket, should there be
// one after all, is sorted here by radix passes through global memory, ping-ponging between the bucket and the tile's slice
// of the output keys (their scratch lies over the LDS sorter's area), so every bucket is sorted whatever the caller expected.
//
// The first workgroup is none of the tiles': in frames of many pairs it orders them by the length of their lists for the blends
// (order_tiles), beside the sorts.  kByWave: behind the workgroups with a tile each come some with a wavefront per tile, four consecutive ones, for the
// buckets of up to 256 pairs, which the others leave.
template <int kT, int kR, bool kByWave>
__global__ __launch_bounds__(kT) void tile_sort_each_kernel(gs355_header* header,
                                                            const uint32_t* __restrict__ ranges,
                                                            uint64_t* __restrict__ buckets,
                                                            uint64_t* __restrict__ out_keys,
                                                            uint32_t* __restrict__ out_vals, bool keys_too, uint32_t skip_classes,
                                                            uint4* __restrict__ order, uint32_t tiles)
{
    extern __shared__ uint32_t s_dyn[];
    if (header->overflow) return;
    if (order && blockIdx.x == 0) {
        static_assert((kOrderBins + kT / 64) * sizeof(uint32_t) <= LdsSorter<kT, kR>::kBytes, "bins and sums");
        if (header->num_keys < kOrderMinPairs * tiles) return;
        order_tiles<kT>(ranges, tiles, order, s_dyn);
        if (threadIdx.x == 0) header->ordered = 1u;
        return;
    }
    constexpr int kThreads = 256;  // of a bucket that goes through global memory
    static_assert((256 + kThreads / 64 * 256 + 8) * sizeof(uint32_t) <= LdsSorter<kT, kR>::kBytes, "scratch of the global passes");
    const uint32_t block = blockIdx.x - (order ? 1u : 0u);
    if (kByWave && block >= tiles) {
        static_assert(!kByWave || WaveSorter::kWords * (kT / 64) * sizeof(uint32_t) <= LdsSorter<kT, kR>::kBytes, "a sorter per wavefront");
        const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), tile = (block - tiles) * (kT / 64) + wave;
        if (tile >= tiles) return;
        const uint2 r = reinterpret_cast<const uint2*>(ranges)[tile];
        WaveSorter(s_dyn + wave * WaveSorter::kWords).run(tile, r.x, r.y - r.x, buckets, keys_too, out_keys, out_vals);
        return;
    }
    const uint32_t tile = block;
    const uint32_t lo = ranges[2 * tile], n = ranges[2 * tile + 1] - lo;
    if (kByWave && n <= (uint32_t)WaveSorter::kCap) return;
    bool through_global = false;
    if (skip_classes != 0u && n > (uint32_t)LdsSorter<kT, kR>::kCap) {
        const int cls = n <= (uint32_t)kTileSortCap[1] ? 0 : n <= (uint32_t)kTileSortCap[2] ? 1 : 2;
        through_global = (skip_classes >> cls) & 1u;
    }
    if (through_global) {  // (uniform over the workgroup; passes of kThreads threads)
        if (threadIdx.x >= kThreads) return;
        const SortScratch sc = {s_dyn, reinterpret_cast<uint32_t(*)[256]>(s_dyn + 256), s_dyn + 256 + kThreads / 64 * 256};
        const GlobalPairs A = {buckets + lo}, B = {out_keys + lo};
        const bool in_b = sort_pairs<kThreads>(A, B, n, sc);
        // when the result sits in the output slice itself, each element is rewritten in place by the thread that read it
        write_sorted<kThreads>(in_b ? B : A, n, tile, keys_too, out_keys + lo, out_vals + lo);
        return;
    }
    const LdsSorter<kT, kR> sorter(s_dyn);
    sorter.run(tile, ranges, buckets, keys_too, out_keys, out_vals);
}

// Larger size classes: one workgroup per entry of the class list made with the layout.  The number of
// entries is only known on the device, so a launch has a workgroup per tile and those past the list's end leave at
// once: the hardware's own dispatch hands out the buckets.  (Persistent workgroups that fetched their work from a
// counter spent 8-14 us per bucket on dependent requests -- counter, list entry, range, pairs -- whatever the
// bucket held, requesting the next bucket inside the current sort did not hide them, and even a plain strided loop
// around the sort costs a sixth of the kernel's time in registers kept alive across it.)
template <int kT, int kR>
__device__ __forceinline__ void tile_sort_list_body(const gs355_header* __restrict__ header,
                                                    const uint32_t* __restrict__ ranges,
                                                    const uint32_t* __restrict__ list,
                                                    const uint32_t* __restrict__ list_count,
                                                    const uint64_t* __restrict__ buckets,
                                                    bool keys_too, uint64_t* __restrict__ out_keys,
                                                    uint32_t* __restrict__ out_vals, uint32_t* lds)
{
    if (header->overflow) return;
    const LdsSorter<kT, kR> sorter(lds);
    if (blockIdx.x < *list_count) sorter.run(list[blockIdx.x], ranges, buckets, keys_too, out_keys, out_vals);
}

// 1024 threads x 5 rounds, held to 64 VGPRs so that two workgroups share a CU
__global__ __launch_bounds__(1024) __attribute__((amdgpu_waves_per_eu(8, 8))) void tile_sort_list_1024x5_kernel(
    const gs355_header* __restrict__ header, const uint32_t* __restrict__ ranges, const uint32_t* __restrict__ list,
    const uint32_t* __restrict__ list_count, const uint64_t* __restrict__ buckets, bool keys_too, uint64_t* __restrict__ out_keys,
    uint32_t* __restrict__ out_vals)
{
    extern __shared__ uint32_t s_dyn[];
    tile_sort_list_body<1024, 5>(header, ranges, list, list_count, buckets, keys_too, out_keys, out_vals, s_dyn);
}

template <int kT, int kR>
__global__ __launch_bounds__(kT) void tile_sort_list_kernel(const gs355_header* __restrict__ header,
                                                            const uint32_t* __restrict__ ranges,
                                                            const uint32_t* __restrict__ list,
                                                            const uint32_t* __restrict__ list_count,
                                                            const uint64_t* __restrict__ buckets, bool keys_too,
                                                            uint64_t* __restrict__ out_keys,
                                                            uint32_t* __restrict__ out_vals)
{
    extern __shared__ uint32_t s_dyn[];
    tile_sort_list_body<kT, kR>(header, ranges, list, list_count, buckets, keys_too, out_keys, out_vals, s_dyn);
}

// The largest class, 5121 pairs and more: a workgroup of it fills a CU, so the launch is the chip's size and strides over the
// list.  A bucket beyond the LDS sorter's capacity is written to the tile's slice of the output keys first, ordered by kBins
// bins of its depths (their range, two counts and a move: the bins' cursors are in LDS), and then goes through LDS piece by
// piece, as many whole bins as fit, where each pair ranks itself among its bin's.  Buckets with a bin of more than kMaxBin pairs
// sort the pieces as LDS sorters do, and a single bin that none holds (equal depths, or nearly) goes through global memory by
// radix passes, between the output keys and the bucket.  Radix passes by 256 threads took eight reads, four writes and a step of
// four barriers per 1024 pairs of each: 6M Gaussians at 979x546 (tiles of up to 12k pairs among 2170) 383 -> 90 us with the smallest
// class's kernel, which sorted them; at 400x300 (475 tiles of 14k) 2158 -> 260.  (Bins of equal width and every piece through the LDS
// sorter: 103 and 299.  Buckets of up to 16k pairs held in LDS and registers throughout: 111 and 288, the registers spill.)
struct LargeSorter {
    using Piece = LdsSorter<1024, 10>;
    static constexpr int kT = 1024, kBins = 4096, kWaves = kT / 64, kAhead = 4;
    static constexpr int kLine = 2 * Piece::kCap + 8;  // words before the map's lines (behind a piece's pairs and four more)
    static constexpr uint32_t kMaxBin = 128;
    static_assert(kBins + 2 * kWaves <= kLine && (kLine + 512) * sizeof(uint32_t) <= Piece::kBytes && kLine % 2 == 0, "apart");
    static constexpr size_t kBytes = Piece::kBytes + kBins * sizeof(uint32_t);
    static_assert(kBins == 4 * kT && kBins == 64 * 64, "four bins a thread; a lane for each 64 of them");
    static_assert(Piece::kBytes % 16 == 0 && kBytes <= 160 * 1024, "in the CU's LDS");
    static_assert((256 + kWaves * 256 + 8) * sizeof(uint32_t) <= Piece::kBytes, "scratch of the global passes");

    uint32_t* lds;
    uint32_t* first;  // [kBins] pairs in the bins before each

    __device__ explicit LargeSorter(uint32_t* s) : lds(s), first(s + Piece::kBytes / sizeof(uint32_t)) {}

    // calls f(pair) for this thread's pairs of the n at `from`, kAhead of them requested together
    template <typename F>
    static __device__ __forceinline__ void each(const uint64_t* from, uint32_t n, F f)
    {
        for (uint32_t j0 = threadIdx.x; j0 < n; j0 += kAhead * kT) {
            uint64_t v[kAhead];
#pragma unroll
            for (int u = 0; u < kAhead; ++u) v[u] = from[min(j0 + (uint32_t)u * kT, n - 1u)];
#pragma unroll
            for (int u = 0; u < kAhead; ++u)
                if (j0 + (uint32_t)u * kT < n) f(v[u]);
        }
    }

    // The map of depths onto bins, as in LdsSorter::counting_sort: 256 coarse bins give a pair's likely position, which is
    // scaled to the fine bins.  (Positions below 2^24 are exact where coarse bins meet.)
    struct Map {
        const float2* line;  // [256] pairs before each coarse bin and in it
        uint32_t dmin;
        float scale, to_bin;
        __device__ __forceinline__ float at(uint64_t v) const { return fminf((float)((uint32_t)(v >> 32) - dmin) * scale, 255.99998f); }
        __device__ __forceinline__ uint32_t bin(uint64_t v) const
        {
            const float a = at(v);
            const float2 l = line[(uint32_t)a];
            return min((uint32_t)(__builtin_fmaf(__builtin_amdgcn_fractf(a), l.y, l.x) * to_bin), (uint32_t)kBins - 1u);
        }
    };

    // Moves the n < 2^24 pairs of `from` to `to`, ordered by bin, and fills `first` and the map; returns the pairs of the fullest
    // bin.  Begins and ends with a barrier.
    __device__ __forceinline__ uint32_t split(const uint64_t* from, uint64_t* to, uint32_t n, Map& map) const
    {
        uint32_t* const cursor = lds;  // [kBins]
        uint32_t* const sums = lds + kBins;  // [2 * kWaves]
        uint32_t* const coarse = lds + kLine;  // [256], then the map's lines
        const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
        uint32_t dmin = 0xFFFFFFFFu, dmax = 0;
        each(from, n, [&](uint64_t v) {
            dmin = min(dmin, (uint32_t)(v >> 32));
            dmax = max(dmax, (uint32_t)(v >> 32));
        });
        dmin = wave_scan(dmin, 0xFFFFFFFFu, [](uint32_t a, uint32_t b) { return min(a, b); });
        dmax = wave_scan(dmax, 0u, [](uint32_t a, uint32_t b) { return max(a, b); });
        __syncthreads();
        reinterpret_cast<uint4*>(cursor)[tid] = make_uint4(0u, 0u, 0u, 0u);
        if (tid < 256) coarse[tid] = 0u;
        if (lane == 63) {
            sums[wave] = dmin;
            sums[kWaves + wave] = dmax;
        }
        __syncthreads();
        dmin = 0xFFFFFFFFu;
        dmax = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            dmin = min(dmin, sums[w]);
            dmax = max(dmax, sums[kWaves + w]);
        }
        map.line = reinterpret_cast<const float2*>(coarse);
        map.dmin = dmin;
        map.scale = 256.0f / ((float)(dmax - dmin) + 1.0f);
        map.to_bin = (float)kBins / (float)n;
        each(from, n, [&](uint64_t v) { atomicAdd(&coarse[(uint32_t)map.at(v)], 1u); });
        __syncthreads();
        uint32_t own = 0, upto = 0;
        if (tid < 256) {  // (wavefronts 0..3)
            own = coarse[tid];
            upto = wave_sum_scan(own);
            if (lane == 63) sums[wave] = upto;
        }
        __syncthreads();
        if (tid < 256) {
            uint32_t before = upto - own;
            for (int w = 0; w < wave; ++w) before += sums[w];
            reinterpret_cast<float2*>(coarse)[tid] = make_float2((float)before, (float)own);
        }
        __syncthreads();
        each(from, n, [&](uint64_t v) { atomicAdd(&cursor[map.bin(v)], 1u); });
        __syncthreads();
        const uint4 mine = reinterpret_cast<const uint4*>(cursor)[tid];
        const uint32_t c = (mine.x + mine.y) + (mine.z + mine.w), inc = wave_sum_scan(c);
        const uint32_t most = wave_scan(max(max(mine.x, mine.y), max(mine.z, mine.w)), 0u, [](uint32_t a, uint32_t b) { return max(a, b); });
        if (lane == 63) {
            sums[wave] = inc;
            sums[kWaves + wave] = most;
        }
        __syncthreads();
        uint32_t f0 = inc - c, fullest = 0;
        for (int w = 0; w < wave; ++w) f0 += sums[w];
#pragma unroll
        for (int w = 0; w < kWaves; ++w) fullest = max(fullest, sums[kWaves + w]);
        const uint32_t f1 = f0 + mine.x, f2 = f1 + mine.y;
        const uint4 firsts = make_uint4(f0, f1, f2, f2 + mine.z);
        reinterpret_cast<uint4*>(cursor)[tid] = firsts;
        reinterpret_cast<uint4*>(first)[tid] = firsts;
        __syncthreads();
        each(from, n, [&](uint64_t v) { to[atomicAdd(&cursor[map.bin(v)], 1u)] = v; });
        __syncthreads();
        return (uint32_t)__builtin_amdgcn_readfirstlane((int)fullest);
    }

    // Writes out the piece [pos, end) of a bucket of n pairs that lie ordered by bin: a pair ranks itself among its bin's, four at a
    // time (what follows a bin is larger than all of it).  Ends with a barrier.
    __device__ __forceinline__ void rank_piece(uint32_t tile, uint32_t lo, uint32_t n, uint32_t pos, uint32_t end, const Map& map, bool keys_too,
                                               uint64_t* out_keys, uint32_t* out_vals) const
    {
        uint64_t* const pairs = reinterpret_cast<uint64_t*>(lds);  // [kCap + 4]
        const uint32_t count = end - pos;
        constexpr int kR = Piece::kCap / kT;
        uint64_t v[kR];
#pragma unroll
        for (int r = 0; r < kR; ++r) v[r] = out_keys[lo + pos + min((uint32_t)(r * kT) + threadIdx.x, count - 1u)];
#pragma unroll
        for (int r = 0; r < kR; ++r)
            if ((uint32_t)(r * kT) + threadIdx.x < count) pairs[r * kT + threadIdx.x] = v[r];
        if (threadIdx.x < 4) pairs[count + threadIdx.x] = ~0ull;
        __syncthreads();
#pragma unroll
        for (int r = 0; r < kR; ++r) {
            if ((uint32_t)(r * kT) + threadIdx.x >= count) continue;
            const uint32_t bin = map.bin(v[r]), stop = (bin + 1u < (uint32_t)kBins ? first[bin + 1u] : n) - pos;
            uint32_t rank = first[bin] - pos;
            for (uint32_t q = rank; q < stop; q += 4) {
#pragma unroll
                for (uint32_t k = 0; k < 4; ++k) rank += pairs[q + k] < v[r] ? 1u : 0u;
            }
            rank += lo + pos;
            if (keys_too) out_keys[rank] = ((uint64_t)tile << 32) | (v[r] >> 32);
            out_vals[rank] = (uint32_t)v[r];
        }
        __syncthreads();
    }

    // Where the piece that starts at `pos` (a bin's first pair, pos < n) ends: behind as many bins as the LDS sorter holds,
    // at least one.
    __device__ __forceinline__ uint32_t piece_end(uint32_t pos, uint32_t n) const
    {
        const uint32_t limit = pos + (uint32_t)Piece::kCap;
        if (n <= limit) return n;
        const int lane = threadIdx.x & 63;
        // the last bin that starts at or before the limit: its 64 bins first (the bins' first pairs do not decrease, the first is 0)
        const int row = __popcll(__ballot(first[lane * 64] <= limit)) - 1;
        const uint32_t v = first[row * 64 + lane];
        const int col = __popcll(__ballot(v <= limit)) - 1;
        const uint32_t end = (uint32_t)__builtin_amdgcn_readlane((int)v, col);
        if (end > pos) return end;
        const int next = row * 64 + col + 1;  // (the bin itself is larger)
        return next < kBins ? first[next] : n;
    }

    __device__ __forceinline__ void run(uint32_t tile, const uint32_t* ranges, uint64_t* buckets, bool keys_too, uint64_t* out_keys,
                                        uint32_t* out_vals) const
    {
        const Piece sorter(lds);
        const uint32_t lo = ranges[2 * tile], n = ranges[2 * tile + 1] - lo;
        const bool whole = n <= (uint32_t)Piece::kCap;
        const bool any_order = n >= (1u << 24);
        Map map;
        uint32_t fullest = 0;
        if (!whole && !any_order) fullest = split(buckets + lo, out_keys + lo, n, map);
        const bool ranked = !whole && !any_order && fullest <= kMaxBin;
        const uint64_t* const from = whole ? buckets : out_keys;
        for (uint32_t pos = 0, end; pos < n; pos = end) {  // (uniform, for all its barriers)
            end = (uint32_t)__builtin_amdgcn_readfirstlane((int)(whole || any_order ? n : piece_end(pos, n)));
            if (ranked) {
                rank_piece(tile, lo, n, pos, end, map, keys_too, out_keys, out_vals);
            } else if (end - pos <= (uint32_t)Piece::kCap) {
                Piece::Fetched f;
                f.tile = tile;
                f.lo = lo + pos;
                f.n = end - pos;
                sorter.fetch_pairs(f, from);
                sorter.sort_fetched(f, keys_too, out_keys, out_vals);
            } else {
                const SortScratch sc = {lds, reinterpret_cast<uint32_t(*)[256]>(lds + 256), lds + 256 + kWaves * 256};
                const GlobalPairs A = {(any_order ? buckets : out_keys) + lo + pos}, B = {(any_order ? out_keys : buckets) + lo + pos};
                const bool in_b = sort_pairs<kT>(A, B, end - pos, sc);
                // (what is rewritten in place is rewritten by the thread that read it)
                write_sorted<kT>(in_b ? B : A, end - pos, tile, keys_too, out_keys + lo + pos, out_vals + lo + pos);
                __syncthreads();
            }
        }
    }
};

__global__ __launch_bounds__(LargeSorter::kT) void tile_sort_large_kernel(const gs355_header* header, const uint32_t* ranges,
                                                                          const uint32_t* list, const uint32_t* list_count,
                                                                          uint64_t* buckets, bool keys_too, uint64_t* out_keys,
                                                                          uint32_t* out_vals)
{
    extern __shared__ uint32_t s_dyn[];
    if (header->overflow) return;
    const uint32_t count = *list_count;
    // Frames without a bucket beyond the LDS sorter's capacity run a loop of their own, in which its registers are those of the LDS
    // sorter alone: with the split beside it 69 of them spill in the place of 44 (337 buckets of 5121 to 10240 pairs among 2170:
    // all sorts 78 us, through the loop below 89).
    if (header->sort_beyond_count == 0u) {
        const LargeSorter::Piece sorter(s_dyn);
        for (uint32_t k = blockIdx.x; k < count; k += gridDim.x) sorter.run(list[k], ranges, buckets, keys_too, out_keys, out_vals);
        return;
    }
    for (uint32_t k = blockIdx.x; k < count; k += gridDim.x) LargeSorter(s_dyn).run(list[k], ranges, buckets, keys_too, out_keys, out_vals);
}

}  // namespace

int bin_groups(int32_t P, int* per_group)
{
    const int per = slice_size(P, kBinMaxGroups);
    *per_group = per;
    const int groups = (P + per - 1) / per;
    return groups < 1 ? 1 : groups;
}

// Dynamic LDS beyond 64 KB has to be allowed per kernel.  The limits are raised once per process and device to
// the largest size any launch can ask for, so that concurrent frames of different image sizes (other streams,
// other threads) never lower the limit under each other.
template <typename K>
static hipError_t raise_lds_limit(K kernel, size_t bytes)
{
    return hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)bytes);
}

static int allow_large_lds()
{
    constexpr int kMaxDevices = 64;
    static std::atomic<int> done[kMaxDevices];
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return set_error(GS355_EHIP, "hipGetDevice: %s", hipGetErrorString(e));
    if (dev < 0 || dev >= kMaxDevices) return set_error(GS355_EINVAL, "device index %d is outside [0, %d)", dev, kMaxDevices);
    if (done[dev].load(std::memory_order_acquire)) return GS355_OK;
    const size_t bin_bytes = (size_t)kBinMaxTiles * sizeof(uint32_t);
    if ((e = raise_lds_limit(tile_count_kernel<false>, bin_bytes)) != hipSuccess ||
        (e = raise_lds_limit(tile_count_kernel<true>, bin_bytes)) != hipSuccess ||
        (e = raise_lds_limit(scatter_kernel<0, false>, bin_bytes)) != hipSuccess ||
        (e = raise_lds_limit(scatter_kernel<kCoarseShift, true>, bin_bytes)) != hipSuccess ||
        (e = raise_lds_limit(tile_sort_list_1024x5_kernel, LdsSorter<1024, 5>::kBytes)) != hipSuccess ||
        (e = raise_lds_limit(tile_sort_each_kernel<1024, 5, false>, LdsSorter<1024, 5>::kBytes)) != hipSuccess ||
        (e = raise_lds_limit(tile_sort_large_kernel, LargeSorter::kBytes)) != hipSuccess)
        return set_error(GS355_EHIP, "LDS limit of the binning / tile sort kernels: %s", hipGetErrorString(e));
    done[dev].store(1, std::memory_order_release);  // racing threads set the same values
    return GS355_OK;
}

static inline int coarse_bins(int tiles) { return (tiles + kCoarseTiles - 1) >> kCoarseShift; }
// the tile_base array: u32[2][tiles], u64[blocks of 64 tiles], u32[coarse bins + 1] chunk bases, u32[blocks] size classes,
// u32[tiles] pairs per tile (up to kBinMaxTiles tiles)
static inline uint64_t* block_totals(uint32_t* tile_base, int tiles) { return reinterpret_cast<uint64_t*>(tile_base + 2 * (size_t)tiles); }
static inline uint32_t* chunk_bases(uint32_t* tile_base, int tiles)
{
    return tile_base + 2 * (size_t)tiles + 2 * (size_t)((tiles + 63) / 64);
}
static inline uint32_t* class_counts(uint32_t* tile_base, int tiles) { return chunk_bases(tile_base, tiles) + coarse_bins(tiles) + 1; }
static inline uint32_t* tile_totals(uint32_t* tile_base, int tiles) { return class_counts(tile_base, tiles) + (tiles + 63) / 64; }

int launch_tile_count(const FrameArgs& f, int32_t P, const uint64_t* rects, const float* records, const uint2* wave_totals,
                      uint32_t* matrix, SliceTotals* slice_totals, hipStream_t s)
{
    int per_group;
    const int groups = bin_groups(P, &per_group);
    const int T = f.grid_x * f.grid_y, n_totals = (int)wave_totals_count(P);
    int rc = allow_large_lds();
    if (rc) return rc;
    if (T <= kBinMaxTiles)
        hipLaunchKernelGGL(tile_count_kernel<false>, dim3(groups), dim3(kBinThreads), (size_t)T * sizeof(uint32_t), s, f,
                           P, per_group, rects, records, wave_totals, n_totals, matrix, slice_totals);
    else
        hipLaunchKernelGGL(tile_count_kernel<true>, dim3(groups), dim3(kBinThreads),
                           (size_t)coarse_bins(T) * sizeof(uint32_t), s, f, P, per_group, rects, records, wave_totals, n_totals,
                           matrix, slice_totals);
    GS355_CHECK_LAUNCH("bin: count");
    return GS355_OK;
}

// Bases of `columns` buckets from their totals (block sums already in `blocks`), and the per-tile outputs with kTiles.
// `bases` may be `totals`, unless `bin_pairs` is `totals` too (workgroup 0 reads every bin's pairs while the others
// already write bases).
template <bool kTiles>
static int launch_layout(const uint32_t* totals, uint32_t* bases, int columns, const uint64_t* blocks,
                         const SliceTotals* slice_totals, int groups, uint32_t n_cap, gs355_header* header,
                         gs355_header* header_copy, bool header_known, uint32_t* ranges, uint32_t* lists, const uint32_t* bin_pairs, int bins,
                         uint32_t* chunk_base, const uint32_t* block_classes, hipStream_t s)
{
    const int n_blocks = (columns + 63) / 64;
    hipLaunchKernelGGL(tile_publish_kernel<kTiles>, dim3((n_blocks + 3) / 4), dim3(256), 0, s, totals, (uint32_t)columns,
                       blocks, (uint32_t)n_blocks, slice_totals, groups, n_cap, header, header_copy, header_known, bases, ranges, lists,
                       bin_pairs, bins, chunk_base, block_classes);
    GS355_CHECK_LAUNCH("bin: layout");
    return GS355_OK;
}

// Up to kBinMaxTiles tiles: everything the later stages need (tile bases, cursors, ranges, size-class lists,
// header).  Beyond: the header and the coarse bins' bases (in tile_cursor[0, bins)); the per-tile layout follows
// in launch_tile_scatter once the pairs of each bin can be counted by tile.  `in_scatter`: the scatter follows in the same
// call and publishes the layout itself (ScatterLayout), where there is one counter per tile.
int launch_tile_layout(int32_t P, uint32_t* matrix, const SliceTotals* slice_totals, int tiles, uint32_t n_cap,
                       gs355_header* header, gs355_header* header_copy, uint32_t* tile_base, uint32_t* ranges, uint32_t* lists,
                       bool in_scatter, hipStream_t s)
{
    int per_group;
    const int groups = bin_groups(P, &per_group);
    uint64_t* blocks = block_totals(tile_base, tiles);
    const int bins = coarse_bins(tiles);
    uint32_t* chunk_base = chunk_bases(tile_base, tiles);
    if (tiles <= kBinMaxTiles) {
        uint32_t* block_classes = class_counts(tile_base, tiles);
        uint32_t* totals = tile_totals(tile_base, tiles);
        // (the pairs of each coarse bin go to chunk_base, which the block scan turns into chunk bases in place)
        hipLaunchKernelGGL(slice_prefix_kernel, dim3((tiles + 63) / 64), dim3(64 * kPrefixParts), 0, s, matrix, groups, tiles,
                           totals, blocks, chunk_base, block_classes, lists);
        GS355_CHECK_LAUNCH("bin: slice prefix");
        if (in_scatter) return GS355_OK;
        return launch_layout<true>(totals, tile_base, tiles, blocks, slice_totals, groups, n_cap, header, header_copy, false, ranges,
                                   lists, chunk_base, bins, chunk_base, block_classes, s);
    }
    // (both in the cursor half of tile_base, which the tile-level layout of launch_tile_scatter overwrites later)
    uint32_t* bin_base = tile_base + tiles;
    uint32_t* bin_pairs = bin_base + bins;
    hipLaunchKernelGGL(slice_prefix_kernel, dim3((bins + 63) / 64), dim3(64 * kPrefixParts), 0, s, matrix, groups, bins, bin_pairs,
                       blocks, (uint32_t*)nullptr, (uint32_t*)nullptr, lists);
    GS355_CHECK_LAUNCH("bin: slice prefix");
    return launch_layout<false>(bin_pairs, bin_base, bins, blocks, slice_totals, groups, n_cap, header, header_copy, false, ranges,
                                lists, bin_pairs, bins, chunk_base, nullptr, s);
}

int launch_tile_scatter(const FrameArgs& f, int32_t P, const uint64_t* rects, const float* records, const uint32_t* depth_bits,
                        gs355_header* header, const uint32_t* matrix, uint32_t n_cap,
                        uint32_t* tile_base, uint32_t* ranges, uint32_t* lists, uint64_t* buckets, uint64_t* coarse,
                        int levels, uint32_t two_from, const ScatterLayout* make, hipStream_t s)
{
    int per_group;
    const int groups = bin_groups(P, &per_group);
    const int T = f.grid_x * f.grid_y, bins = coarse_bins(T);
    uint32_t* tile_cursor = tile_base + T;
    const size_t coarse_lds = (size_t)bins * sizeof(uint32_t);
    int rc = allow_large_lds();
    if (rc) return rc;
    uint32_t min_keys = 0;  // pairs from which the two levels run
    bool fine = true;
    if (T <= kBinMaxTiles) {
        LayoutArgs layout = {};  // (the first launch makes it)
        if (make)
            layout = {tile_totals(tile_base, T), block_totals(tile_base, T), class_counts(tile_base, T), make->slice_totals, n_cap,
                      header, make->header_copy, ranges, lists, chunk_bases(tile_base, T)};
        if (levels != 2) {
            min_keys = levels == 1 ? UINT32_MAX : two_from;
            hipLaunchKernelGGL((scatter_kernel<0, false>), dim3(groups), dim3(kBinThreads), (size_t)T * sizeof(uint32_t), s,
                               f, P, per_group, rects, records, depth_bits, header, 0u, min_keys, matrix, tile_base, buckets, layout);
            GS355_CHECK_LAUNCH("bin: scatter");
            layout.totals = nullptr;
        }
        fine = levels != 1;
        if (fine) {
            hipLaunchKernelGGL((scatter_kernel<kCoarseShift, false>), dim3(groups), dim3(kBinThreads), coarse_lds, s, f, P,
                               per_group, rects, records, depth_bits, header, min_keys, UINT32_MAX, matrix, tile_base, coarse, layout);
            GS355_CHECK_LAUNCH("bin: coarse scatter");
        }
    } else {
        uint32_t* bin_base = tile_cursor;  // (replaced by the tiles' cursors once the coarse level is done)
        hipLaunchKernelGGL((scatter_kernel<kCoarseShift, true>), dim3(groups), dim3(kBinThreads), coarse_lds, s, f, P,
                           per_group, rects, records, depth_bits, header, 0u, UINT32_MAX, matrix, bin_base, coarse, LayoutArgs{});
        GS355_CHECK_LAUNCH("bin: coarse scatter");
        uint64_t* blocks = block_totals(tile_base, T);
        if ((rc = launch_fill_u32(tile_base, (size_t)T, 0u, s))) return rc;
        if ((rc = launch_fill_u32(reinterpret_cast<uint32_t*>(blocks), 2 * (size_t)((T + 63) / 64), 0u, s))) return rc;
        hipLaunchKernelGGL(fine_count_kernel, dim3(kFineGrid), dim3(kFineThreads), 0, s, header, bin_base, bins, T,
                           chunk_bases(tile_base, T), coarse, tile_base, blocks, lists);
        GS355_CHECK_LAUNCH("bin: fine count");
        if ((rc = launch_layout<true>(tile_base, tile_base, T, blocks, (const SliceTotals*)nullptr, groups, n_cap, header, nullptr, true, ranges,
                                      lists, (const uint32_t*)nullptr, 0, (uint32_t*)nullptr, nullptr, s)))
            return rc;
    }
    if (fine) {
        hipLaunchKernelGGL(fine_scatter_kernel, dim3(kFineGrid), dim3(kFineThreads), 0, s, header, min_keys, tile_base,
                           tile_cursor, T, chunk_bases(tile_base, T), coarse, buckets);
        GS355_CHECK_LAUNCH("bin: fine scatter");
    }
    return GS355_OK;
}

// Up to this many tiles the 5120-pair sorter takes the smaller buckets too, all of them side by side in one launch (two
// workgroups of it fit a CU): 10k Gaussians at 256x256, three launches of 7 us each against 8.9 us.  Beyond, buckets of
// small classes hold back too many threads in it: a 2048-pair sorter for the two smallest classes already took 21 us
// against 19 at 2170 tiles, 53 against 24 at 8160.
constexpr int kOneLaunchTiles = 512;

int launch_tile_sort(gs355_header* header, int tiles, const uint32_t* ranges, uint32_t* lists, uint64_t* buckets,
                     uint64_t* out_keys, uint32_t* out_vals, bool keys_too, uint32_t skip_classes, hipStream_t s)
{
    using S0 = LdsSorter<256, 4>;    // <= 1024 pairs, one workgroup per tile
    using S1 = LdsSorter<512, 4>;    // <= 2048
    using S2 = LdsSorter<1024, 5>;   // <= 5120
    using S3 = LargeSorter::Piece;   // <= 10240, and larger ones in pieces
    static_assert(S0::kCap == kTileSortCap[0] && S1::kCap == kTileSortCap[1] && S2::kCap == kTileSortCap[2] &&
                      S3::kCap == kTileSortCap[3], "size classes out of step with the layout kernel");
    int rc;
    if ((rc = allow_large_lds())) return rc;
    const uint32_t* list0 = lists + kListHeader;
    const bool one_launch = tiles <= kOneLaunchTiles;
    uint4* order = tiles >= kOrderMinTiles && tiles <= kOrderMaxTiles ? tile_order(lists, tiles) : nullptr;
    const int each = tiles + (order ? 1 : 0);
    if (one_launch)
        hipLaunchKernelGGL((tile_sort_each_kernel<1024, 5, false>), dim3(each), dim3(1024), S2::kBytes, s, header, ranges, buckets,
                           out_keys, out_vals, keys_too, skip_classes, order, (uint32_t)tiles);
    else
        hipLaunchKernelGGL((tile_sort_each_kernel<256, 4, true>), dim3(each + (tiles + 3) / 4), dim3(256), S0::kBytes, s, header, ranges, buckets,
                           out_keys, out_vals, keys_too, skip_classes, order, (uint32_t)tiles);
    GS355_CHECK_LAUNCH("tile sort: class 0");
    // A launch per larger class, a workgroup per tile: those past the end of the class's list leave at once, which
    // costs nothing measurable (sizing the launch by the list's expected length changed no kernel's time).  The
    // largest class is the exception: a workgroup of it fills a CU, so its launch is the chip's size and strides.
    // (skip_classes: bit c set = the caller expects list c to be empty; the kernel above has sorted what is on it)
    if (!(skip_classes & 1u) && !one_launch) {
        hipLaunchKernelGGL((tile_sort_list_kernel<512, 4>), dim3(tiles), dim3(512), S1::kBytes, s, header, ranges,
                           list0, lists + 0, buckets, keys_too, out_keys, out_vals);
        GS355_CHECK_LAUNCH("tile sort: class 1");
    }
    if (!(skip_classes & 2u) && !one_launch) {
        hipLaunchKernelGGL(tile_sort_list_1024x5_kernel, dim3(tiles), dim3(1024), S2::kBytes, s, header, ranges,
                           list0 + (size_t)tiles, lists + 1, buckets, keys_too, out_keys, out_vals);
        GS355_CHECK_LAUNCH("tile sort: class 2");
    }
    if (!(skip_classes & 4u)) {
        hipLaunchKernelGGL(tile_sort_large_kernel, dim3(tiles < 256 ? tiles : 256), dim3(LargeSorter::kT), LargeSorter::kBytes,
                           s, header, ranges, list0 + 2 * (size_t)tiles, lists + 2, buckets, keys_too, out_keys, out_vals);
        GS355_CHECK_LAUNCH("tile sort: class 3");
    }
    return GS355_OK;
}

}  // namespace gs355
