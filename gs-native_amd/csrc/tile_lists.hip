// Per-tile Gaussian lists in depth order, without sorting the records.
//
// The reference (renderer.cu:223-271, 534-569) writes 64-bit keys (tile << 32 | depth bits)
// for every record in Gaussian-id order and radix-sorts all 32 + ceil(log2 T) key bits over R
// records. Here
//   1. the N visible Gaussians are stably sorted by depth bits (radix_sort.hip),
//   2. their tile rectangles are gathered in that order, once,
//   3. the records per (chunk of the depth-ordered list, tile) are counted: a workgroup takes a chunk
//      and a 32x32-tile part of the screen, adds the four corners of each rectangle to a difference
//      array in LDS and sums that along both axes at the end,
//   4. prefixes over the chunks and over the tiles give every (chunk, tile) its place in the output,
//   5. workgroups of the same shape write the ids there, in list order.
// Every step keeps the order of the list, so a tile's ids are ordered by (depth bits, Gaussian id):
// exactly a stable sort of the reference keys over id-ordered records (each Gaussian has at most
// one record per tile, and equal depth bits keep id order in both).
// Why not a sort: a record then costs 4 bytes written, once, instead of about 48 bytes of traffic
// through the emission of (tile, id) pairs, two radix passes over them and the search for the tiles'
// ranges. What bounds it now: the gather of step 2 (a random line per Gaussian) and step 5 (see
// tile_write_kernel). Emission to ranges with the sort and so: 10K Gaussians at 256x256 45 and 25 us, 200K
// at 979x546 88 and 71, 500K at 1248x832 160 and 114, 3M at 1920x1080 660 and 467, 2M at 3840x2160
// 2,100 and 605.
// Lists with few records per entry and part are sorted after all (lists_by_records).
#include "raster_common.h"

#include <algorithm>

namespace gsn {
namespace {

// One 4096-key radix tile per workgroup (512 threads, eight Gaussians each, k * 512 apart so each
// access stays coalesced; loads issued before the stores). The workgroup also counts its keys'
// low eight bits, the first depth-sort pass's histogram column, so that pass needs no histogram
// kernel.
constexpr int kDepthKeyThreads = 512;
constexpr int kDepthKeyItems = kRadixTile / kDepthKeyThreads;

__global__ __launch_bounds__(kDepthKeyThreads) void depth_keys_kernel(const float* depths, const int* record_offsets,
    uint32_t* keys, uint32_t* ids, int count, int tiles, bool by_tile, int* histogram) {
    __shared__ int s_digits[256];
    const int t = threadIdx.x;
    if (t < 256) {
        s_digits[t] = 0;
    }
    const int64_t first = static_cast<int64_t>(blockIdx.x) * kRadixTile + t;
    float depth[kDepthKeyItems];
    int begin[kDepthKeyItems], end[kDepthKeyItems];
#pragma unroll
    for (int k = 0; k < kDepthKeyItems; ++k) {
        const int64_t i = first + k * kDepthKeyThreads;
        if (i < count) {
            depth[k] = depths[i];
            begin[k] = record_offsets[i];
            end[k] = record_offsets[i + 1];
        }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kDepthKeyItems; ++k) {
        const int64_t i = first + k * kDepthKeyThreads;
        if (i < count) {
            const uint32_t key = end[k] > begin[k] ? float_to_bits(depth[k]) : 0xffffffffu;
            keys[i] = key;
            ids[i] = static_cast<uint32_t>(i);
            atomicAdd(&s_digits[key & 0xffu], 1);
        }
    }
    __syncthreads();
    if (t < 256) {
        histogram[radix_table_index(t, static_cast<int>(blockIdx.x), tiles, by_tile)] = s_digits[t];
    }
}

// The depth order of few Gaussians by counting: a Gaussian's place is the number of keys before its
// own (smaller, or equal with a smaller id). N^2 comparisons, two vector instructions for 64 of them,
// but two launches, where the radix sort's eight to twelve dependent ones of about 5 us each set the
// time. Lists of 4K, 10K, 16K, 20K, 24K and 32K Gaussians in all:
// 66, 73, 73, 75, 77 and 79 us with the radix sort, 31, 40, 46, 64, 68 and 94 us so.
constexpr int kRankCount = 24576;  // most Gaussians ordered this way
constexpr int kRankThreads = 256;
constexpr int kRankRun = kRankThreads;  // keys that a workgroup compares its 256 Gaussians with

__device__ __forceinline__ uint32_t depth_key(const float* depths, const int* record_offsets, int i) {
    return record_offsets[i + 1] > record_offsets[i] ? float_to_bits(depths[i]) : 0xffffffffu;
}

// Many short runs: each is a chain of LDS reads, and the chip needs a few thousand waves to hide it.
__global__ __launch_bounds__(kRankThreads) void depth_rank_kernel(const float* __restrict__ depths,
    const int* __restrict__ record_offsets, int count, int* __restrict__ before) {
    __shared__ __align__(16) uint32_t s_keys[kRankRun];
    const int i = blockIdx.x * kRankThreads + threadIdx.x;
    const int other = blockIdx.y * kRankRun + threadIdx.x;
    const uint32_t own = i < count ? depth_key(depths, record_offsets, i) : 0u;
    // Past the last key: none is before another (equal ones have larger ids).
    s_keys[threadIdx.x] = other < count ? depth_key(depths, record_offsets, other) : 0xffffffffu;
    __syncthreads();
    const uint4* fours = reinterpret_cast<const uint4*>(s_keys);
    int ranked = 0;
    if (blockIdx.y < blockIdx.x) {
        // All ids of the run are smaller: equal keys come before.
#pragma unroll 8
        for (int j = 0; j < kRankRun / 4; ++j) {
            const uint4 k = fours[j];
            ranked += (k.x <= own) + (k.y <= own) + (k.z <= own) + (k.w <= own);
        }
    }
    else if (blockIdx.y > blockIdx.x) {
#pragma unroll 8
        for (int j = 0; j < kRankRun / 4; ++j) {
            const uint4 k = fours[j];
            ranked += (k.x < own) + (k.y < own) + (k.z < own) + (k.w < own);
        }
    }
    else {
        const int self = static_cast<int>(threadIdx.x);
#pragma unroll 8
        for (int j = 0; j < kRankRun / 4; ++j) {
            const uint4 k = fours[j];
            ranked += (k.x < own) + (k.y < own) + (k.z < own) + (k.w < own);
            ranked += (k.x == own && 4 * j < self) + (k.y == own && 4 * j + 1 < self) +
                      (k.z == own && 4 * j + 2 < self) + (k.w == own && 4 * j + 3 < self);
        }
    }
    if (i < count) {
        before[static_cast<int64_t>(blockIdx.y) * count + i] = ranked;
    }
}

__global__ __launch_bounds__(kRankThreads) void depth_rank_scatter_kernel(const float* __restrict__ depths,
    const int* __restrict__ record_offsets, int count, int runs, const int* __restrict__ before,
    uint32_t* __restrict__ sorted_keys, uint32_t* __restrict__ sorted_ids) {
    const int i = blockIdx.x * kRankThreads + threadIdx.x;
    if (i >= count) {
        return;
    }
    int place = 0;
#pragma unroll 16
    for (int run = 0; run < runs; ++run) {
        place += before[static_cast<int64_t>(run) * count + i];
    }
    sorted_keys[place] = depth_key(depths, record_offsets, i);
    sorted_ids[place] = static_cast<uint32_t>(i);
}

// A part of the screen: 32x32 tiles.
constexpr int kPartSide = 32;
constexpr int kPartTiles = kPartSide * kPartSide;
constexpr int kPartThreads = 1024;

// How the screen and the list are cut. Task (chunk, part) is number chunk * parts + part.
struct ScreenGrid {
    int tiles_x, tiles_y;
    int parts_x, parts;
    int chunk, chunks;  // list entries per task
};

// A list entry's tile rectangle in 8 bytes: x0 | x1 << 16, y0 | y1 << 16 (ends exclusive).
__device__ __forceinline__ uint2 pack_rect(int x0, int y0, int x1, int y1) {
    return make_uint2(static_cast<uint32_t>(x0) | static_cast<uint32_t>(x1) << 16,
        static_cast<uint32_t>(y0) | static_cast<uint32_t>(y1) << 16);
}

// Tile rectangles in depth order: the one gather by Gaussian id of the tile lists. Invisible
// Gaussians (sorted last, with the key 0xffffffff that no finite depth has) get an empty one; their
// rectangles, which the projection leaves unwritten, are not read. Clamped to the grid, so that
// rectangles made for another camera cannot lead outside it.
// Bound by the gather (16 random bytes pull a line each): several loads in flight per thread.
constexpr int kGatherThreads = 256;
constexpr int kGatherItems = 4;

__global__ __launch_bounds__(kGatherThreads) void depth_order_rects_kernel(const uint32_t* __restrict__ sorted_ids,
    const uint32_t* __restrict__ sorted_keys, const int4* __restrict__ tile_rects, uint2* __restrict__ rects, int count,
    int tiles_x, int tiles_y) {
    const int64_t first = static_cast<int64_t>(blockIdx.x) * (kGatherThreads * kGatherItems) + threadIdx.x;
    int4 rect[kGatherItems];
#pragma unroll
    for (int j = 0; j < kGatherItems; ++j) {
        const int64_t k = first + j * kGatherThreads;
        rect[j] = make_int4(0, 0, 0, 0);
        if (k < count && sorted_keys[k] != 0xffffffffu) {
            rect[j] = tile_rects[min(sorted_ids[k], static_cast<uint32_t>(count - 1))];
        }
    }
#pragma unroll
    for (int j = 0; j < kGatherItems; ++j) {
        const int64_t k = first + j * kGatherThreads;
        if (k < count) {
            const int x0 = min(max(rect[j].x, 0), tiles_x), x1 = min(max(rect[j].z, 0), tiles_x);
            const int y0 = min(max(rect[j].y, 0), tiles_y), y1 = min(max(rect[j].w, 0), tiles_y);
            rects[k] = x1 > x0 && y1 > y0 ? pack_rect(x0, y0, x1, y1) : make_uint2(0u, 0u);
        }
    }
}

// The chunk and part of task `number`. Tiles are numbered inside the part, 32 y + x.
struct PartTask {
    int64_t begin, end;  // list entries
    int tile_x, tile_y;  // the part's first tile
};

__device__ __forceinline__ PartTask part_task(const ScreenGrid& grid, int number, int count) {
    const int chunk = number / grid.parts;
    const int part = number - chunk * grid.parts;
    PartTask task;
    task.begin = static_cast<int64_t>(chunk) * grid.chunk;
    task.end = min(task.begin + grid.chunk, static_cast<int64_t>(count));
    task.tile_x = part % grid.parts_x * kPartSide;
    task.tile_y = part / grid.parts_x * kPartSide;
    return task;
}

// A rectangle inside the part, ends in [0, 32], one byte each (x0, x1, y0, y1); false when it is
// outside.
__device__ __forceinline__ bool clip_to_part(uint2 rect, const PartTask& task, uint32_t& clipped) {
    const int x0 = static_cast<int>(rect.x & 0xffff) - task.tile_x, x1 = static_cast<int>(rect.x >> 16) - task.tile_x;
    const int y0 = static_cast<int>(rect.y & 0xffff) - task.tile_y, y1 = static_cast<int>(rect.y >> 16) - task.tile_y;
    clipped = static_cast<uint32_t>(max(x0, 0)) | static_cast<uint32_t>(min(x1, kPartSide)) << 8 |
              static_cast<uint32_t>(max(y0, 0)) << 16 | static_cast<uint32_t>(min(y1, kPartSide)) << 24;
    return x0 < kPartSide && x1 > 0 && y0 < kPartSide && y1 > 0;
}

constexpr int kCornerStride = kPartSide + 1;

// The number of the task's entries on the thread's tile of the part, by a whole workgroup of
// kPartThreads. An entry costs about twelve instructions for the test and, where it meets the part,
// four LDS adds, whatever its size; integer sums, so their order does not matter.
__device__ __forceinline__ int count_entries(const uint2* __restrict__ rects, const PartTask& task,
    int (&s_corner)[kCornerStride * kCornerStride]) {
    constexpr int kStride = kCornerStride;
    uint2 next = make_uint2(0u, 0u);
    if (task.begin + threadIdx.x < task.end) {
        next = rects[task.begin + threadIdx.x];
    }
    for (int i = threadIdx.x; i < kStride * kStride; i += kPartThreads) {
        s_corner[i] = 0;
    }
    __syncthreads();
    for (int64_t k = task.begin + threadIdx.x; k < task.end; k += kPartThreads) {
        const uint2 rect = next;
        if (k + kPartThreads < task.end) {
            next = rects[k + kPartThreads];
        }
        uint32_t clipped;
        if (clip_to_part(rect, task, clipped)) {
            const int x0 = clipped & 0xff, x1 = (clipped >> 8) & 0xff, y0 = (clipped >> 16) & 0xff, y1 = clipped >> 24;
            atomicAdd(&s_corner[y0 * kStride + x0], 1);
            atomicAdd(&s_corner[y0 * kStride + x1], -1);
            atomicAdd(&s_corner[y1 * kStride + x0], -1);
            atomicAdd(&s_corner[y1 * kStride + x1], 1);
        }
    }
    __syncthreads();
    // Running sums along x (one thread a row), then along y (one thread a column).
    if (threadIdx.x < kPartSide) {
        int running = 0;
        for (int x = 0; x < kPartSide; ++x) {
            running += s_corner[threadIdx.x * kStride + x];
            s_corner[threadIdx.x * kStride + x] = running;
        }
    }
    __syncthreads();
    if (threadIdx.x < kPartSide) {
        int running = 0;
        for (int y = 0; y < kPartSide; ++y) {
            running += s_corner[y * kStride + threadIdx.x];
            s_corner[y * kStride + threadIdx.x] = running;
        }
    }
    __syncthreads();
    static_assert(kPartThreads == kPartTiles, "one tile per thread");
    return s_corner[(threadIdx.x / kPartSide) * kStride + threadIdx.x % kPartSide];
}

// Step 3.
__global__ __launch_bounds__(kPartThreads) void tile_count_kernel(const uint2* __restrict__ rects, int count,
    ScreenGrid grid, int* __restrict__ counts) {
    __shared__ int s_corner[kCornerStride * kCornerStride];
    const PartTask task = part_task(grid, static_cast<int>(blockIdx.x), count);
    counts[static_cast<int64_t>(blockIdx.x) * kPartTiles + threadIdx.x] = count_entries(rects, task, s_corner);
}

// Step 4, first half: exclusive prefixes of a part's counts over the chunks, in place, and the tiles'
// totals. One workgroup per (part, 64 tiles): 64 tiles x 8 runs of chunks.
__global__ __launch_bounds__(512) void tile_prefix_kernel(int* __restrict__ counts, ScreenGrid grid,
    int* __restrict__ totals) {
    constexpr int kRuns = 8;
    __shared__ int s_sum[kRuns][64];
    const int part = blockIdx.x / (kPartTiles / 64);
    const int tile = (blockIdx.x % (kPartTiles / 64)) * 64 + (threadIdx.x & 63);
    const int run = threadIdx.x >> 6;
    const int rows = (grid.chunks + kRuns - 1) / kRuns;
    const int first = min(run * rows, grid.chunks), last = min(first + rows, grid.chunks);
    int* column = counts + static_cast<int64_t>(part) * kPartTiles + tile;
    const int64_t stride = static_cast<int64_t>(grid.parts) * kPartTiles;
    int sum = 0;
#pragma unroll 8
    for (int chunk = first; chunk < last; ++chunk) {
        sum += column[chunk * stride];
    }
    s_sum[run][threadIdx.x & 63] = sum;
    __syncthreads();
    int running = 0, total = 0;
#pragma unroll
    for (int r = 0; r < kRuns; ++r) {
        const int value = s_sum[r][threadIdx.x & 63];
        running += r < run ? value : 0;
        total += value;
    }
#pragma unroll 8
    for (int chunk = first; chunk < last; ++chunk) {
        const int value = column[chunk * stride];
        column[chunk * stride] = running;
        running += value;
    }
    const int x = part % grid.parts_x * kPartSide + tile % kPartSide, y = part / grid.parts_x * kPartSide + tile / kPartSide;
    if (run == 0 && x < grid.tiles_x && y < grid.tiles_y) {
        totals[y * grid.tiles_x + x] = total;
    }
}

// a + b, 0xffffffff where that is more: sums past 32 bits still compare as more than any record count.
__device__ __forceinline__ uint32_t add_capped(uint32_t a, uint32_t b) {
    return __builtin_elementwise_add_sat(a, b);
}

// Inclusive sums over the lanes of a wave.
__device__ __forceinline__ uint32_t wave_prefix(uint32_t value) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int offset = 1; offset < 64; offset <<= 1) {
        const uint32_t other = __shfl_up(value, offset);
        value = add_capped(value, lane >= offset ? other : 0u);
    }
    return value;
}

// Step 4, second half: offsets[0 .. tiles], the exclusive prefix of the tiles' totals, by one
// workgroup. Bound by latency: eight tiles a thread, the next 8,192 loaded meanwhile, and the results
// go through LDS so that consecutive threads store consecutive entries. Returns the sum.
constexpr int kOffsetItems = 8;
constexpr int kOffsetRound = 1024 * kOffsetItems;

__device__ __forceinline__ uint32_t scan_totals(const int* totals, int tiles, int64_t* offsets,
    uint32_t (&s_out)[kOffsetRound], uint32_t (&s_wave)[16]) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    auto load = [&](int64_t first, uint32_t (&values)[kOffsetItems]) {
#pragma unroll
        for (int i = 0; i < kOffsetItems; ++i) {
            values[i] = first + i < tiles ? totals[first + i] : 0;
        }
    };
    uint32_t carry = 0;
    uint32_t next[kOffsetItems];
    load(threadIdx.x * kOffsetItems, next);
    for (int64_t base = 0; base < tiles; base += kOffsetRound) {
        uint32_t values[kOffsetItems];
        uint32_t sum = 0;
#pragma unroll
        for (int i = 0; i < kOffsetItems; ++i) {
            values[i] = next[i];
            sum = add_capped(sum, values[i]);
        }
        load(base + kOffsetRound + threadIdx.x * kOffsetItems, next);
        const uint32_t inclusive = wave_prefix(sum);
        if (lane == 63) {
            s_wave[wave] = inclusive;
        }
        __syncthreads();  // also ends the reads of the previous round's results
        uint32_t running = carry + inclusive - sum;
#pragma unroll
        for (int w = 0; w < 16; ++w) {
            const uint32_t total = s_wave[w];
            running += w < wave ? total : 0;
            carry = add_capped(carry, total);
        }
#pragma unroll
        for (int i = 0; i < kOffsetItems; ++i) {
            s_out[threadIdx.x * kOffsetItems + i] = running;
            running += values[i];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kOffsetItems; ++i) {
            const int64_t tile = base + i * 1024 + threadIdx.x;
            if (tile < tiles) {
                offsets[tile] = s_out[i * 1024 + threadIdx.x];
            }
        }
    }
    if (threadIdx.x == 0) {
        offsets[tiles] = carry;
    }
    return carry;
}

// The tiles' totals when the rectangles hold more than record_count records (a buffer of fixed
// capacity, or rectangles of another projection): the lists keep the first record_count of them,
// entry by entry, the last one's row by row. The prefixes of the chunk where that ends stay valid;
// what its entries before the end add is counted again. By one workgroup, since no caller whose
// arguments agree gets here.
__device__ __forceinline__ void cut_totals(int* totals, const int* __restrict__ prefixes,
    const uint2* __restrict__ rects, int count, const ScreenGrid& grid, uint32_t record_count,
    int (&s_corner)[kCornerStride * kCornerStride], uint32_t (&s_wave)[16], int& s_last, uint32_t& s_kept) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    uint32_t before = 0;  // records of the entries before this round
    for (int64_t base = 0; base < count && before <= record_count; base += 1024) {
        const int64_t k = base + threadIdx.x;
        const uint2 rect = k < count ? rects[k] : make_uint2(0u, 0u);
        const uint32_t inclusive = wave_prefix(((rect.x >> 16) - (rect.x & 0xffff)) * ((rect.y >> 16) - (rect.y & 0xffff)));
        uint32_t from = __shfl_up(inclusive, 1);
        from = lane == 0 ? 0u : from;
        if (lane == 63) {
            s_wave[wave] = inclusive;
        }
        __syncthreads();
        uint32_t waves_before = before;
        for (int w = 0; w < 16; ++w) {
            waves_before = add_capped(waves_before, w < wave ? s_wave[w] : 0u);
            before = add_capped(before, s_wave[w]);
        }
        from = add_capped(from, waves_before);
        if (from <= record_count && add_capped(inclusive, waves_before) > record_count) {
            s_last = static_cast<int>(k);
            s_kept = record_count - from;
        }
        __syncthreads();
    }
    const int last = s_last;
    const uint2 rect = rects[last];
    const int x0 = rect.x & 0xffff, x1 = rect.x >> 16, y0 = rect.y & 0xffff, y1 = rect.y >> 16;
    const int first_task = last / grid.chunk * grid.parts;
    for (int part = 0; part < grid.parts; ++part) {
        PartTask task = part_task(grid, first_task + part, count);
        task.end = last;
        int total = count_entries(rects, task, s_corner);
        total += prefixes[static_cast<int64_t>(first_task + part) * kPartTiles + threadIdx.x];
        const int x = task.tile_x + static_cast<int>(threadIdx.x) % kPartSide;
        const int y = task.tile_y + static_cast<int>(threadIdx.x) / kPartSide;
        if (x < grid.tiles_x && y < grid.tiles_y) {
            const bool kept = x >= x0 && x < x1 && y >= y0 && y < y1 &&
                              static_cast<uint32_t>(y - y0) * static_cast<uint32_t>(x1 - x0) + (x - x0) < s_kept;
            totals[y * grid.tiles_x + x] = total + kept;
        }
        __syncthreads();
    }
}

// totals[tiles] tells the writing kernel whether the lists were cut.
__global__ __launch_bounds__(1024) void tile_offsets_kernel(int* totals, const int* __restrict__ prefixes,
    const uint2* __restrict__ rects, int count, ScreenGrid grid, int record_count, int64_t* offsets) {
    static_assert(kPartThreads == 1024, "counts with the same workgroup");
    __shared__ uint32_t s_out[kOffsetRound];
    __shared__ int s_corner[kCornerStride * kCornerStride];
    __shared__ uint32_t s_wave[16];
    __shared__ int s_last;
    __shared__ uint32_t s_kept;
    const int tiles = grid.tiles_x * grid.tiles_y;
    const bool cut = scan_totals(totals, tiles, offsets, s_out, s_wave) > static_cast<uint32_t>(record_count);
    if (cut) {
        __syncthreads();
        cut_totals(totals, prefixes, rects, count, grid, static_cast<uint32_t>(record_count), s_corner, s_wave, s_last,
            s_kept);
        scan_totals(totals, tiles, offsets, s_out, s_wave);
    }
    if (threadIdx.x == 0) {
        totals[tiles] = cut;
    }
}

// Step 5. A workgroup of 16 waves per (chunk, part). It first gathers the chunk's entries that meet
// the part in LDS, in order (one test for the whole part instead of one per region); then each wave
// takes an 8x8-tile region of the part and walks that list without further barriers. Entries that
// meet the region wait in a queue until a full wave of them is there. Every tile's set of queued
// entries is a lane mask, the AND of a row's and a column's, and the places of the region's tiles,
// one per lane, advance by its population count.
// What bounds it: the length of a wave's chains (list, queue, masks, stores) and the barriers around
// a workgroup's list, which wait for its busiest region, since splats of one depth crowd together: at
// 3M Gaussians, 1920x1080, its 319 us fill 0.36 of the VALU's issue slots, and a wave waits half its
// time. Half of it are the seven instructions per tile and queue (store_row), a quarter the walk of the
// list and a quarter the gathering (195, 85 and 92 us of 385 with four-byte corners in the list and the
// compiler's selects; without the stores themselves 371). Eight waves a SIMD let two workgroups fit on
// a CU. Dealing out the rows of the regions evenly, with a list per region, took more time (732 against
// 501 us, both before the stores were written out); counters in LDS and a scattered store per record
// 826 us; ids staged per tile in LDS 1,032 us (three waves on a SIMD).
constexpr int kListEntries = 4096;
constexpr int kRegionSide = 8;
constexpr int kRegions = kPartTiles / 64;  // waves of a workgroup

// For every lane the mask of its tile's column (low, high), under one constant lane mask per column:
// three instructions a column where a select takes six.
// The scalar registers named here and in store_row are below the 74 that the compiler gives out at
// eight waves a SIMD. With s76 to s81, which are reserved then (it warns that such need not be
// preserved), the kernel also allocated more of them: 2M Gaussians at 3840x2160 1,328 us a render, 1,282 so.
__device__ __forceinline__ void column_masks(const uint64_t (&column)[8], int& low, int& high) {
#define GSN_COLUMN(low_half, high_half, next) \
    "v_mov_b32 %[low], " low_half "\nv_mov_b32 %[high], " high_half "\n" next
#define GSN_NEXT_COLUMN "s_lshl_b64 exec, exec, 1\n"
    auto half = [&](int i, int part) { return static_cast<uint32_t>(column[i] >> (32 * part)); };
    asm volatile("s_mov_b64 s[64:65], exec\n"
        "s_mov_b32 exec_lo, 0x01010101\n"
        "s_mov_b32 exec_hi, 0x01010101\n"
        GSN_COLUMN("%[l0]", "%[h0]", GSN_NEXT_COLUMN)
        GSN_COLUMN("%[l1]", "%[h1]", GSN_NEXT_COLUMN)
        GSN_COLUMN("%[l2]", "%[h2]", GSN_NEXT_COLUMN)
        GSN_COLUMN("%[l3]", "%[h3]", GSN_NEXT_COLUMN)
        GSN_COLUMN("%[l4]", "%[h4]", GSN_NEXT_COLUMN)
        GSN_COLUMN("%[l5]", "%[h5]", GSN_NEXT_COLUMN)
        GSN_COLUMN("%[l6]", "%[h6]", GSN_NEXT_COLUMN)
        GSN_COLUMN("%[l7]", "%[h7]", "")
        "s_mov_b64 exec, s[64:65]"
        : [low] "+v"(low), [high] "+v"(high)
        : [l0] "s"(half(0, 0)), [h0] "s"(half(0, 1)), [l1] "s"(half(1, 0)), [h1] "s"(half(1, 1)),
        [l2] "s"(half(2, 0)), [h2] "s"(half(2, 1)), [l3] "s"(half(3, 0)), [h3] "s"(half(3, 1)),
        [l4] "s"(half(4, 0)), [h4] "s"(half(4, 1)), [l5] "s"(half(5, 0)), [h5] "s"(half(5, 1)),
        [l6] "s"(half(6, 0)), [h6] "s"(half(6, 1)), [l7] "s"(half(7, 0)), [h7] "s"(half(7, 1))
        : "s64", "s65", "scc");
#undef GSN_COLUMN
#undef GSN_NEXT_COLUMN
}

// Row Row of the region: to each of its eight tiles, the id of the lanes in the row's and the column's
// mask, at the address that the tile's lane holds (low, high), one id per lane below; the row's mask
// to its tiles' lanes. Written out because seven instructions per tile is what the kernel's time is
// made of (the compiler's form took fourteen: a branch around the store and the address in scalar
// arithmetic). Addresses are read one tile ahead: a store may use a scalar register five instructions
// after a lane read wrote it.
template<int Row>
__device__ __forceinline__ void store_row(int low, int high, int id, uint32_t rows, const uint64_t (&column)[8],
    int& row_low, int& row_high) {
    const uint64_t row = lanes_where((rows >> Row & 1) != 0);
    if (row == 0) {
        return;
    }
    int offset;
#define GSN_STORE_TILE(column_mask, now, next)                          \
    "s_and_b64 exec, %[row], " column_mask "\n"                         \
    "v_mbcnt_lo_u32_b32 %[offset], exec_lo, 0\n"                        \
    "v_mbcnt_hi_u32_b32 %[offset], exec_hi, %[offset]\n" next           \
    "v_lshlrev_b32 %[offset], 2, %[offset]\n"                           \
    "global_store_dword %[offset], %[id], s[" now "]\n"
#define GSN_NEXT_TILE(first, second, tile) \
    "v_readlane_b32 s" first ", %[low], " tile "\nv_readlane_b32 s" second ", %[high], " tile "\n"
    asm volatile("s_mov_b64 s[64:65], exec\n"
        "s_mov_b32 exec_lo, %[lanes_low]\n"
        "s_mov_b32 exec_hi, %[lanes_high]\n"
        "v_mov_b32 %[row_low], %[mask_low]\n"
        "v_mov_b32 %[row_high], %[mask_high]\n"
        GSN_NEXT_TILE("60", "61", "%[t0]")
        GSN_STORE_TILE("%[c0]", "60:61", GSN_NEXT_TILE("62", "63", "%[t1]"))
        GSN_STORE_TILE("%[c1]", "62:63", GSN_NEXT_TILE("60", "61", "%[t2]"))
        GSN_STORE_TILE("%[c2]", "60:61", GSN_NEXT_TILE("62", "63", "%[t3]"))
        GSN_STORE_TILE("%[c3]", "62:63", GSN_NEXT_TILE("60", "61", "%[t4]"))
        GSN_STORE_TILE("%[c4]", "60:61", GSN_NEXT_TILE("62", "63", "%[t5]"))
        GSN_STORE_TILE("%[c5]", "62:63", GSN_NEXT_TILE("60", "61", "%[t6]"))
        GSN_STORE_TILE("%[c6]", "60:61", GSN_NEXT_TILE("62", "63", "%[t7]"))
        GSN_STORE_TILE("%[c7]", "62:63", "")
        "s_mov_b64 exec, s[64:65]"
        : [offset] "=&v"(offset), [row_low] "+&v"(row_low), [row_high] "+&v"(row_high)
        : [low] "v"(low), [high] "v"(high), [id] "v"(id), [row] "s"(row), [c0] "s"(column[0]), [c1] "s"(column[1]),
        [c2] "s"(column[2]), [c3] "s"(column[3]), [c4] "s"(column[4]), [c5] "s"(column[5]), [c6] "s"(column[6]),
        [c7] "s"(column[7]), [mask_low] "s"(static_cast<uint32_t>(row)), [mask_high] "s"(static_cast<uint32_t>(row >> 32)),
        [lanes_low] "n"(Row < 4 ? 0xff << (8 * (Row & 3)) : 0), [lanes_high] "n"(Row < 4 ? 0 : 0xff << (8 * (Row & 3))),
        [t0] "n"(8 * Row), [t1] "n"(8 * Row + 1), [t2] "n"(8 * Row + 2), [t3] "n"(8 * Row + 3),
        [t4] "n"(8 * Row + 4), [t5] "n"(8 * Row + 5), [t6] "n"(8 * Row + 6), [t7] "n"(8 * Row + 7)
        : "s60", "s61", "s62", "s63", "s64", "s65", "scc", "memory");
#undef GSN_STORE_TILE
#undef GSN_NEXT_TILE
}

__global__ __launch_bounds__(64 * kRegions, 8) void tile_write_kernel(const uint2* __restrict__ rects,
    const uint32_t* __restrict__ list_ids, int count, ScreenGrid grid, const int* __restrict__ prefixes,
    const int64_t* __restrict__ offsets, const int* __restrict__ cut_flag, int* __restrict__ ids) {
    __shared__ uint32_t s_id[kListEntries];
    __shared__ uint2 s_bits[kListEntries];  // columns and rows of the part, a bit each
    __shared__ uint2 s_queue[kRegions][128];  // id, columns | rows << 8 in the region
    __shared__ int s_hits[kRegions];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int number = static_cast<int>(blockIdx.x);
    const PartTask task = part_task(grid, number, count);
    const int region_x = wave % (kPartSide / kRegionSide) * kRegionSide;
    const int region_y = wave / (kPartSide / kRegionSide) * kRegionSide;
    int place = 0, end = 0;  // of the lane's tile: the next id's place, and the list's end
    {
        const int x = region_x + lane % kRegionSide, y = region_y + lane / kRegionSide;
        if (task.tile_x + x < grid.tiles_x && task.tile_y + y < grid.tiles_y) {
            const int64_t* begin = offsets + static_cast<int64_t>(task.tile_y + y) * grid.tiles_x + task.tile_x + x;
            end = static_cast<int>(begin[1]);
            place = static_cast<int>(min(
                begin[0] + prefixes[static_cast<int64_t>(number) * kPartTiles + y * kPartSide + x], begin[1]));
        }
    }
    // Lists that end before their last entry: every store looks at the end.
    const bool cut = *cut_flag != 0;
    uint2* queue = s_queue[wave];
    int queued = 0;
    for (int64_t batch = task.begin; batch < task.end; batch += kListEntries) {
        const int entries = static_cast<int>(min(task.end - batch, static_cast<int64_t>(kListEntries)));
        // The part's list: each wave takes a run of the batch.
        const int run = ((entries + kRegions - 1) / kRegions + 63) & ~63;
        const int first = wave * run;
        constexpr int kSteps = kListEntries / kRegions / 64;
        uint32_t id[kSteps], clipped[kSteps];
        uint64_t meets[kSteps];
        uint2 rect[kSteps];
#pragma unroll
        for (int j = 0; j < kSteps; ++j) {
            const int e = first + j * 64 + lane;
            const bool exists = j * 64 < run && e < entries;
            rect[j] = exists ? rects[batch + e] : make_uint2(0u, 0u);
            id[j] = exists ? list_ids[batch + e] : 0u;
        }
        int hits = 0;
#pragma unroll
        for (int j = 0; j < kSteps; ++j) {
            meets[j] = lanes_where(clip_to_part(rect[j], task, clipped[j]));
            hits += __popcll(meets[j]);
        }
        if (batch != task.begin) {
            __syncthreads();  // the previous batch's list is done with
        }
        if (lane == 0) {
            s_hits[wave] = hits;
        }
        __syncthreads();
        // Prefix over the waves, in the lanes of a row of sixteen.
        static_assert(kRegions == 16, "a wave's total per lane of a row");
        int hits_to = s_hits[lane & 15];
        hits_to += __builtin_amdgcn_update_dpp(0, hits_to, 0x111, 0xf, 0xf, true);  // row_shr:1
        hits_to += __builtin_amdgcn_update_dpp(0, hits_to, 0x112, 0xf, 0xf, true);
        hits_to += __builtin_amdgcn_update_dpp(0, hits_to, 0x114, 0xf, 0xf, true);
        hits_to += __builtin_amdgcn_update_dpp(0, hits_to, 0x118, 0xf, 0xf, true);
        const int listed = readlane_i(hits_to, 15);
        int at = readlane_i(hits_to, wave) - hits;
#pragma unroll
        for (int j = 0; j < kSteps; ++j) {
            if (in_lanes(meets[j])) {
                const int place_in_list = at + lanes_below(meets[j]);
                const uint32_t x0 = clipped[j] & 0xff, x1 = clipped[j] >> 8 & 0xff;
                const uint32_t y0 = clipped[j] >> 16 & 0xff, y1 = clipped[j] >> 24;
                s_id[place_in_list] = id[j];
                s_bits[place_in_list] = make_uint2(~0u >> (32 - (x1 - x0)) << x0, ~0u >> (32 - (y1 - y0)) << y0);
            }
            at += __popcll(meets[j]);
        }
        __syncthreads();
        const bool last = batch + kListEntries >= task.end;
        int base = 0;
        uint2 next_bits = lane < listed ? s_bits[lane] : make_uint2(0u, 0u);
        uint32_t next_id = s_id[lane];
#pragma unroll 1
        while (true) {
            // 64 entries of the list at a time: those that meet the region join the queue.
#pragma unroll 1
            while (queued < 64 && base < listed) {
                const uint32_t columns = next_bits.x >> region_x & 0xff, rows = next_bits.y >> region_y & 0xff;
                const uint32_t entry_id = next_id;
                base += 64;
                const int e = min(base + lane, kListEntries - 1);
                next_bits = s_bits[e];
                next_id = s_id[e];
                if (base + lane >= listed) {
                    next_bits.x = 0;
                }
                const uint64_t hit = lanes_where(columns != 0) & lanes_where(rows != 0);
                if (in_lanes(hit)) {
                    queue[queued + lanes_below(hit)] = make_uint2(entry_id, columns | rows << kRegionSide);
                }
                queued += __popcll(hit);
            }
            if (queued < 64 && (!last || queued == 0)) {
                break;
            }
            wave_lds_fence();
            if (cut) {
#pragma unroll 1
                for (int q = 0; q < min(queued, 64); ++q) {
                    const uint2 entry = queue[q];
                    if ((entry.y >> (lane % kRegionSide) & entry.y >> (kRegionSide + lane / kRegionSide) & 1) && place < end) {
                        ids[place++] = static_cast<int>(entry.x);
                    }
                }
                const uint2 rest = queue[64 + lane];
                wave_lds_fence();
                queue[lane] = rest;
                queued = max(queued - 64, 0);
                continue;
            }
            const uint2 entry = lane < queued ? queue[lane] : make_uint2(0u, 0u);
            const uint2 rest = queue[64 + lane];
            const int id = static_cast<int>(entry.x);
            const uint32_t columns = entry.y & 0xff, rows = entry.y >> kRegionSide;
            uint64_t column[kRegionSide];
#pragma unroll
            for (int i = 0; i < kRegionSide; ++i) {
                column[i] = lanes_where((columns >> i & 1) != 0);
            }
            int row_low = 0, row_high = 0, column_low = 0, column_high = 0;  // the masks of the lane's tile
            column_masks(column, column_low, column_high);
            const uint64_t to = reinterpret_cast<uint64_t>(ids + place);
            const int low = static_cast<int>(to), high = static_cast<int>(to >> 32);
            store_row<0>(low, high, id, rows, column, row_low, row_high);
            store_row<1>(low, high, id, rows, column, row_low, row_high);
            store_row<2>(low, high, id, rows, column, row_low, row_high);
            store_row<3>(low, high, id, rows, column, row_low, row_high);
            store_row<4>(low, high, id, rows, column, row_low, row_high);
            store_row<5>(low, high, id, rows, column, row_low, row_high);
            store_row<6>(low, high, id, rows, column, row_low, row_high);
            store_row<7>(low, high, id, rows, column, row_low, row_high);
            place += __popc(static_cast<uint32_t>(row_low & column_low)) +
                     __popc(static_cast<uint32_t>(row_high & column_high));
            wave_lds_fence();
            queue[lane] = rest;
            queued = max(queued - 64, 0);
        }
    }
}

// The reference's sort keys of the finished lists (optional output): a record's tile is the last one
// that begins at or before it. All ones past the last list's end, where no id was written.
__global__ __launch_bounds__(256) void sorted_keys_kernel(const int64_t* __restrict__ offsets, int tiles,
    const int* __restrict__ ids, const float* __restrict__ depths, uint64_t* __restrict__ keys, int records) {
    int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= records) {
        return;
    }
    if (r >= offsets[tiles]) {
        keys[r] = ~0ull;
        return;
    }
    int low = 0, high = tiles;
    while (high - low > 1) {
        const int middle = (low + high) >> 1;
        if (offsets[middle] <= r) {
            low = middle;
        }
        else {
            high = middle;
        }
    }
    keys[r] = (static_cast<uint64_t>(static_cast<uint32_t>(low)) << 32) | float_to_bits(depths[ids[r]]);
}

__global__ void zero_offsets_kernel(int64_t* offsets, int entries) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < entries) {
        offsets[i] = 0;
    }
}

} // namespace

// Chunks: at least about 2,048 tasks, so that short lists still spread over the CUs (200K Gaussians at
// 979x546, chunks of 512 and 256: writing 50 and 70 us, counting 9 and 16; 500K at 1248x832, 2,048 and
// 1,024: writing 88 and 87, counting and prefixes 19 and 29), up to 8,192 entries, where counts and
// prefixes have become short (2M at 3840x2160, 4,096, 8,192 and 16,384: all three kernels 690, 623 and
// 654 us; 3M at 1920x1080: 459, 473 and 562). Longer ones only where the counts would exceed 65,536
// tasks of 4 KB.
static ScreenGrid screen_grid(int count, int tiles_x, int tiles_y) {
    ScreenGrid grid{};
    grid.tiles_x = tiles_x;
    grid.tiles_y = tiles_y;
    grid.parts_x = (tiles_x + kPartSide - 1) / kPartSide;
    grid.parts = grid.parts_x * ((tiles_y + kPartSide - 1) / kPartSide);
    const int64_t work = static_cast<int64_t>(count) * grid.parts;
    int64_t chunk = 256;
    while (chunk < count && ((chunk < 8192 && chunk * 2048 < work) || chunk * 65536 < work)) {
        chunk *= 2;
    }
    grid.chunk = static_cast<int>(std::min<int64_t>(chunk, 1 << 30));
    grid.chunks = static_cast<int>((static_cast<int64_t>(count) + grid.chunk - 1) / grid.chunk);
    return grid;
}

// Whether sorting the records (record_lists.hip) is the shorter way: its cost goes with the records,
// that of counting and writing with the tests of every list entry against every part, which are many
// where most Gaussians are culled or cover a tile or two of a large screen. Of 165 lists of 0.2M to 6M
// Gaussians at 1248x832 to 5187x3361 the sort is the shorter way below 0.2 records per test and the
// longer one above 0.38; between, it depends on how many are visible, which is not known here. In all, by
// records and by counting: 3M at 1920x1080, 5% visible, 0.7M records 69 and 131 us, 30% 8M 168 and 173,
// all 27M 443 and 303; 2M at 3840x2160, 5% 0.9M 69 and 244, all 18M 323 and 406, all 30M 526 and 409; 4M at
// 5187x3361, 5% 1.8M 104 and 798. Below 4M tests (0.3M at 1920x1080, 5%: 47 and 51 us) counting's fewer
// launches decide.
static bool lists_by_records(const ScreenGrid& grid, int count, int record_count) {
    const int64_t tests = static_cast<int64_t>(count) * grid.parts;
    return tests > 4'000'000 && 4 * static_cast<int64_t>(record_count) < tests;
}

// The lists, from the depth order: steps 2 to 5.
static int enqueue_lists(gsn_context* context, const ScreenGrid& grid, int count, const int4* tile_rects,
    int record_count, int* ids, int64_t* offsets) {
    const size_t n = static_cast<size_t>(count);
    const size_t tile_count = static_cast<size_t>(grid.tiles_x) * grid.tiles_y;
    const int64_t tasks = static_cast<int64_t>(grid.chunks) * grid.parts;
    const uint32_t* sorted_ids = static_cast<uint32_t*>(scratch(context, kSlotDepthSortedIds, n * 4));
    const uint32_t* sorted_keys = static_cast<uint32_t*>(scratch(context, kSlotDepthSortedKeys, n * 4));
    uint2* rects = static_cast<uint2*>(scratch(context, kSlotDepthRects, n * sizeof(uint2)));
    int* counts = static_cast<int*>(scratch(context, kSlotTileCounts, static_cast<size_t>(tasks) * kPartTiles * 4));
    int* totals = static_cast<int*>(scratch(context, kSlotTileTotals, (tile_count + 1) * 4));
    if (!sorted_ids || !sorted_keys || !rects || !counts || !totals) {
        return GSN_ERROR_OUT_OF_MEMORY;
    }
    hipStream_t stream = context->stream;
    {
        StageScope scope(context, kStageEmit);
        depth_order_rects_kernel<<<grid_for(count, kGatherThreads * kGatherItems), kGatherThreads, 0, stream>>>(
            sorted_ids, sorted_keys, tile_rects, rects, count, grid.tiles_x, grid.tiles_y);
        GSN_TRY(check_launch("depth_order_rects_kernel"));
    }
    {
        StageScope scope(context, kStageRanges);
        tile_count_kernel<<<static_cast<unsigned>(tasks), kPartThreads, 0, stream>>>(rects, count, grid, counts);
        GSN_TRY(check_launch("tile_count_kernel"));
        tile_prefix_kernel<<<static_cast<unsigned>(grid.parts * (kPartTiles / 64)), 512, 0, stream>>>(counts, grid, totals);
        GSN_TRY(check_launch("tile_prefix_kernel"));
        tile_offsets_kernel<<<1, 1024, 0, stream>>>(totals, counts, rects, count, grid, record_count, offsets);
        GSN_TRY(check_launch("tile_offsets_kernel"));
    }
    StageScope scope(context, kStageTileSort);
    tile_write_kernel<<<static_cast<unsigned>(tasks), 64 * kRegions, 0, stream>>>(rects, sorted_ids, count, grid,
        counts, offsets, totals + tile_count, ids);
    return check_launch("tile_write_kernel");
}

// Stable order of the N Gaussians by depth bits (visible ones first) into the depth-order slots:
// sorted ids and sorted keys.
int enqueue_depth_order(gsn_context* context, const float* depths, const int* record_offsets, int count) {
    size_t n = static_cast<size_t>(count);
    uint32_t* sorted_ids = static_cast<uint32_t*>(scratch(context, kSlotDepthSortedIds, n * 4));
    uint32_t* sorted_keys = static_cast<uint32_t*>(scratch(context, kSlotDepthSortedKeys, n * 4));
    if (count <= kRankCount) {
        const unsigned groups = grid_for(count, kRankThreads), runs = grid_for(count, kRankRun);
        int* before = static_cast<int*>(scratch(context, kSlotDepthKeys, n * runs * 4));
        if (!sorted_ids || !sorted_keys || !before) {
            return GSN_ERROR_OUT_OF_MEMORY;
        }
        StageScope scope(context, kStageDepthSort);
        depth_rank_kernel<<<dim3(groups, runs), kRankThreads, 0, context->stream>>>(depths, record_offsets, count,
            before);
        GSN_TRY(check_launch("depth_rank_kernel"));
        depth_rank_scatter_kernel<<<groups, kRankThreads, 0, context->stream>>>(depths, record_offsets, count,
            static_cast<int>(runs), before, sorted_keys, sorted_ids);
        return check_launch("depth_rank_scatter_kernel");
    }
    uint32_t* depth_keys = static_cast<uint32_t*>(scratch(context, kSlotDepthKeys, n * 4));
    uint32_t* depth_ids = static_cast<uint32_t*>(scratch(context, kSlotDepthIds, n * 4));
    if (!depth_keys || !depth_ids || !sorted_ids || !sorted_keys) {
        return GSN_ERROR_OUT_OF_MEMORY;
    }
    int* histogram = radix_histogram_buffer(context, count);
    if (!histogram) {
        return GSN_ERROR_OUT_OF_MEMORY;
    }
    static_assert(kDepthKeyThreads * kDepthKeyItems == kRadixTile, "one radix tile per workgroup");
    const int tiles = static_cast<int>((static_cast<int64_t>(count) + kRadixTile - 1) / kRadixTile);
    StageScope scope(context, kStageDepthSort);
    // 32 key bits: the first pass takes radix_first_digit_bits(32) = 8 bits, the low byte counted here.
    depth_keys_kernel<<<tiles, kDepthKeyThreads, 0, context->stream>>>(depths, record_offsets, depth_keys, depth_ids,
        count, tiles, radix_table_by_tile(count), histogram);
    GSN_TRY(check_launch("depth_keys_kernel"));
    return radix_sort_pairs(context, depth_keys, depth_ids, count, 32, sorted_keys, sorted_ids, true);
}

} // namespace gsn

extern "C" int gsn_scan_record_offsets(gsn_context* context, int* record_offsets, int count, int* record_count) {
    using namespace gsn;
    if (!context || !record_offsets || count < 0 || count == 0x7fffffff || !record_count) {
        return fail(GSN_ERROR_INVALID_ARGUMENT, "gsn_scan_record_offsets: invalid arguments");
    }
    {
        StageScope scope(context, kStageScan);
        GSN_TRY(exclusive_scan_int(context, record_offsets, record_offsets, static_cast<int64_t>(count) + 1));
    }
    int* pinned = static_cast<int*>(context->pinned);
    GSN_HIP(hipMemcpyAsync(pinned, record_offsets + count, sizeof(int), hipMemcpyDeviceToHost, context->stream));
    GSN_HIP(hipEventRecord(context->readback_event, context->stream));
    // The depth order of the last projection does not need R: queue it behind the copy, so the
    // GPU sorts while the caller reads R and queues the kernels that do.
    const bool prepare = count > 0 && context->projected_depths && context->projected_offsets == record_offsets &&
                         context->projected_count == count;
    const float* depths = context->projected_depths;
    context->projected_depths = nullptr;
    context->projected_offsets = nullptr;
    context->projected_count = -1;
    if (prepare) {
        GSN_TRY(enqueue_depth_order(context, depths, record_offsets, count));
        context->ordered_depths = depths;
        context->ordered_offsets = record_offsets;
        context->ordered_count = count;
    }
    GSN_HIP(hipEventSynchronize(context->readback_event));
    *record_count = pinned[0];
    if (*record_count < 0) {
        return fail(GSN_ERROR_CAPACITY, "gsn_scan_record_offsets: record count overflowed int32");
    }
    return GSN_OK;
}

extern "C" int gsn_build_tile_lists(gsn_context* context, const gsn_camera* camera, int count, const int* tile_rects,
    const float* depths, const int* record_offsets, int record_count, int* tile_gaussian_ids, int64_t* tile_offsets,
    uint64_t* sorted_keys) {
    using namespace gsn;
    if (!context || !camera || count < 0 || record_count < 0 || !tile_offsets || !record_offsets) {
        return fail(GSN_ERROR_INVALID_ARGUMENT, "gsn_build_tile_lists: invalid arguments");
    }
    int64_t tile_count_long = static_cast<int64_t>(camera->tile_count_x) * camera->tile_count_y;
    if (camera->tile_count_x <= 0 || camera->tile_count_y <= 0 || tile_count_long >= 0x7fffffff) {
        return fail(GSN_ERROR_INVALID_ARGUMENT, "gsn_build_tile_lists: invalid tile grid");
    }
    if (camera->tile_count_x > 0xffff || camera->tile_count_y > 0xffff) {
        return fail(GSN_ERROR_CAPACITY, "gsn_build_tile_lists: more than 65535 tiles along an axis");
    }
    int tile_count = static_cast<int>(tile_count_long);
    hipStream_t stream = context->stream;
    if (record_count == 0 || count == 0) {
        zero_offsets_kernel<<<grid_for(tile_count + 1, 256), 256, 0, stream>>>(tile_offsets, tile_count + 1);
        return check_launch("zero_offsets_kernel");
    }
    if (!tile_rects || !depths || !tile_gaussian_ids) {
        return fail(GSN_ERROR_INVALID_ARGUMENT, "gsn_build_tile_lists: null buffer");
    }
    const bool ordered = context->ordered_depths == depths && context->ordered_offsets == record_offsets &&
                         context->ordered_count == count;
    context->ordered_depths = nullptr;
    context->ordered_offsets = nullptr;
    context->ordered_count = -1;
    if (!ordered) {
        GSN_TRY(enqueue_depth_order(context, depths, record_offsets, count));
    }
    const ScreenGrid grid = screen_grid(count, camera->tile_count_x, camera->tile_count_y);
    const int4* rects = reinterpret_cast<const int4*>(tile_rects);
    GSN_TRY(lists_by_records(grid, count, record_count)
                ? enqueue_lists_by_records(context, grid.tiles_x, grid.tiles_y, count, rects, record_count, tile_gaussian_ids,
                      tile_offsets)
                : enqueue_lists(context, grid, count, rects, record_count, tile_gaussian_ids, tile_offsets));
    if (sorted_keys) {
        sorted_keys_kernel<<<grid_for(record_count, 256), 256, 0, stream>>>(tile_offsets, tile_count, tile_gaussian_ids,
            depths, sorted_keys, record_count);
        GSN_TRY(check_launch("sorted_keys_kernel"));
    }
    return GSN_OK;
}
