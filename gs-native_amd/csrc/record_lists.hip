// Per-tile Gaussian lists through a sort of the records: the other way to what tile_lists.hip does from
// the depth order on, for lists whose entries have few records (lists_by_records there).
//   1. tile rectangles gathered in depth order with their record counts, and the counts scanned,
//   2. (tile, id) records emitted in that order, row-major tiles inside each rectangle,
//   3. a stable sort of the records by tile (ceil(log2 T) bits, two passes for T <= 65536),
//   4. each tile's range: where the tile changes.
// Costs about 60 us and 15 to 17 us a million records, whatever the number of Gaussians that have
// none and the size of the screen; bound by the traffic of the records, about 48 bytes each.
#include "gsn_internal.h"

namespace gsn {
namespace {

// A record past the last one that the rectangles hold: sorts behind every tile, is in no list.
constexpr uint32_t kNoTile = 0xffffffffu;

// Record counts and tile rectangles (x0 | x1 << 16, y0 | y1 << 16) in depth order: the one gather by
// Gaussian id. Invisible Gaussians (sorted last, with the key 0xffffffff that no finite depth has)
// get none, and their rectangles, which the projection leaves unwritten, are not read. Clamped to
// the grid, so that rectangles made for another camera cannot lead outside it.
// One kScanBlock-entry block of [0, count] per workgroup: it also sums its counts into
// block_totals[block], the first half of the counts' scan.
constexpr int kOrderThreads = 512;
constexpr int kOrderItems = kScanBlock / kOrderThreads;

__global__ __launch_bounds__(kOrderThreads) void depth_order_counts_kernel(const uint32_t* __restrict__ sorted_ids,
    const uint32_t* __restrict__ sorted_keys, const int4* __restrict__ tile_rects, int* __restrict__ counts,
    uint2* __restrict__ rects, int count, int tiles_x, int tiles_y, int* __restrict__ block_totals) {
    __shared__ int s_wave_sums[kOrderThreads / 64];
    const int t = threadIdx.x;
    const int64_t first = static_cast<int64_t>(blockIdx.x) * kScanBlock + t;
    int4 rect[kOrderItems];
#pragma unroll
    for (int j = 0; j < kOrderItems; ++j) {
        const int64_t k = first + j * kOrderThreads;
        rect[j] = make_int4(0, 0, 0, 0);
        if (k < count && sorted_keys[k] != 0xffffffffu) {
            rect[j] = tile_rects[min(sorted_ids[k], static_cast<uint32_t>(count - 1))];
        }
    }
    int sum = 0;
#pragma unroll
    for (int j = 0; j < kOrderItems; ++j) {
        const int64_t k = first + j * kOrderThreads;
        const int x0 = min(max(rect[j].x, 0), tiles_x), x1 = min(max(rect[j].z, x0), tiles_x);
        const int y0 = min(max(rect[j].y, 0), tiles_y), y1 = min(max(rect[j].w, y0), tiles_y);
        const int records = max(x1 - x0, 0) * max(y1 - y0, 0);
        if (k < count) {
            rects[k] = make_uint2(static_cast<uint32_t>(x0) | static_cast<uint32_t>(x1) << 16,
                static_cast<uint32_t>(y0) | static_cast<uint32_t>(y1) << 16);
        }
        if (k <= count) {
            counts[k] = records;  // zero at `count`
        }
        sum = __builtin_elementwise_add_sat(sum, records);
    }
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) {
        sum = __builtin_elementwise_add_sat(sum, __shfl_xor(sum, offset));
    }
    if ((t & 63) == 0) {
        s_wave_sums[t >> 6] = sum;
    }
    __syncthreads();
    if (t == 0) {
        int total = 0;
#pragma unroll
        for (int w = 0; w < kOrderThreads / 64; ++w) {
            total = __builtin_elementwise_add_sat(total, s_wave_sums[w]);
        }
        block_totals[blockIdx.x] = total;
    }
}

// Records are emitted in blocks of kRadixTile consecutive positions, one workgroup per block, so
// every workgroup writes the same amount whatever the footprints (a near-camera Gaussian can own
// thousands of records, a distant one a single record). A workgroup first needs the Gaussians
// (in depth order) that own its positions: emit_owners_kernel stores, for every block, the
// depth-order index of the Gaussian owning the block's first record, and in entry `blocks` the
// owner of the last record, so block b's owners are the contiguous range [owners[b], owners[b+1]].
// starts[count] is the number of records that the rectangles hold; positions from there on, where
// that is less than record_count, get no tile.
constexpr int kEmitThreads = 512;
constexpr int kEmitItems = kRadixTile / kEmitThreads;
constexpr int kEmitOwners = kRadixTile + 1;

__global__ __launch_bounds__(256) void emit_owners_kernel(const int* __restrict__ starts, int count, int record_count,
    int* __restrict__ owners, int blocks) {
    const int64_t k = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (k >= count) {
        return;
    }
    const int held = min(starts[count], record_count);
    const int64_t begin = starts[k];
    const int64_t end = min(starts[k + 1], held);
    if (end <= begin) {
        return;
    }
    for (int64_t b = (begin + kRadixTile - 1) / kRadixTile; b * kRadixTile < end; ++b) {
        owners[b] = static_cast<int>(k);
    }
    if (end == held) {
        owners[blocks] = static_cast<int>(k);
    }
}

// One workgroup per block of kRadixTile records. Owner data (record start, id, rectangle) is
// staged in LDS, every position is mapped to its owner by a max-scan over the positions where
// owners start, and consecutive lanes then write consecutive records: (row-major tile inside the
// owner's rectangle, Gaussian id). The workgroup also counts the low `digit_bits` bits of its
// tile ids, which is the first pass's histogram of the radix sort that follows (the block is exactly
// one radix tile).
__global__ __launch_bounds__(kEmitThreads) void emit_records_kernel(const uint32_t* __restrict__ sorted_ids,
    const int* __restrict__ starts, const int* __restrict__ owners, const uint2* __restrict__ rects,
    uint32_t* __restrict__ record_tiles, uint32_t* __restrict__ record_ids, int count, int tiles_x, int record_count,
    int blocks, int digit_bits, bool by_tile, int* __restrict__ histogram) {
    __shared__ __align__(16) int s_owner[kRadixTile];
    __shared__ int s_start[kEmitOwners];
    __shared__ uint32_t s_id[kEmitOwners];
    __shared__ uint32_t s_corner[kEmitOwners];  // x0 | y0 << 16
    __shared__ uint16_t s_width[kEmitOwners];
    __shared__ int s_digits[256];
    __shared__ int s_wave_max[kEmitThreads / 64];
    const int t = threadIdx.x;
    const int block = blockIdx.x;
    const int64_t base = static_cast<int64_t>(block) * kRadixTile;
    const int held = min(starts[count], record_count);
    const int valid = static_cast<int>(min(static_cast<int64_t>(kRadixTile), record_count - base));
    const int owned = static_cast<int>(min(max(held - base, int64_t{0}), static_cast<int64_t>(valid)));
    const uint32_t digit_mask = (1u << digit_bits) - 1u;
    if (t < 256) {
        s_digits[t] = 0;
    }
    int first = 0, owner_count = 0;
    if (owned > 0) {
        first = owners[block];
        owner_count = owners[base + kRadixTile < held ? block + 1 : blocks] - first + 1;
    }
    const bool staged = owner_count <= kEmitOwners;
    if (staged) {
        for (int i = t; i < kRadixTile; i += kEmitThreads) {
            s_owner[i] = 0;
        }
        __syncthreads();
        for (int o = t; o < owner_count; o += kEmitThreads) {
            const int k = first + o;
            const int start = starts[k];
            const uint2 rect = rects[k];
            s_start[o] = start;
            s_id[o] = min(sorted_ids[k], static_cast<uint32_t>(count - 1));
            s_corner[o] = (rect.x & 0xffff) | rect.y << 16;
            s_width[o] = static_cast<uint16_t>(max((rect.x >> 16) - (rect.x & 0xffff), 1u));
            const int64_t position = static_cast<int64_t>(start) - base;
            if (position < kRadixTile) {
                // The block's first owner starts at or before the block; later owners start inside
                // it, and of several owners starting at one position (owners without records) the
                // last is the one whose records follow.
                atomicMax(&s_owner[max(position, int64_t{0})], o);
            }
        }
        __syncthreads();
        // Inclusive max-scan over the positions: thread t owns positions [kEmitItems t, kEmitItems (t + 1)).
        static_assert(kEmitItems % 4 == 0, "positions are read as int4");
        int v[kEmitItems];
#pragma unroll
        for (int q = 0; q < kEmitItems / 4; ++q) {
            const int4 quad = *reinterpret_cast<const int4*>(&s_owner[kEmitItems * t + 4 * q]);
            v[4 * q] = quad.x;
            v[4 * q + 1] = quad.y;
            v[4 * q + 2] = quad.z;
            v[4 * q + 3] = quad.w;
        }
#pragma unroll
        for (int i = 1; i < kEmitItems; ++i) {
            v[i] = max(v[i], v[i - 1]);
        }
        const int lane = t & 63;
        const int wave = t >> 6;
        int scan = v[kEmitItems - 1];
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int other = __shfl_up(scan, d);
            scan = lane >= d ? max(scan, other) : scan;
        }
        if (lane == 63) {
            s_wave_max[wave] = scan;
        }
        int carry = __shfl_up(scan, 1);
        if (lane == 0) {
            carry = 0;
        }
        __syncthreads();
        for (int w = 0; w < wave; ++w) {
            carry = max(carry, s_wave_max[w]);
        }
#pragma unroll
        for (int q = 0; q < kEmitItems / 4; ++q) {
            *reinterpret_cast<int4*>(&s_owner[kEmitItems * t + 4 * q]) = make_int4(max(v[4 * q], carry),
                max(v[4 * q + 1], carry), max(v[4 * q + 2], carry), max(v[4 * q + 3], carry));
        }
    }
    __syncthreads();
    for (int p = t; p < valid; p += kEmitThreads) {
        uint32_t tile = kNoTile, id = 0;
        if (p < owned) {
            int local, width;
            uint32_t corner;
            if (staged) {
                const int o = s_owner[p];
                local = static_cast<int>(base + p - s_start[o]);
                width = s_width[o];
                corner = s_corner[o];
                id = s_id[o];
            }
            else {
                // Only reachable when entries without records sit between ones with records (the
                // projection never produces that): the owner by binary search.
                const int r = static_cast<int>(base + p);
                int low = 0, high = count;
                while (high - low > 1) {
                    const int middle = (low + high) >> 1;
                    if (starts[middle] <= r) {
                        low = middle;
                    }
                    else {
                        high = middle;
                    }
                }
                const uint2 rect = rects[low];
                local = r - starts[low];
                width = static_cast<int>(max((rect.x >> 16) - (rect.x & 0xffff), 1u));
                corner = (rect.x & 0xffff) | rect.y << 16;
                id = min(sorted_ids[low], static_cast<uint32_t>(count - 1));
            }
            const int row = local / width;
            const int column = local - row * width;
            tile = ((corner >> 16) + row) * tiles_x + (corner & 0xffffu) + column;
        }
        // Written once and read once by the next sort pass: non-temporal stores keep the 240 MB of
        // records (30M at 1080p) from displacing cached data (emit + tile sort 0.506 -> 0.473 ms).
        __builtin_nontemporal_store(tile, record_tiles + base + p);
        __builtin_nontemporal_store(id, record_ids + base + p);
        atomicAdd(&s_digits[tile & digit_mask], 1);
    }
    __syncthreads();
    if (t < (1 << digit_bits)) {
        histogram[radix_table_index(t, block, blocks, by_tile)] = s_digits[t];
    }
}

// Four records per thread (one 16-byte load when the run is whole): a tile's range starts at
// the first record whose tile differs from its predecessor's.
__global__ __launch_bounds__(256) void tile_ranges_kernel(const uint32_t* __restrict__ sorted_tiles,
    int64_t* __restrict__ offsets, int records, int tile_count) {
    const int64_t first = 4 * (static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x);
    if (first >= records) {
        return;
    }
    uint32_t tiles[4];
    if (first + 4 <= records) {
        const uint4 quad = *reinterpret_cast<const uint4*>(sorted_tiles + first);
        tiles[0] = quad.x;
        tiles[1] = quad.y;
        tiles[2] = quad.z;
        tiles[3] = quad.w;
    }
    else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            tiles[i] = first + i < records ? sorted_tiles[first + i] : kNoTile;
        }
    }
    const uint32_t end = static_cast<uint32_t>(tile_count);
    int previous = first == 0 ? -1 : static_cast<int>(min(sorted_tiles[first - 1], end));
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int64_t r = first + i;
        if (r >= records) {
            break;
        }
        // Records without a tile come last: the first of them is where the lists end.
        const int tile = static_cast<int>(min(tiles[i], end));
        for (int t = previous + 1; t <= tile; ++t) {
            offsets[t] = r;
        }
        previous = tile;
        if (r == records - 1) {
            for (int t = tile + 1; t <= tile_count; ++t) {
                offsets[t] = records;
            }
        }
    }
}

} // namespace

int enqueue_lists_by_records(gsn_context* context, int tiles_x, int tiles_y, int count, const int4* tile_rects,
    int record_count, int* ids, int64_t* offsets) {
    const size_t n = static_cast<size_t>(count);
    const size_t r = static_cast<size_t>(record_count);
    const int tile_count = tiles_x * tiles_y;
    int tile_bits = 1;
    while (tile_bits < 31 && (tile_count - 1) >> tile_bits) {
        ++tile_bits;
    }
    const int blocks = static_cast<int>((static_cast<int64_t>(record_count) + kRadixTile - 1) / kRadixTile);
    const int count_blocks = static_cast<int>((static_cast<int64_t>(count) + kScanBlock) / kScanBlock);  // count + 1 entries
    const uint32_t* sorted_ids = static_cast<uint32_t*>(scratch(context, kSlotDepthSortedIds, n * 4));
    const uint32_t* sorted_keys = static_cast<uint32_t*>(scratch(context, kSlotDepthSortedKeys, n * 4));
    uint2* rects = static_cast<uint2*>(scratch(context, kSlotDepthRects, n * sizeof(uint2)));
    int* starts = static_cast<int*>(scratch(context, kSlotDepthCounts, (n + 1) * 4));
    int* count_totals = static_cast<int*>(scratch(context, kSlotDepthCountTotals, static_cast<size_t>(count_blocks) * 4));
    uint32_t* record_tiles = static_cast<uint32_t*>(scratch(context, kSlotRecordTiles, r * 4));
    uint32_t* record_ids = static_cast<uint32_t*>(scratch(context, kSlotRecordIds, r * 4));
    uint32_t* sorted_tiles = static_cast<uint32_t*>(scratch(context, kSlotSortKeysB, r * 4));
    int* owners = static_cast<int*>(scratch(context, kSlotEmitOwners, (static_cast<size_t>(blocks) + 1) * 4));
    int* histogram = radix_histogram_buffer(context, record_count);
    if (!sorted_ids || !sorted_keys || !rects || !starts || !count_totals || !record_tiles || !record_ids ||
        !sorted_tiles || !owners || !histogram) {
        return GSN_ERROR_OUT_OF_MEMORY;
    }
    hipStream_t stream = context->stream;
    {
        StageScope scope(context, kStageEmit);
        depth_order_counts_kernel<<<count_blocks, kOrderThreads, 0, stream>>>(sorted_ids, sorted_keys, tile_rects, starts,
            rects, count, tiles_x, tiles_y, count_totals);
        GSN_TRY(check_launch("depth_order_counts_kernel"));
        GSN_TRY(exclusive_scan_capped_from_totals(context, starts, starts, static_cast<int64_t>(count) + 1, count_totals));
        emit_owners_kernel<<<grid_for(count, 256), 256, 0, stream>>>(starts, count, record_count, owners, blocks);
        GSN_TRY(check_launch("emit_owners_kernel"));
        emit_records_kernel<<<blocks, kEmitThreads, 0, stream>>>(sorted_ids, starts, owners, rects, record_tiles,
            record_ids, count, tiles_x, record_count, blocks, radix_first_digit_bits(tile_bits),
            radix_table_by_tile(record_count), histogram);
        GSN_TRY(check_launch("emit_records_kernel"));
    }
    {
        StageScope scope(context, kStageTileSort);
        GSN_TRY(radix_sort_pairs(context, record_tiles, record_ids, record_count, tile_bits, sorted_tiles,
            reinterpret_cast<uint32_t*>(ids), true));
    }
    // Writes every entry of offsets[0 .. tiles].
    StageScope scope(context, kStageRanges);
    tile_ranges_kernel<<<grid_for((static_cast<int64_t>(record_count) + 3) / 4, 256), 256, 0, stream>>>(sorted_tiles,
        offsets, record_count, tile_count);
    return check_launch("tile_ranges_kernel");
}

} // namespace gsn
