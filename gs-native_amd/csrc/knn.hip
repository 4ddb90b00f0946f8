// Three nearest neighbours of every point through a bounding-volume hierarchy over Morton-ordered
// points (reference src/core/knn/knn.cu).
//
//   1. bounding box (block min/max, finished by every workgroup of the next kernel),
//   2. 30-bit Morton code of each point over the box (10 bits per axis), stable radix sort,
//   3. points gathered into Morton order; axis-aligned boxes of each 8 consecutive points (the
//      leaves) and of each 8 consecutive boxes of the level below,
//   4. eight lanes search for one point, from its own leaf upwards: they test the eight children of a
//      node together, go on with the nearest and leave the others, with their distances, on a stack
//      in LDS; a leaf's eight points are tested the same way. When nothing waits, the next ancestor's
//      other children follow. A box is left out only when its lower bound is strictly greater than
//      the current third-best distance.
// What bounds it: the latency of the walk's dependent loads, hidden by eight searches per wave and
// the waves of a SIMD. One thread per point with a stack of its own took the same walk with a
// different node in every lane and its stack in scratch memory; a wave walking for 64 points at once
// tested nearly every block, since the sparsest of its points set the reach of all. 200,000 points
// of 64 blobs: the search 1,473 us (thread per point), 917 (wave per 64 points), 317 (eight lanes,
// from the root down: about 40 nodes and leaves a point), 237 (so). Letting the searches of a wave
// wait for each other at their leaves was slower (389 against 318, from the root down). The bounds
// of the points, reduced by one thread per workgroup 32 us, by all 5.
// Candidates are ordered by (squared distance, original index), so the three neighbours are
// unique even with duplicate points and equal the exhaustive search with the same tie rule.
// Squared distances are (dx*dx + dy*dy) + dz*dz with FP contraction off, as in the host
// restatement. Box lower bounds use the same operation order on per-axis gaps, and FP rounding
// is monotonic, so a box bound never exceeds the distance to any point inside it; a NaN gap counts
// as none.
#include "raster_common.h"

namespace gsn {
namespace {

// Children of a node (a leaf's are points), and the children of its children.
constexpr int kFanBits = 3;
constexpr int kFan = 1 << kFanBits;
constexpr int kFan2 = kFan * kFan;
// Levels of boxes of 2^31 points (level 0 = leaves), the root's children being the last of at most
// kFan boxes.
constexpr int kMaxLevels = 11;

struct Box {
    float4 lower;  // xyz, w unused
    float4 upper;
};

__device__ __forceinline__ float ordered_min(float a, float b) {
    return a < b ? a : b;
}

__device__ __forceinline__ float ordered_max(float a, float b) {
    return a > b ? a : b;
}

__global__ __launch_bounds__(256) void knn_bounds_kernel(const float* points, int n, float* block_bounds) {
    __shared__ float s[6][256];
    int t = threadIdx.x;
    float lo[3] = {3.0e38f, 3.0e38f, 3.0e38f};
    float hi[3] = {-3.0e38f, -3.0e38f, -3.0e38f};
    for (int i = blockIdx.x * blockDim.x + t; i < n; i += gridDim.x * blockDim.x) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            float v = points[3ll * i + a];
            lo[a] = ordered_min(lo[a], v);
            hi[a] = ordered_max(hi[a], v);
        }
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        s[a][t] = lo[a];
        s[3 + a][t] = hi[a];
    }
    __syncthreads();
    for (int stride = 128; stride > 0; stride >>= 1) {
        if (t < stride) {
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                s[a][t] = ordered_min(s[a][t], s[a][t + stride]);
                s[3 + a][t] = ordered_max(s[3 + a][t], s[3 + a][t + stride]);
            }
        }
        __syncthreads();
    }
    if (t < 6) {
        block_bounds[blockIdx.x * 6 + t] = s[t][0];
    }
}

__global__ __launch_bounds__(256) void knn_morton_kernel(const float* points, int n, const float* block_bounds,
    int bound_blocks, uint32_t* keys, uint32_t* ids) {
    // The bounds of the (at most 256) blocks, one per thread, reduced by the workgroup.
    __shared__ float wave_bounds[4][6];
    __shared__ float bounds[6];
    const int from = min(static_cast<int>(threadIdx.x), bound_blocks - 1);
    float v[6];
#pragma unroll
    for (int a = 0; a < 6; ++a) {
        v[a] = block_bounds[from * 6 + a];
    }
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) {
#pragma unroll
        for (int a = 0; a < 6; ++a) {
            const float w = __shfl_xor(v[a], offset);
            v[a] = a < 3 ? ordered_min(v[a], w) : ordered_max(v[a], w);
        }
    }
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int a = 0; a < 6; ++a) {
            wave_bounds[threadIdx.x >> 6][a] = v[a];
        }
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        float all = wave_bounds[0][threadIdx.x];
        for (int w = 1; w < 4; ++w) {
            const float other = wave_bounds[w][threadIdx.x];
            all = threadIdx.x < 3 ? ordered_min(all, other) : ordered_max(all, other);
        }
        bounds[threadIdx.x] = all;
    }
    __syncthreads();
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) {
        return;
    }
    uint32_t key = 0;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        float extent = bounds[3 + a] - bounds[a];
        float scaled = extent > 0.0f ? (points[3ll * i + a] - bounds[a]) / extent * 1023.0f : 0.0f;
        uint32_t q = static_cast<uint32_t>(fminf(fmaxf(scaled, 0.0f), 1023.0f));
        for (int bit = 0; bit < 10; ++bit) {
            key |= ((q >> bit) & 1u) << (3 * bit + a);
        }
    }
    keys[i] = key;
    ids[i] = static_cast<uint32_t>(i);
}

// Smallest and largest of a value over the aligned group of `lanes` lanes around this one (fminf and
// fmaxf pass over NaN).
template<int Lanes>
__device__ __forceinline__ void group_bounds(float value, float& low, float& high) {
    low = value;
    high = value;
#pragma unroll
    for (int offset = 1; offset < Lanes; offset <<= 1) {
        low = fminf(low, __shfl_xor(low, offset));
        high = fmaxf(high, __shfl_xor(high, offset));
    }
}

// Points in Morton order, padded to whole 64s with NaN points (at no distance from any other), and
// the boxes of each 8 and each 64 of them. Lanes past the last point repeat it for the boxes, which
// leaves those as they are.
__global__ __launch_bounds__(256) void knn_leaves_kernel(const float* __restrict__ points,
    const uint32_t* __restrict__ order, int n, float4* __restrict__ sorted, Box* __restrict__ leaves,
    Box* __restrict__ parents) {
    const int64_t k = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if ((k & ~static_cast<int64_t>(63)) >= n) {
        return;  // whole waves
    }
    const int i = static_cast<int>(order[min(k, static_cast<int64_t>(n) - 1)]);
    const float3 p = make_float3(points[3ll * i], points[3ll * i + 1], points[3ll * i + 2]);
    const float nan = __int_as_float(0x7fc00000);
    sorted[k] = k < n ? make_float4(p.x, p.y, p.z, __int_as_float(i)) : make_float4(nan, nan, nan, __int_as_float(-1));
    Box leaf, parent;
    group_bounds<kFan>(p.x, leaf.lower.x, leaf.upper.x);
    group_bounds<kFan>(p.y, leaf.lower.y, leaf.upper.y);
    group_bounds<kFan>(p.z, leaf.lower.z, leaf.upper.z);
    group_bounds<kFan2>(p.x, parent.lower.x, parent.upper.x);
    group_bounds<kFan2>(p.y, parent.lower.y, parent.upper.y);
    group_bounds<kFan2>(p.z, parent.lower.z, parent.upper.z);
    leaf.lower.w = leaf.upper.w = parent.lower.w = parent.upper.w = 0.0f;
    if (k % kFan == 0 && k < n) {
        leaves[k / kFan] = leaf;
    }
    if (k % kFan2 == 0) {
        parents[k / kFan2] = parent;
    }
}

// The two levels above `count` boxes: those of each 8 and of each 64.
__global__ __launch_bounds__(256) void knn_parents_kernel(const Box* __restrict__ children, int count,
    Box* __restrict__ parents, Box* __restrict__ grandparents) {
    const int64_t child = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if ((child & ~static_cast<int64_t>(63)) >= count) {
        return;
    }
    Box box = children[min(child, static_cast<int64_t>(count) - 1)];
#pragma unroll
    for (int offset = 1; offset < kFan2; offset <<= 1) {
        box.lower.x = fminf(box.lower.x, __shfl_xor(box.lower.x, offset));
        box.lower.y = fminf(box.lower.y, __shfl_xor(box.lower.y, offset));
        box.lower.z = fminf(box.lower.z, __shfl_xor(box.lower.z, offset));
        box.upper.x = fmaxf(box.upper.x, __shfl_xor(box.upper.x, offset));
        box.upper.y = fmaxf(box.upper.y, __shfl_xor(box.upper.y, offset));
        box.upper.z = fmaxf(box.upper.z, __shfl_xor(box.upper.z, offset));
        if (2 * offset == kFan && child % kFan == 0 && child < count) {
            parents[child / kFan] = box;
        }
    }
    if (child % kFan2 == 0) {
        grandparents[child / kFan2] = box;
    }
}

__device__ __forceinline__ float box_distance(float4 p, const Box& box) {
#pragma clang fp contract(off)
    float gx = fmaxf(fmaxf(box.lower.x - p.x, p.x - box.upper.x), 0.0f);
    float gy = fmaxf(fmaxf(box.lower.y - p.y, p.y - box.upper.y), 0.0f);
    float gz = fmaxf(fmaxf(box.lower.z - p.z, p.z - box.upper.z), 0.0f);
    return gx * gx + gy * gy + gz * gz;
}

__device__ __forceinline__ float point_distance(float4 p, float4 q) {
#pragma clang fp contract(off)
    float dx = p.x - q.x;
    float dy = p.y - q.y;
    float dz = p.z - q.z;
    return dx * dx + dy * dy + dz * dz;
}

__device__ __forceinline__ bool before(float d, int i, float bd, int bi) {
    return d < bd || (d == bd && i < bi);
}

// A search's three best candidates so far, nearest first.
struct Nearest {
    float d0, d1, d2;
    int i0, i1, i2;
};

__device__ __forceinline__ void consider(Nearest& best, float d, int id) {
    const bool third = before(d, id, best.d2, best.i2);
    const bool second = before(d, id, best.d1, best.i1);
    const bool first = before(d, id, best.d0, best.i0);
    best.d2 = second ? best.d1 : (third ? d : best.d2);
    best.i2 = second ? best.i1 : (third ? id : best.i2);
    best.d1 = first ? best.d0 : (second ? d : best.d1);
    best.i1 = first ? best.i0 : (second ? id : best.i1);
    best.d0 = first ? d : best.d0;
    best.i0 = first ? id : best.i0;
}

// The levels of boxes in one array: level L has counts[L] boxes from offsets[L] on.
struct Levels {
    int offsets[kMaxLevels];
    int counts[kMaxLevels];
    int top;  // the level of the root's children
};

// A node on the stack: its level above 28 bits of number, and its distance.
struct Waiting {
    uint32_t node;
    float distance;
};
constexpr int kNodeBits = 28;
// The root's children and then seven a level can wait at once.
constexpr int kStack = kFan * kMaxLevels;
// Waves of a workgroup, which ends with its longest search: 328 us with four, 317 with two, 318 with
// one (200,000 points, from the root down).
constexpr int kQueryWaves = 2;

// The value of another lane of the aligned eight: across pairs, across halves of four (mirrored) or
// the other four (mirrored).
constexpr int kDppPairs = 0xb1;    // quad_perm:[1,0,3,2]
constexpr int kDppHalves = 0x4e;   // quad_perm:[2,3,0,1]
constexpr int kDppMirror = 0x141;  // row_half_mirror
template<int Control>
__device__ __forceinline__ int of_eight(int v) {
    return __builtin_amdgcn_update_dpp(0, v, Control, 0xf, 0xf, true);
}

template<int Control>
__device__ __forceinline__ float of_eight(float v) {
    return __int_as_float(of_eight<Control>(__float_as_int(v)));
}

// The smallest of the eight lanes' values (no NaN), in all of them.
template<class T>
__device__ __forceinline__ T smallest_of_eight(T v) {
    v = min(v, of_eight<kDppPairs>(v));
    v = min(v, of_eight<kDppHalves>(v));
    return min(v, of_eight<kDppMirror>(v));
}

__global__ __launch_bounds__(64 * kQueryWaves) void knn_query_kernel(const float4* __restrict__ sorted,
    const Box* __restrict__ boxes, int n, Levels levels, int* __restrict__ neighbors, float* __restrict__ mean_dist2) {
#pragma clang fp contract(off)
    __shared__ Waiting s_stack[kQueryWaves][64 / kFan][kStack];
    __shared__ int s_offsets[kMaxLevels], s_counts[kMaxLevels];
    if (threadIdx.x < kMaxLevels) {
        s_offsets[threadIdx.x] = levels.offsets[threadIdx.x];
        s_counts[threadIdx.x] = levels.counts[threadIdx.x];
    }
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int child = lane % kFan;
    const int group = lane / kFan;
    Waiting* stack = s_stack[threadIdx.x >> 6][group];
    const int64_t k = (static_cast<int64_t>(blockIdx.x) * kQueryWaves + (threadIdx.x >> 6)) * (64 / kFan) + group;
    const bool searching = k < n;
    const float4 p = sorted[min(k, static_cast<int64_t>(n) - 1)];
    const int self = __float_as_int(p.w);
    const float inf = __int_as_float(0x7f800000);
    // Every lane of the eight holds the search's three best.
    Nearest best = {inf, inf, inf, 0x7fffffff, 0x7fffffff, 0x7fffffff};

    if (!searching) {
        return;  // whole eights; nothing below spans them
    }
    const int own_leaf = static_cast<int>(k / kFan);
    int size = 0;
    uint32_t node = static_cast<uint32_t>(own_leaf);  // level 0: the leaf
    // Upwards from the point's own leaf: when nothing waits, the next ancestor's other children.
    int ancestor = 1;
#pragma unroll 1
    while (true) {
        const int level = static_cast<int>(node >> kNodeBits);
        const int number = static_cast<int>(node & ((1u << kNodeBits) - 1));
        const int index = number * kFan + child;
        const bool leaf = level == 0;
        bool next = false;
        if (leaf) {
            const float4 other = sorted[index];
            const float d = point_distance(p, other);
            const int id = __float_as_int(other.w);
            bool open = d <= best.d2 && id != self;  // false for NaN
            // The nearest (the smallest id of equals) of the points that can enter the list, until
            // none is left: three at most.
            while (true) {
                const float near = smallest_of_eight(open ? d : inf);
                const int near_id = smallest_of_eight(open && d == near ? id : 0x7fffffff);
                if (!before(near, near_id, best.d2, best.i2)) {
                    break;
                }
                consider(best, near, near_id);
                open = open && id != near_id;
            }
        }
        else {
            const uint32_t below = static_cast<uint32_t>(level - 1) << kNodeBits;
            // An ancestor's child on the way to the own leaf has been walked.
            bool needed = index < s_counts[level - 1] && index != own_leaf >> (kFanBits * (level - 1));
            float d = inf;
            if (needed) {
                d = box_distance(p, boxes[s_offsets[level - 1] + index]);
            }
            needed = needed && d <= best.d2;
            // The nearest child (the first of equals) is next, the other needed ones wait.
            const float near = smallest_of_eight(needed ? d : inf);
            const int shift = lane & ~(kFan - 1);
            uint32_t waiting = static_cast<uint32_t>(lanes_where(needed) >> shift) & 0xffu;
            const uint32_t nearest = static_cast<uint32_t>(lanes_where(needed && d == near) >> shift) & 0xffu;
            if (waiting) {
                const int chosen = __builtin_ctz(nearest);
                waiting &= ~(1u << chosen);
                if (waiting >> child & 1) {
                    stack[size + __popc(waiting & ((1u << child) - 1))] = {below | static_cast<uint32_t>(index), d};
                }
                size += __popc(waiting);
                node = below | static_cast<uint32_t>(number * kFan + chosen);
                next = true;
            }
        }
        wave_lds_fence();
        // Else the next box that can still hold a candidate.
        while (!next && size > 0) {
            const Waiting top = stack[--size];
            node = top.node;
            next = top.distance <= best.d2;
        }
        if (!next) {
            if (ancestor > levels.top + 1) {
                break;
            }
            node = static_cast<uint32_t>(ancestor) << kNodeBits | static_cast<uint32_t>(own_leaf >> (kFanBits * ancestor));
            ++ancestor;
        }
    }
    if (child != 0) {
        return;
    }
    int others = n - 1;
    float result;
    if (others >= 3) {
        result = (best.d0 + best.d1 + best.d2) / 3.0f;
    }
    else {
        float sum = best.d0;
        if (others == 2) {
            sum += best.d1;
        }
        result = sum / static_cast<float>(others);
    }
    mean_dist2[self] = result;
    if (neighbors) {
        const int found[3] = {best.i0, best.i1, best.i2};
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            neighbors[3ll * self + j] = j < others ? found[j] : -1;
        }
    }
}

__global__ void knn_small_kernel(int n, int* neighbors, float* mean_dist2) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        mean_dist2[i] = 0.0f;
        if (neighbors) {
            neighbors[3ll * i] = -1;
            neighbors[3ll * i + 1] = -1;
            neighbors[3ll * i + 2] = -1;
        }
    }
}

} // namespace
} // namespace gsn

extern "C" int gsn_knn3(gsn_context* context, const float* points, int n, int32_t* neighbors, float* mean_dist2) {
    using namespace gsn;
    if (!context || n < 0 || (n > 0 && (!points || !mean_dist2))) {
        return fail(GSN_ERROR_INVALID_ARGUMENT, "gsn_knn3: invalid arguments");
    }
    if (n == 0) {
        return GSN_OK;
    }
    hipStream_t stream = context->stream;
    if (n < 2) {
        knn_small_kernel<<<1, 64, 0, stream>>>(n, neighbors, mean_dist2);
        return check_launch("knn_small_kernel");
    }
    int bound_blocks = static_cast<int>(grid_for(n, 256));
    if (bound_blocks > 256) {
        bound_blocks = 256;
    }
    size_t count = static_cast<size_t>(n);
    float* bounds = static_cast<float*>(scratch(context, kSlotReduce, static_cast<size_t>(bound_blocks) * 6 * 4));
    uint32_t* keys = static_cast<uint32_t*>(scratch(context, kSlotKnnKeys, count * 4));
    uint32_t* ids = static_cast<uint32_t*>(scratch(context, kSlotKnnIds, count * 4));
    uint32_t* order = static_cast<uint32_t*>(scratch(context, kSlotKnnOrder, count * 4));
    float4* sorted = static_cast<float4*>(scratch(context, kSlotKnnPoints, (count + kFan2 - 1) / kFan2 * kFan2 * sizeof(float4)));
    // The levels of boxes, each an eighth of the one below, until at most eight are left; two more
    // entries than that may be written (levels come in pairs).
    Levels levels{};
    size_t total = 0;
    int level_count = 0;
    for (size_t boxes = (count + kFan - 1) / kFan; level_count < kMaxLevels; boxes = (boxes + kFan - 1) / kFan) {
        levels.offsets[level_count] = static_cast<int>(total);
        levels.counts[level_count] = static_cast<int>(boxes);
        total += boxes;
        levels.top = level_count++;
        if (boxes <= kFan && level_count % 2 == 0) {
            break;
        }
    }
    while (levels.top > 0 && levels.counts[levels.top - 1] <= kFan) {
        --levels.top;
    }
    Box* boxes = static_cast<Box*>(scratch(context, kSlotKnnNodes, total * sizeof(Box)));
    if (!bounds || !keys || !ids || !order || !sorted || !boxes) {
        return GSN_ERROR_OUT_OF_MEMORY;
    }
    StageScope scope(context, kStageKnn);
    knn_bounds_kernel<<<bound_blocks, 256, 0, stream>>>(points, n, bounds);
    GSN_TRY(check_launch("knn_bounds_kernel"));
    knn_morton_kernel<<<grid_for(n, 256), 256, 0, stream>>>(points, n, bounds, bound_blocks, keys, ids);
    GSN_TRY(check_launch("knn_morton_kernel"));
    GSN_TRY(radix_sort_pairs(context, keys, ids, n, 30, nullptr, order));
    knn_leaves_kernel<<<grid_for(n, 256), 256, 0, stream>>>(points, order, n, sorted, boxes,
        boxes + levels.offsets[1]);
    GSN_TRY(check_launch("knn_leaves_kernel"));
    for (int level = 1; level + 2 < level_count; level += 2) {
        knn_parents_kernel<<<grid_for(levels.counts[level], 256), 256, 0, stream>>>(boxes + levels.offsets[level],
            levels.counts[level], boxes + levels.offsets[level + 1], boxes + levels.offsets[level + 2]);
        GSN_TRY(check_launch("knn_parents_kernel"));
    }
    knn_query_kernel<<<grid_for(n, kQueryWaves * (64 / kFan)), 64 * kQueryWaves, 0, stream>>>(sorted, boxes, n, levels,
        neighbors, mean_dist2);
    return check_launch("knn_query_kernel");
}
