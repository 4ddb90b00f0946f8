// Tile rasteriser backward (reference src/core/solver/solver.cu:325-466), recompute form.
//
// Nothing is stored per pixel by the forward pass: each pixel replays its splats front to back
// from T = 1 and uses the final colour C (image) to recover the colour behind every splat:
//   dL/dalpha_k = sum_c g_c (prefix_c + T_k c_c - C_c) / (1 - alpha_k),
// with prefix_c = sum_{i<k} c_i alpha_i T_i. Geometry and opacity gradients are taken only when
// the raw alpha is below the 0.99 cap (solver.cu:398-408).
//
// Gradient accumulation without global atomics: the 64 lanes' contributions for a splat are
// summed with wave_sum12 and the tile's total for that (tile, Gaussian) record is written to a
// per-record partial slot. The slot index is the record's position in the Gaussian-id-ordered
// enumeration, record_offsets[g] + row * width + column of the tile inside g's rectangle, so
// each Gaussian's partials are contiguous and a later per-Gaussian pass reduces them in a fixed
// order (deterministic results).
#include "raster_common.h"

namespace gsn {

namespace {

// Everything the backward needs of one Gaussian in 48 bytes, so that each record costs one
// gather instead of five (means, conics, colours, rectangles, record offsets):
//   a = (mean x, mean y, conic A, conic B), b = (conic C, opacity, red, green),
//   c = (blue, record offset, rectangle x0 | y0 << 16, rectangle width) (last three as int bits).
struct alignas(16) PackedSplat {
    float4 a, b, c;
};

__global__ __launch_bounds__(256) void pack_splats_kernel(const float2* __restrict__ means,
    const float4* __restrict__ conics, const float* __restrict__ colors, const int4* __restrict__ rects,
    const int* __restrict__ record_offsets, int count, PackedSplat* __restrict__ packed) {
    int id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= count || record_offsets[id + 1] == record_offsets[id]) {
        return;  // culled: never referenced by a record
    }
    float2 mean = means[id];
    float4 conic = conics[id];
    int4 rect = rects[id];
    const float* color = colors + static_cast<int64_t>(id) * 3;
    PackedSplat out;
    out.a = make_float4(mean.x, mean.y, conic.x, conic.y);
    out.b = make_float4(conic.z, conic.w, color[0], color[1]);
    out.c = make_float4(color[2], __int_as_float(record_offsets[id]), __int_as_float(rect.x | (rect.y << 16)),
        __int_as_float(rect.z - rect.x));
    packed[id] = out;
}

__device__ __forceinline__ int64_t partial_slot(float4 c, int tile_x, int tile_y) {
    int origin = __float_as_int(c.z);
    int width = __float_as_int(c.w);
    return static_cast<int64_t>(__float_as_int(c.y)) + (tile_y - (origin >> 16)) * width + (tile_x - (origin & 0xffff));
}

// Heavy-first tile schedule. The backward holds 4 waves per SIMD, so a 1080p frame's 8 160 tiles
// run in two rounds and a long tile (several times the mean record count) that starts late sets
// the kernel's end. Tiles are dispatched in descending order of record count instead (longest
// processing time first), bucketed at 4 buckets per octave. The order within a bucket depends on
// LDS atomics and is not fixed, which does not matter: each tile writes only its own pixels and
// record slots, so results do not depend on the schedule.
constexpr int kScheduleBins = 128;
constexpr int kScheduleThreads = 1024;

__device__ __forceinline__ int schedule_bin(int64_t records) {
    uint32_t v = static_cast<uint32_t>(min(max(records, int64_t{0}), int64_t{0x7ffffffe})) + 1u;
    int octave = 31 - __clz(v);
    int fraction = octave >= 2 ? static_cast<int>((v >> (octave - 2)) & 3u) : static_cast<int>((v << (2 - octave)) & 3u);
    return kScheduleBins - 1 - (octave * 4 + fraction);
}

// Heavy-first order of `units` work units; unit u owns records [offsets[u * stride],
// offsets[min((u + 1) * stride, count)]). Run by one whole workgroup. The bins of the first
// kScheduleItems * kScheduleThreads units are computed once into registers, with all their offset
// loads in flight together; units past that recompute their bin. (Matching equal bins across the
// wave to issue one LDS atomic per bin measured slower: the strided offset loads dominate.)
constexpr int kScheduleItems = 16;

template<typename Offset>
__device__ void schedule_units(const Offset* __restrict__ offsets, int stride, int count, int units,
    int* __restrict__ order, int* histogram, int* cursor) {
    auto bin = [&](int u) {
        int64_t begin = offsets[min(static_cast<int64_t>(u) * stride, static_cast<int64_t>(count))];
        int64_t end = offsets[min(static_cast<int64_t>(u + 1) * stride, static_cast<int64_t>(count))];
        return schedule_bin(end - begin);
    };
    int bins[kScheduleItems];
#pragma unroll
    for (int i = 0; i < kScheduleItems; ++i) {
        const int u = threadIdx.x + i * kScheduleThreads;
        bins[i] = u < units ? bin(u) : -1;
    }
    for (int b = threadIdx.x; b < kScheduleBins; b += kScheduleThreads) {
        histogram[b] = 0;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kScheduleItems; ++i) {
        if (bins[i] >= 0) {
            atomicAdd(&histogram[bins[i]], 1);
        }
    }
    for (int u = threadIdx.x + kScheduleItems * kScheduleThreads; u < units; u += kScheduleThreads) {
        atomicAdd(&histogram[bin(u)], 1);
    }
    __syncthreads();
    // Exclusive scan of the bins by the first wave, two bins per lane.
    static_assert(kScheduleBins == 128, "the scan below covers 2 x 64 bins");
    if (threadIdx.x < 64) {
        const int lane = threadIdx.x;
        const int first = histogram[2 * lane];
        const int pair = first + histogram[2 * lane + 1];
        int inclusive = pair;
#pragma unroll
        for (int offset = 1; offset < 64; offset <<= 1) {
            const int below = __shfl_up(inclusive, offset);
            inclusive += lane >= offset ? below : 0;
        }
        cursor[2 * lane] = inclusive - pair;
        cursor[2 * lane + 1] = inclusive - pair + first;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kScheduleItems; ++i) {
        if (bins[i] >= 0) {
            order[atomicAdd(&cursor[bins[i]], 1)] = threadIdx.x + i * kScheduleThreads;
        }
    }
    for (int u = threadIdx.x + kScheduleItems * kScheduleThreads; u < units; u += kScheduleThreads) {
        order[atomicAdd(&cursor[bin(u)], 1)] = u;
    }
}

// Two schedules, one per workgroup of the launch: the backward's tiles by record count, and the
// per-Gaussian pass's workgroups (kGradientGroup consecutive Gaussians) by the length of their
// record run. Density control appends its clones and split children, high-gradient Gaussians
// whose records are all reached, at the end of the id range; in id order their workgroups, the
// longest of the pass, were dispatched last and set its end (measured 1.3 -> 2.3 ms after one
// density step at 3M).
__global__ __launch_bounds__(kScheduleThreads) void tile_schedule_kernel(const int64_t* __restrict__ tile_offsets,
    int tile_count, int* __restrict__ order, const int* __restrict__ record_offsets, int gaussian_count,
    int* __restrict__ gaussian_order) {
    __shared__ int histogram[kScheduleBins];
    __shared__ int cursor[kScheduleBins];
    if (blockIdx.x == 0) {
        schedule_units(tile_offsets, 1, tile_count, tile_count, order, histogram, cursor);
    }
    else {
        schedule_units(record_offsets, kGradientGroup, gaussian_count,
            (gaussian_count + kGradientGroup - 1) / kGradientGroup, gaussian_order, histogram, cursor);
    }
}

// Plain stores: non-temporal stores of these scattered 16-byte pieces measured 2.3x the write
// traffic and twice the kernel time (each piece left the cache on its own).
__device__ __forceinline__ void store_partial(float* destination, const float4& value) {
    *reinterpret_cast<float4*>(destination) = value;
}

// One pixel of a lane.
// Recompute form: T is the transmittance in front of the next splat and `walked` the colour of the
// splats walked so far, summed with the forward's own operations, so that walked - final is exact
// where the two nearly cancel (walking -final + sums instead, one register less per channel, left
// the last splats' gradients with the rounding of the whole sum: the share of dmean_x within 1e-5
// of FP64 on 10,000 Gaussians fell from 0.89 to 0.86). Stored form: T is the transmittance behind
// the splat being walked and `walked` the colour behind it; `final` is not used. A pixel that is
// done (outside the image, or terminated) carries T = 0 in the recompute form: every later splat
// then finds T (1 - alpha) below the termination threshold and blends nothing.
struct BackwardPixel {
    float y, T, walked[3], final[3], grad[3];
    int last;
};

// Both backward forms. A tile's workgroup has 4 / Bands waves; each owns `Bands` of its four
// 4-row bands and walks the tile's records in the same batches of 64. A wave's sums over its
// pixels go to LDS; after the batch the workgroup adds the waves' sums of each record in a fixed
// order and writes the partials, three lanes a record, so a record's 48 bytes are one piece.
//
// What bounds it: VALU issue where there are several waves per SIMD (1080p), the latency of one
// wave's chain where there are not (a 256x256 image has 256 tiles on 1024 SIMDs), hence the split.
// The wave-wide sums cost about 30 slots per (record, wave), which is why many tiles keep one wave.
//
// Per pair the gradient terms are kept as sums of common * Q d and of its products with Q d; the
// exact factors (-1 for the mean, 1/2 for the covariance diagonal) are applied to the record's
// totals. Every record that is walked gets this step's flag, but only those that some pixel of the
// tile blended get a partial: the others would add exact zeros, 48 bytes written and read each.
//
// Stored form (no counterpart in the reference; kept for the memory comparison). The forward stored,
// per pixel, the final transmittance T_N and the tile-relative index + 1 of the last blended splat.
// The pass walks each tile's records back to front from the last contributor of any of its pixels,
// recovering T_k = T_{k+1} / (1 - alpha_k) and the colour behind splat k,
// B_k = T_N * background + sum_{j > k} c_j alpha_j T_j, so that
//   dL/dalpha_k = sum_c g_c (T_k c_c - B_c / (1 - alpha_k)),
// the same quantity as the recompute form's sum_c g_c (prefix_c + T_k c_c - C_c) / (1 - alpha_k).
template<int Bands, bool Stored>
__global__ __launch_bounds__(64 * (4 / Bands)) void raster_backward_kernel(const int* __restrict__ ids,
    const int64_t* __restrict__ tile_offsets, const PackedSplat* __restrict__ splats,
    const int* __restrict__ tile_order, Camera cam, const float* __restrict__ image,
    const float* __restrict__ final_transmittance, const int* __restrict__ last_contributor,
    const float* __restrict__ image_gradients, float bg_r, float bg_g, float bg_b, float* __restrict__ partials,
    uint8_t* __restrict__ record_flags, uint8_t epoch, int record_count) {
    static_assert(Bands == 1 || Bands == 4, "the forms that are launched");
    constexpr int kWaves = 4 / Bands;
    constexpr bool kIfs = Stored && Bands > 1, kSelects = Stored && Bands == 1;
    // A wave's records of the batch, in order: centre x, y, conic a, b | conic c, opacity, red, green |
    // blue, 1 - opacity, band mask, lane (the last two as int bits). Every lane reads the same entry
    // (no lane reads). Once walked, an entry's place takes the record's sums (kPartialFloats is its
    // size too).
    static_assert(kPartialFloats == 12, "an entry's place holds a record's sums");
    __shared__ float4 s_list[kWaves][65][3];
    __shared__ uint64_t s_hits[kWaves];
    __shared__ uint64_t s_contributed[kWaves];  // by place in the list
    __shared__ int s_wave[kWaves];  // Stored: a wave's last contributor; else whether it has open pixels
    __shared__ int s_slot[64];
    const int tile = tile_order[blockIdx.x];
    const int lane = threadIdx.x & 63;
    const int wave = kWaves == 1 ? 0 : __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
    const int first_band = wave * Bands;
    const int tile_x = tile % cam.tile_count_x;
    const int tile_y = tile / cam.tile_count_x;
    const int x0 = tile_x * kTileSize;
    const int y0 = tile_y * kTileSize;
    const int px = x0 + (lane & 15);
    const int py = y0 + 4 * first_band + (lane >> 4);
    float fx = static_cast<float>(px);
    keep(fx);
    BackwardPixel p0, p1, p2, p3;
    auto each = [&](auto f) { each_band<Bands>(p0, p1, p2, p3, f); };
    int tile_last = 0;
    each([&](BackwardPixel& p, int b) {
        const int y = py + 4 * b;
        const bool inside = px < cam.width && y < cam.height;
        const int64_t pixel = static_cast<int64_t>(y) * cam.width + px;
        p.y = static_cast<float>(y);
        keep(p.y);
        p.T = inside ? (Stored ? final_transmittance[pixel] : 1.0f) : (Stored ? 1.0f : 0.0f);
        p.last = Stored && inside ? last_contributor[pixel] : 0;
        tile_last = max(tile_last, p.last);
        const float background[3] = {bg_r, bg_g, bg_b};
#pragma unroll
        for (int c = 0; c < 3; ++c) {
            p.grad[c] = inside ? image_gradients[pixel * 3 + c] : 0.0f;
            p.walked[c] = Stored ? p.T * background[c] : 0.0f;
            p.final[c] = !Stored && inside ? image[pixel * 3 + c] : 0.0f;
        }
    });
    const int64_t begin = tile_offsets[tile];
    int64_t end = tile_offsets[tile + 1];
    if (Stored) {
        // Largest last contributor over the tile.
#pragma unroll
        for (int offset = 32; offset > 0; offset >>= 1) {
            tile_last = max(tile_last, __shfl_xor(tile_last, offset));
        }
        if (kWaves > 1) {
            if (lane == 0) {
                s_wave[wave] = tile_last;
            }
            __syncthreads();
            for (int w = 0; w < kWaves; ++w) {
                tile_last = max(tile_last, s_wave[w]);
            }
        }
        end = min(end, begin + static_cast<int64_t>(tile_last));
    }
    // Batch k's records: front to back, or back to front from `end`.
    const int64_t batches = (end - begin + 63) / 64;
    auto record_of = [&](int64_t k) {
        // Of the back-to-front walk the last batch may be the short one: it keeps the lanes of a
        // full batch, those below `begin` being empty.
        return Stored ? end - 64 * (k + 1) + lane : begin + 64 * k + lane;
    };
    auto has_record = [&](int64_t k) {
        const int64_t record = record_of(k);
        return k < batches && record >= begin && record < end;
    };
    // Software pipeline over record batches: while batch k is processed, the splat records of
    // batch k + 1 and the ids of batch k + 2 are in flight, so the two dependent gathers of a
    // batch (id, then its 48-byte record) are hidden behind a batch of compute.
    const float4 zero = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    PackedSplat following = {zero, zero, zero};
    if (has_record(0)) {
        following = splats[ids[record_of(0)]];
    }
    int following_id = has_record(1) ? ids[record_of(1)] : -1;
    for (int64_t k = 0; k < batches; ++k) {
        int active = (1 << Bands) - 1;
        if (!Stored) {
            active = 0;
            each([&](BackwardPixel& p, int b) { active |= lanes_where(p.T > 0.0f) ? 1 << b : 0; });
            if (kWaves == 1) {
                if (active == 0) {
                    break;
                }
            }
            else if (lane == 0) {
                s_wave[wave] = active;
            }
        }
        if (kWaves > 1) {
            // Also ends the reads of the previous batch's sums.
            __syncthreads();
            if (!Stored) {
                int any = 0;
#pragma unroll
                for (int w = 0; w < kWaves; ++w) {
                    any |= s_wave[w];
                }
                if (any == 0) {
                    break;
                }
            }
        }
        const bool valid = has_record(k);
        const float4 conic = make_float4(following.a.z, following.a.w, following.b.x, following.b.y);
        int mask = 0;
        if (valid) {
            mask = band_mask<Bands>(following.a.x, following.a.y, conic, x0, y0, first_band) & active;
        }
        const uint64_t hits = lanes_where(mask != 0);
        if (mask != 0) {
            const int place = lanes_below(hits);
            // No pixel is below the cap with an opacity that is not finite: its factor is not needed.
            const float rest = Stored && !isfinite(conic.w) ? 0.0f : 1.0f - conic.w;
            s_list[wave][place][0] = make_float4(following.a.x, following.a.y, conic.x, conic.y);
            s_list[wave][place][1] = make_float4(conic.z, conic.w, following.b.z, following.b.w);
            s_list[wave][place][2] =
                make_float4(following.c.x, rest, __int_as_float(mask), __int_as_float(lane));
        }
        if (wave == 0) {
            s_slot[lane] = valid ? static_cast<int>(partial_slot(following.c, tile_x, tile_y)) : -1;
        }
        if (following_id >= 0) {
            following = splats[following_id];
        }
        following_id = has_record(k + 2) ? ids[record_of(k + 2)] : -1;
        const int tile_index = static_cast<int>(record_of(k) - lane - begin);  // of lane 0's record
        uint64_t contributed = 0;
        const int entries = __popcll(hits);
        auto place_of = [&](int step) { return Stored ? entries - 1 - step : step; };
        wave_lds_fence();
        float4 next_a = s_list[wave][max(place_of(0), 0)][0];
        float4 next_b = s_list[wave][max(place_of(0), 0)][1];
        float4 next_c = s_list[wave][max(place_of(0), 0)][2];
        for (int step = 0; step < entries; ++step) {
            const int place = place_of(step);
            const float4 a = next_a, b4 = next_b, c4 = next_c;
            const int ahead = Stored ? max(place - 1, 0) : place + 1;
            next_a = s_list[wave][ahead][0];
            next_b = s_list[wave][ahead][1];
            next_c = s_list[wave][ahead][2];
            const int smask = Bands == 1 ? 1 : __builtin_amdgcn_readfirstlane(__float_as_int(c4.z));
            const float ca = a.z, cbv = a.w, cc = b4.x, op = b4.y;
            const float dx = a.x - fx;
            const float along = cbv * dx;
            const float ca_dx = ca * dx;
            const float across = dx * ca_dx;
            float acc[12];
#pragma unroll
            for (int f = 0; f < 12; ++f) {
                acc[f] = 0.0f;
                // Opaque to the optimiser: otherwise it folds the zero into the first band's
                // update and rebuilds twelve zeros on every path that skips a band.
                if (Bands > 1) {
                    keep(acc[f]);
                }
            }
            uint64_t blended = 0;
            each([&](BackwardPixel& p, int b) {
#pragma clang fp contract(off)
                if (smask & (1 << b)) {
                    const float dy = a.y - p.y;
                    float power;
                    const float raw_alpha = splat_alpha(across, along, cc, op, dy, power);
                    const float alpha = fminf(kAlphaMax, raw_alpha);
                    const float through = 1.0f - alpha;
                    const uint64_t take = lanes_where(!(power > 0.0f)) & lanes_where(alpha >= kAlphaMin);
                    const float next = p.T * through;
                    const uint64_t open = Stored ? lanes_where(tile_index + __float_as_int(c4.w) < p.last)
                                                 : lanes_where(next >= kTransmittanceMin);
                    const uint64_t blend = take & open;
                    // Uniform branch on "some lane blends". Recompute form: inside, lanes that do not
                    // blend add exact zeros (selects, not divergent ifs), which keeps the accumulators
                    // in place instead of merging per-lane control paths. Stored form: lanes that do
                    // not blend stay out, so that a gradient, colour or conic that is not finite
                    // reaches only the sums of splats blended at its pixel (0 times it would not be 0):
                    // by divergent ifs with four bands a wave (4,108 tiles of 400 records: 398 us, without
                    // them 399, selects 435), by selects with one, where ifs need the sums' zeros in
                    // registers first (1,024 tiles of 300: 130 us, without them 127, ifs 138).
                    if (blend) {
                        blended |= blend;
                        const float inv = __builtin_amdgcn_rcpf(through);
                        const float before = Stored ? p.T * inv : p.T;
                        const float weight = kIfs || in_lanes(blend) ? alpha * before : 0.0f;
                        const float colour[3] = {b4.z, b4.w, c4.x};
                        const uint64_t uncapped = blend & lanes_where(raw_alpha < kAlphaMax);
                        if (!kIfs || in_lanes(blend)) {
                            float sum = 0.0f;
#pragma unroll
                            for (int c = 0; c < 3; ++c) {
                                const float difference = Stored ? fmaf(before, colour[c], -p.walked[c] * inv)
                                                                : fmaf(colour[c], before, p.walked[c]) - p.final[c];
                                sum = Stored ? fmaf(p.grad[c], difference, sum) : fmaf(inv, p.grad[c] * difference, sum);
                                acc[6 + c] = fmaf(weight, !kSelects || in_lanes(blend) ? p.grad[c] : 0.0f, acc[6 + c]);
                                const float walked = fmaf(colour[c], weight, p.walked[c]);
                                p.walked[c] = !kSelects || in_lanes(blend) ? walked : p.walked[c];
                            }
                            p.T = in_lanes(blend) ? (Stored ? before : next) : p.T;
                            if (!kIfs || in_lanes(uncapped)) {
                                const float common = in_lanes(uncapped) ? raw_alpha * sum : 0.0f;
                                const float qx = !kSelects || in_lanes(uncapped) ? fmaf(cbv, dy, ca_dx) : 0.0f;
                                const float qy = !kSelects || in_lanes(uncapped) ? along + cc * dy : 0.0f;
                                const float gx = common * qx;
                                const float gy = common * qy;
                                acc[0] = fmaf(qx, common, acc[0]);
                                acc[1] = fmaf(qy, common, acc[1]);
                                acc[2] = fmaf(qx, gx, acc[2]);
                                acc[3] = fmaf(qy, gx, acc[3]);
                                acc[4] = fmaf(qy, gy, acc[4]);
                                acc[5] = fmaf(c4.y, common, acc[5]);
                                acc[9] += fabsf(gx);
                                acc[10] += fabsf(gy);
                            }
                        }
                    }
                    if (!Stored && (take & ~open)) {
                        keep(p.T);
                        p.T = in_lanes(take & ~open) ? 0.0f : p.T;
                    }
                }
            });
            if (blended) {
                contributed |= 1ull << place;
                float sums[3];
                wave_sum12(acc, sums);
                if ((lane & 15) == 0) {
                    float* destination = reinterpret_cast<float*>(s_list[wave][place]) + 3 * (lane >> 4);
#pragma unroll
                    for (int f = 0; f < 3; ++f) {
                        destination[f] = sums[f];
                    }
                }
            }
        }
        if (kWaves > 1 && lane == 0) {
            s_hits[wave] = hits;
            s_contributed[wave] = contributed;
        }
        __syncthreads();
        // 64 records x three 16-byte pieces; consecutive lanes write a record's consecutive pieces.
        for (int item = threadIdx.x; item < 64 * 3; item += 64 * kWaves) {
            const int record = item / 3;
            const int piece = item - 3 * record;
            float4 sum = zero;
            bool any = false;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) {
                const uint64_t listed = kWaves == 1 ? hits : s_hits[w];
                const uint64_t mine = kWaves == 1 ? contributed : s_contributed[w];
                const int place = __popcll(listed & ((1ull << record) - 1));
                if (((listed >> record) & 1) && ((mine >> place) & 1)) {
                    const float4 v = s_list[w][place][piece];
                    sum = make_float4(sum.x + v.x, sum.y + v.y, sum.z + v.z, sum.w + v.w);
                    any = true;
                }
            }
            const int slot = s_slot[record];
            if (slot >= 0 && slot < record_count) {
                if (piece == 0) {
                    record_flags[slot] = any ? epoch | kFlagPartial : epoch;
                    sum = make_float4(-sum.x, -sum.y, 0.5f * sum.z, sum.w);
                }
                else if (piece == 1) {
                    sum.x *= 0.5f;
                }
                if (any) {
                    store_partial(partials + static_cast<int64_t>(slot) * kPartialFloats + 4 * piece, sum);
                }
            }
        }
        if (kWaves == 1) {
            __syncthreads();  // the next batch rewrites the sums (one wave: no barrier, an ordering)
        }
    }
    // Records after every pixel of the tile terminated (Stored: behind every pixel's last
    // contributor) contribute nothing; they get neither a partial nor this step's flag.
}

__global__ __launch_bounds__(64) void wave_sum12_selftest_kernel(const float* input, float* output) {
    int lane = threadIdx.x;
    float v[12];
#pragma unroll
    for (int k = 0; k < 12; ++k) {
        v[k] = input[lane * 12 + k];
    }
    float sums[3];
    wave_sum12(v, sums);
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        output[lane * 3 + k] = sums[k];
    }
}

__global__ __launch_bounds__(256) void clear_flags_kernel(uint32_t* flags, int64_t words) {
    int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
    if (i < words) {
        flags[i] = 0u;
    }
}

} // namespace

// The backward's splat copy and its two schedules (tile order, per-Gaussian group order).
struct BackwardBuffers {
    PackedSplat* splats = nullptr;
    int* order = nullptr;
    int* groups_order = nullptr;
};

static int backward_buffers(gsn_context* context, const Camera& cam, int count, BackwardBuffers* buffers) {
    const int64_t tiles = static_cast<int64_t>(cam.tile_count_x) * cam.tile_count_y;
    const int groups = (count + kGradientGroup - 1) / kGradientGroup;
    buffers->splats = static_cast<PackedSplat*>(
        scratch(context, kSlotSplats, static_cast<size_t>(count > 0 ? count : 1) * sizeof(PackedSplat)));
    buffers->order = static_cast<int*>(scratch(context, kSlotTileOrder, static_cast<size_t>(tiles) * 4));
    buffers->groups_order =
        static_cast<int*>(scratch(context, kSlotGaussianOrder, static_cast<size_t>(groups > 0 ? groups : 1) * 4));
    return buffers->splats && buffers->order && buffers->groups_order ? GSN_OK : GSN_ERROR_OUT_OF_MEMORY;
}

static int launch_backward_preparation(hipStream_t stream, const Camera& cam, int count, const int64_t* tile_offsets,
    const float* means, const float* conics, const float* colors, const int* rects, const int* record_offsets,
    const BackwardBuffers& buffers) {
    const int64_t tiles = static_cast<int64_t>(cam.tile_count_x) * cam.tile_count_y;
    pack_splats_kernel<<<grid_for(count, 256), 256, 0, stream>>>(reinterpret_cast<const float2*>(means),
        reinterpret_cast<const float4*>(conics), colors, reinterpret_cast<const int4*>(rects), record_offsets, count,
        buffers.splats);
    GSN_TRY(check_launch("pack_splats_kernel"));
    tile_schedule_kernel<<<2, kScheduleThreads, 0, stream>>>(tile_offsets, static_cast<int>(tiles), buffers.order,
        record_offsets, count, buffers.groups_order);
    return check_launch("tile_schedule_kernel");
}

int join_backward_prefetch(gsn_context* context) {
    if (!context->prefetch_pending) {
        return GSN_OK;
    }
    context->prefetch_pending = false;
    return check_hip(hipStreamWaitEvent(context->stream, context->join_event, 0), "hipStreamWaitEvent");
}

int fork_backward_prefetch(gsn_context* context, const Camera& cam, bool* forked) {
    *forked = false;
    GSN_TRY(join_backward_prefetch(context));
    const int count = context->projected_gaussians;
    if (count <= 0 || !context->aux_stream || cam.tile_count_x > 0xffff || cam.tile_count_y > 0x7fff) {
        return GSN_OK;
    }
    // Allocations first: growing a slot synchronises both streams before it frees the old buffer.
    BackwardBuffers buffers;
    GSN_TRY(backward_buffers(context, cam, count, &buffers));
    GSN_HIP(hipEventRecord(context->fork_event, context->stream));
    *forked = true;
    return GSN_OK;
}

int queue_backward_prefetch(gsn_context* context, const Camera& cam, const int64_t* tile_offsets) {
    const int count = context->projected_gaussians;
    BackwardBuffers buffers;
    GSN_TRY(backward_buffers(context, cam, count, &buffers));  // allocated by the fork: no growth here
    GSN_HIP(hipStreamWaitEvent(context->aux_stream, context->fork_event, 0));
    GSN_TRY(launch_backward_preparation(context->aux_stream, cam, count, tile_offsets, context->projected_means,
        context->projected_conics, context->projected_colors, context->projected_rects,
        context->projected_record_offsets, buffers));
    GSN_HIP(hipEventRecord(context->join_event, context->aux_stream));
    context->prefetch_pending = true;
    BackwardPrefetch& queued = context->prefetch;
    queued.means = context->projected_means;
    queued.conics = context->projected_conics;
    queued.colors = context->projected_colors;
    queued.rects = context->projected_rects;
    queued.offsets = context->projected_record_offsets;
    queued.tile_offsets = tile_offsets;
    queued.count = count;
    queued.tiles_x = cam.tile_count_x;
    queued.tiles_y = cam.tile_count_y;
    queued.generation = context->projection_generation;
    return GSN_OK;
}

int launch_splat_backward(gsn_context* context, const Camera& cam, int count, const int* ids,
    const int64_t* tile_offsets, const float* means, const float* conics, const float* colors, const int* rects,
    const int* record_offsets, const float* image, const float* image_gradients, float* partials, int record_count,
    const uint8_t** flags, uint8_t* epoch, const int** gaussian_order, const StoredState* stored) {
    if (cam.tile_count_x > 0xffff || cam.tile_count_y > 0x7fff) {
        return fail(GSN_ERROR_INVALID_ARGUMENT, "raster backward: tile grid exceeds 65535 x 32767");
    }
    int64_t tiles = static_cast<int64_t>(cam.tile_count_x) * cam.tile_count_y;
    // Work queued by an armed gsn_render_tiles is joined first, and reused when it was computed
    // from these buffers of the current projection.
    const BackwardPrefetch& queued = context->prefetch;
    const bool prefetched = context->prefetch_pending && queued.generation == context->projection_generation &&
        queued.means == means && queued.conics == conics && queued.colors == colors && queued.rects == rects &&
        queued.offsets == record_offsets && queued.tile_offsets == tile_offsets && queued.count == count &&
        queued.tiles_x == cam.tile_count_x && queued.tiles_y == cam.tile_count_y;
    GSN_TRY(join_backward_prefetch(context));
    context->prefetch = BackwardPrefetch{};
    BackwardBuffers buffers;
    GSN_TRY(backward_buffers(context, cam, count, &buffers));
    PackedSplat* splats = buffers.splats;
    int* order = buffers.order;
    int* groups_order = buffers.groups_order;
    // One flag byte per record, read 16 at a time by the per-Gaussian pass (scratch slots are
    // allocated in multiples of 256 bytes, so an aligned 16-byte read below the record count
    // stays inside the allocation).
    uint8_t* record_flags = static_cast<uint8_t*>(scratch(context, kSlotRecordFlags, static_cast<size_t>(record_count)));
    if (!splats || !order || !groups_order || !record_flags) {
        return GSN_ERROR_OUT_OF_MEMORY;
    }
    // The epoch runs 1..127 (the flag's eighth bit says that the record has a partial). After a wrap,
    // or in a newly allocated buffer, every byte is cleared first, so that a stale byte never equals
    // the current epoch.
    uint8_t next = static_cast<uint8_t>(context->record_epoch + 1);
    const size_t flag_bytes = context->slot_bytes[kSlotRecordFlags];
    if (next == kFlagPartial || context->record_flags_cleared != record_flags ||
        context->record_flags_cleared_bytes != flag_bytes) {
        int64_t words = static_cast<int64_t>(flag_bytes / 4);
        clear_flags_kernel<<<grid_for(words, 256), 256, 0, context->stream>>>(reinterpret_cast<uint32_t*>(record_flags),
            words);
        GSN_TRY(check_launch("clear_flags_kernel"));
        context->record_flags_cleared = record_flags;
        context->record_flags_cleared_bytes = flag_bytes;
        next = 1;
    }
    context->record_epoch = next;
    *flags = record_flags;
    *epoch = next;
    StageScope scope(context, kStageRasterBackward);
    if (prefetched) {
        ++context->prefetch_reused;
    }
    else {
        GSN_TRY(launch_backward_preparation(context->stream, cam, count, tile_offsets, means, conics, colors, rects,
            record_offsets, buffers));
    }
    *gaussian_order = groups_order;
    auto launch = [&](auto kernel, int waves) {
        kernel<<<static_cast<unsigned>(tiles), 64 * waves, 0, context->stream>>>(ids, tile_offsets, splats, order, cam,
            image, stored ? stored->final_transmittance : nullptr, stored ? stored->last_contributor : nullptr,
            image_gradients, stored ? stored->background[0] : 0.0f, stored ? stored->background[1] : 0.0f,
            stored ? stored->background[2] : 0.0f, partials, record_flags, next, record_count);
    };
    // Four waves per tile while the tiles are few, one otherwise. Measured (us, four / two / one wave
    // per tile): 256 tiles 102 / 156 / 226, 1,024 tiles 110 / 161 / 236, 4,056 tiles 274 / 240 / 238,
    // 8,160 tiles 468 / 389 / 345; with one wave per tile and ten lane reads per splat the same images
    // took 241, 241, 256 and 397. Stored form, 4,108 tiles: 259 / 233 / 204, before 236. Over ten scenes a
    // tile count, even and clustered, 60 to 1,500 records a tile, as shares of those times in the
    // geometric mean [worst], four waves and one: 1,024 tiles .65 [.80], 1.00 [1.01]; 2,560 .75 [.96], .93
    // [1.02]; 3,072 .79 [1.07], .92 [1.01]; 4,000 .89 [1.11], .91 [1.01]; 6,144 1.00 [1.17], .90 [.98]. Even
    // lists would want the line at about 2,000 tiles, clustered ones past 6,000; the tile count does not
    // tell them apart. Two waves were measured and are not launched.
    if (tiles <= 3072) {
        stored ? launch(raster_backward_kernel<1, true>, 4) : launch(raster_backward_kernel<1, false>, 4);
    }
    else {
        stored ? launch(raster_backward_kernel<4, true>, 1) : launch(raster_backward_kernel<4, false>, 1);
    }
    return check_launch("raster_backward_kernel");
}

} // namespace gsn

namespace gsn {
namespace {

__global__ __launch_bounds__(256) void band_mask_selftest_kernel(const float* splats, const int* origins, int count,
    int* masks) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= count) {
        return;
    }
    const float* s = splats + static_cast<int64_t>(i) * 6;
    masks[i] = band_mask<4>(s[0], s[1], make_float4(s[2], s[3], s[4], s[5]), origins[2 * i], origins[2 * i + 1], 0);
}

} // namespace
} // namespace gsn

// Diagnostic: the rasterisers' band mask on `count` (splat, tile) cases.
extern "C" int gsn_selftest_band_mask(gsn_context* context, const float* splats, const int* origins, int count,
    int* masks) {
    using namespace gsn;
    if (!context || count < 0 || (count > 0 && (!splats || !origins || !masks))) {
        return fail(GSN_ERROR_INVALID_ARGUMENT, "gsn_selftest_band_mask: invalid arguments");
    }
    if (count == 0) {
        return GSN_OK;
    }
    band_mask_selftest_kernel<<<grid_for(count, 256), 256, 0, context->stream>>>(splats, origins, count, masks);
    return check_launch("band_mask_selftest_kernel");
}

// Diagnostic: runs the wave reduction on one wave. input float[64][12] -> output float[64][3].
extern "C" int gsn_selftest_wave_sum12(gsn_context* context, const float* input, float* output) {
    using namespace gsn;
    if (!context || !input || !output) {
        return fail(GSN_ERROR_INVALID_ARGUMENT, "gsn_selftest_wave_sum12: null argument");
    }
    wave_sum12_selftest_kernel<<<1, 64, 0, context->stream>>>(input, output);
    return check_launch("wave_sum12_selftest_kernel");
}
