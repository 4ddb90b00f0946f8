// Tile rasteriser forward (reference src/core/render/renderer.cu:273-338).
// Per pixel, front to back: skip power > 0; alpha = min(0.99, o * e^power); skip alpha < 1/255;
// if T * (1 - alpha) < 1e-4 the pixel is done without blending that splat; otherwise
// C += c * alpha * T and T *= 1 - alpha. Output = C + T * background.
#include "raster_common.h"

#include <type_traits>

namespace gsn {
namespace {

// A record of the current batch as the wave's list in LDS holds it: every lane reads the same
// entry, so an entry costs three LDS reads and no vector instructions (lane reads of the nine
// values, one instruction each, were a quarter of the kernel's issue slots).
struct ForwardEntry {
    float4 a;  // centre x, y, conic a, b
    float4 b;  // conic c, opacity, red, green
    float blue;
    int band_mask;
    int index;  // tile-relative index + 1
    int unused;
};

// One pixel of a lane. A pixel that is done (outside the image, or terminated) carries T = 0: every
// later splat then finds the transmittance behind it below the termination threshold and blends
// nothing. `left` keeps the value that weights the background.
struct ForwardPixel {
    float y, T, left, red, green, blue;
    int last;
};

// A wave owns `Bands` of the tile's four 4-row bands, so a tile is run by 4 / Bands waves that do
// not need each other: every pixel still walks its records in order and the image does not depend
// on the split. What bounds it: VALU issue, about 25 slots per band evaluation (six
// for the exponent, a quarter-rate v_exp, the blend under its lanes' mask), and the length of
// the longest walk where tiles are few (forward_bands). Tiles are taken in order, neighbours on
// different XCDs: the heavy tiles of an image lie together, and a contiguous range per XCD left
// some XCDs idle (8 to 26 us slower at 4,056 and 32,400 tiles).
// Store = true additionally writes, per pixel, the final transmittance and the tile-relative
// index + 1 of the last splat blended (0 when none): the state a back-to-front backward needs.
// Count = true adds the number of (pixel, splat) pairs evaluated (pixel not yet done, splat's
// band kept by the mask) to *pair_count: the operation count of the VALU roofline.
template<int Bands, bool Store, bool Count>
__global__ __launch_bounds__(64) void raster_forward_kernel(const int* __restrict__ ids,
    const int64_t* __restrict__ tile_offsets, const float2* __restrict__ means, const float4* __restrict__ conics,
    const float* __restrict__ colors, Camera cam, float* __restrict__ image, float bg_r, float bg_g, float bg_b,
    float* __restrict__ final_transmittance, int* __restrict__ last_contributor,
    unsigned long long* __restrict__ pair_count) {
    constexpr int kParts = 4 / Bands;
    __shared__ ForwardEntry s_list[65];
    const int unit = static_cast<int>(blockIdx.x);
    const int tile = unit / kParts;
    const int first_band = (unit % kParts) * Bands;
    const int lane = threadIdx.x;
    const int x0 = (tile % cam.tile_count_x) * kTileSize;
    const int y0 = (tile / cam.tile_count_x) * kTileSize;
    const int px = x0 + (lane & 15);
    const int py = y0 + 4 * first_band + (lane >> 4);
    float fx = static_cast<float>(px);
    keep(fx);
    ForwardPixel p0, p1, p2, p3;
    unsigned evaluated = 0;
    auto each = [&](auto f) { each_band<Bands>(p0, p1, p2, p3, f); };
    each([&](ForwardPixel& p, int b) {
        const int y = py + 4 * b;
        p.y = static_cast<float>(y);
        keep(p.y);
        p.T = px < cam.width && y < cam.height ? 1.0f : 0.0f;
        p.left = 0.0f;
        p.red = 0.0f;
        p.green = 0.0f;
        p.blue = 0.0f;
        p.last = 0;
    });
    const int64_t begin = tile_offsets[tile];
    const int64_t end = tile_offsets[tile + 1];
    // While batch k is processed, the splats of batch k + 1 and the ids of batch k + 2 are in
    // flight: the two dependent gathers of a batch are then hidden behind a batch of compute also
    // when a SIMD holds a single wave.
    float2 following_mean = make_float2(0.0f, 0.0f);
    float4 following_conic = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    float following_red = 0.0f, following_green = 0.0f, following_blue = 0.0f;
    auto load = [&](int id) {
        const float* color = colors + static_cast<int64_t>(id) * 3;
        following_mean = means[id];
        following_conic = conics[id];
        following_red = color[0];
        following_green = color[1];
        following_blue = color[2];
    };
    if (begin + lane < end) {
        load(ids[begin + lane]);
    }
    int following_id = begin + 64 + lane < end ? ids[begin + 64 + lane] : -1;
    for (int64_t base = begin; base < end; base += 64) {
        int active = 0;
        each([&](ForwardPixel& p, int b) { active |= lanes_where(p.T > 0.0f) ? 1 << b : 0; });
        if (active == 0) {
            break;
        }
        int mask = 0;
        if (base + lane < end) {
            mask = band_mask<Bands>(following_mean.x, following_mean.y, following_conic, x0, y0, first_band) & active;
        }
        // The records that can reach one of the wave's open bands, in order.
        const uint64_t hits = lanes_where(mask != 0);
        if (mask != 0) {
            ForwardEntry entry;
            entry.a = make_float4(following_mean.x, following_mean.y, following_conic.x, following_conic.y);
            entry.b = make_float4(following_conic.z, following_conic.w, following_red, following_green);
            entry.blue = following_blue;
            entry.band_mask = mask;
            entry.index = static_cast<int>(base - begin) + lane + 1;
            entry.unused = 0;
            s_list[lanes_below(hits)] = entry;
        }
        if (following_id >= 0) {
            load(following_id);
        }
        following_id = base + 128 + lane < end ? ids[base + 128 + lane] : -1;
        wave_lds_fence();
        const int entries = __popcll(hits);
        ForwardEntry next_entry = s_list[0];
        for (int k = 0; k < entries; ++k) {
            const ForwardEntry e = next_entry;
            next_entry = s_list[k + 1];  // the entry after the last is allocated and not used
            const int smask = Bands == 1 ? 1 : __builtin_amdgcn_readfirstlane(e.band_mask);
            const float dx = e.a.x - fx;
            const float along = e.a.w * dx;
            const float across = dx * (e.a.z * dx);
            each([&](ForwardPixel& p, int b) {
                if (smask & (1 << b)) {
                    if (Count) {
                        evaluated += p.T > 0.0f ? 1u : 0u;
                    }
                    const float dy = e.a.y - p.y;
                    float power;
                    const float alpha = fminf(kAlphaMax, splat_alpha(across, along, e.b.x, e.b.y, dy, power));
                    const float next = p.T * (1.0f - alpha);
                    const uint64_t take = lanes_where(!(power > 0.0f)) & lanes_where(alpha >= kAlphaMin);
                    const uint64_t open = lanes_where(next >= kTransmittanceMin);
                    if (take & ~open) {
                        // Some pixel ends here (or has ended before, which changes nothing).
                        keep(p.left);
                        const uint64_t finish = take & ~open;
                        p.left = in_lanes(finish & lanes_where(p.T > 0.0f)) ? p.T : p.left;
                        p.T = in_lanes(finish) ? 0.0f : p.T;
                    }
                    if (in_lanes(take & open)) {
                        const float weight = alpha * p.T;
                        p.red = fmaf(e.b.z, weight, p.red);
                        p.green = fmaf(e.b.w, weight, p.green);
                        p.blue = fmaf(e.blue, weight, p.blue);
                        p.T = next;
                        if (Store) {
                            p.last = e.index;
                        }
                    }
                }
            });
        }
        wave_lds_fence();
    }
    each([&](ForwardPixel& p, int b) {
        const int y = py + 4 * b;
        if (px < cam.width && y < cam.height) {
            const float remaining = p.T > 0.0f ? p.T : p.left;
            const int64_t index = static_cast<int64_t>(y) * cam.width + px;
            float* pixel = image + index * 3;
            pixel[0] = p.red + remaining * bg_r;
            pixel[1] = p.green + remaining * bg_g;
            pixel[2] = p.blue + remaining * bg_b;
            if (Store) {
                final_transmittance[index] = remaining;
                last_contributor[index] = p.last;
            }
        }
    });
    if (Count) {
        unsigned long long total = evaluated;
#pragma unroll
        for (int offset = 32; offset > 0; offset >>= 1) {
            total += __shfl_xor(total, offset);
        }
        if (lane == 0) {
            atomicAdd(pair_count, total);
        }
    }
}

} // namespace
} // namespace gsn

namespace gsn {
namespace {

int launch_forward(gsn_context* context, const Camera& cam, const int* tile_gaussian_ids,
    const int64_t* tile_offsets, const float* means, const float* conic_opacities, const float* colors,
    const float* background, float* image, float* final_transmittance, int* last_contributor, unsigned tiles);

int render_tiles(gsn_context* context, const gsn_camera* camera, const int* tile_gaussian_ids,
    const int64_t* tile_offsets, const float* means, const float* conic_opacities, const float* colors,
    const float* background, float* image, float* final_transmittance, int* last_contributor) {
    if (!context || !camera || !tile_offsets || !background || !image || camera->width <= 0 || camera->height <= 0 ||
        camera->tile_count_x <= 0 || camera->tile_count_y <= 0) {
        return fail(GSN_ERROR_INVALID_ARGUMENT, "gsn_render_tiles: invalid arguments");
    }
    int64_t tiles = static_cast<int64_t>(camera->tile_count_x) * camera->tile_count_y;
    if (tiles >= 0x7fffffff) {
        return fail(GSN_ERROR_INVALID_ARGUMENT, "gsn_render_tiles: too many tiles");
    }
    Camera cam;
    memcpy(&cam, camera, sizeof(cam));
    bool forked = false;
    if (context->prefetch_armed) {
        // Armed by gsn_context_prefetch_backward: the backward's preparation of this projection
        // runs on the auxiliary stream beside this kernel and the image gradient. The fork point
        // is recorded before the kernel and the auxiliary launches are issued after it, so the
        // host's work for them does not delay the forward.
        context->prefetch_armed = false;
        if (means == context->projected_means && conic_opacities == context->projected_conics &&
            colors == context->projected_colors) {
            GSN_TRY(fork_backward_prefetch(context, cam, &forked));
        }
    }
    GSN_TRY(launch_forward(context, cam, tile_gaussian_ids, tile_offsets, means, conic_opacities, colors, background,
        image, final_transmittance, last_contributor, static_cast<unsigned>(tiles)));
    return forked ? queue_backward_prefetch(context, cam, tile_offsets) : GSN_OK;
}

// Bands per wave by the number of tiles. The chip holds 1024 SIMDs: with few tiles the kernel lasts
// as long as one wave's walk and a tile is split over four waves; with many it is bound by VALU
// issue, and bands that share a wave share its list and masks. Measured (us, one / two / four bands
// per wave): 256 tiles 42 / 72 / 123, 1,024 tiles 54 / 84 / 131, 2,170 tiles 66 / 72 / 90, 4,056 tiles
// 101 / 96 / 110, 8,160 tiles 175 / 158 / 162, 32,400 tiles 524 / 440 / 399; with one wave per tile
// and nine lane reads per splat the same images took 142, 140, 131, 153, 211 and 570. Over ten scenes a
// tile count, even and clustered, 60 to 1,500 records a tile, as shares of those times in the geometric
// mean [worst]: 3,072 tiles .56 [.85] / .60 [.74] / .78 [.86], 8,160 .84 [1.67] / .71 [.91] / .74 [.89],
// 9,600 .83 / .69 [.93] / .69 [.78], 12,288 .85 / .68 [1.04] / .66 [.76].
int forward_bands(unsigned tiles) {
    return tiles <= 3072 ? 1 : tiles <= 9600 ? 2 : 4;
}

int launch_forward(gsn_context* context, const Camera& cam, const int* tile_gaussian_ids,
    const int64_t* tile_offsets, const float* means, const float* conic_opacities, const float* colors,
    const float* background, float* image, float* final_transmittance, int* last_contributor, unsigned tiles) {
    unsigned long long* pair_count = context->count_raster_pairs ? context->raster_pairs : nullptr;
    StageScope scope(context, kStageRasterForward);
    const int bands = forward_bands(tiles);
    const unsigned units = tiles * static_cast<unsigned>(4 / bands);
    const float2* m = reinterpret_cast<const float2*>(means);
    const float4* q = reinterpret_cast<const float4*>(conic_opacities);
    auto launch = [&](auto kernel) {
        kernel<<<units, 64, 0, context->stream>>>(tile_gaussian_ids, tile_offsets, m, q, colors, cam, image,
            background[0], background[1], background[2], final_transmittance, last_contributor, pair_count);
    };
    auto with_bands = [&](auto bands_constant) {
        constexpr int kBands = decltype(bands_constant)::value;
        if (final_transmittance) {
            pair_count ? launch(raster_forward_kernel<kBands, true, true>)
                       : launch(raster_forward_kernel<kBands, true, false>);
        }
        else {
            pair_count ? launch(raster_forward_kernel<kBands, false, true>)
                       : launch(raster_forward_kernel<kBands, false, false>);
        }
    };
    switch (bands) {
    case 1:
        with_bands(std::integral_constant<int, 1>{});
        break;
    case 2:
        with_bands(std::integral_constant<int, 2>{});
        break;
    default:
        with_bands(std::integral_constant<int, 4>{});
        break;
    }
    return check_launch("raster_forward_kernel");
}

} // namespace
} // namespace gsn

extern "C" int gsn_render_tiles(gsn_context* context, const gsn_camera* camera, const int* tile_gaussian_ids,
    const int64_t* tile_offsets, const float* means, const float* conic_opacities, const float* colors,
    const float* background, float* image) {
    return gsn::render_tiles(context, camera, tile_gaussian_ids, tile_offsets, means, conic_opacities, colors,
        background, image, nullptr, nullptr);
}

extern "C" int gsn_render_tiles_stored(gsn_context* context, const gsn_camera* camera, const int* tile_gaussian_ids,
    const int64_t* tile_offsets, const float* means, const float* conic_opacities, const float* colors,
    const float* background, float* image, float* final_transmittance, int32_t* last_contributor) {
    if (!final_transmittance || !last_contributor) {
        return gsn::fail(GSN_ERROR_INVALID_ARGUMENT, "gsn_render_tiles_stored: null per-pixel state");
    }
    return gsn::render_tiles(context, camera, tile_gaussian_ids, tile_offsets, means, conic_opacities, colors,
        background, image, final_transmittance, last_contributor);
}
