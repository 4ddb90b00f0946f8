// Fused L1 + SSIM image gradient (reference src/core/solver/solver.cu:26-168) and the loss /
// metric reduction the reference lacks.
//
// L = 0.8 * mean|I - T| + 0.2 * (1 - mean SSIM) over 3*W*H values; SSIM uses the separable
// 11-tap Gaussian window (sigma 1.5, normalised) with zero padding, C1 = 1e-4, C2 = 9e-4.
// One workgroup computes a 32x32 output tile of one channel: a 10-pixel halo is staged in LDS,
// the five window moments are filtered horizontally then vertically, the per-position SSIM
// derivative coefficients (a, b, c) are formed, and the adjoint filter is applied (again
// separably) to give dL/dI = (0.8 sign(I - T) - 0.2 (Wa + T Wb + 2 I Wc)) / (3 W H).
#include "gsn_internal.h"

#include <cmath>
#include <vector>

namespace gsn {
namespace {

constexpr int kTw = 32;
constexpr int kTh = 32;
constexpr int kIw = kTw + 20;  // input columns (10-pixel halo each side)
constexpr int kIh = kTh + 20;  // input rows
constexpr int kMw = kTw + 10;  // moment columns (output +- 5)
constexpr int kMh = kTh + 10;  // moment rows after the vertical pass
constexpr int kThreads = 512;

struct Window {
    float w[11];
};

Window make_window() {
    // Normalised Gaussian, sigma = 1.5, radius 5 (cv::getGaussianKernel(11, 1.5)).
    double values[11], sum = 0.0;
    for (int i = 0; i < 11; ++i) {
        double x = i - 5;
        values[i] = std::exp(-x * x / (2.0 * 1.5 * 1.5));
        sum += values[i];
    }
    Window window;
    for (int i = 0; i < 11; ++i) {
        window.w[i] = static_cast<float>(values[i] / sum);
    }
    return window;
}

struct SsimTile {
    float in[2 * kIh * kIw];
    float h[5 * kIh * kMw];
};

// Register blocking: each thread filters a run of adjacent outputs from one window of values read
// from LDS once (11-tap windows overlap by 10), which cuts LDS reads 3-4x against one thread per
// output; every output still sums its taps in the same order, so results are unchanged.
constexpr int kRunH = 6;   // horizontal moments: outputs per thread (kMw = 42 = 7 runs)
constexpr int kRunV = 4;   // vertical moments: rows per thread (kMh = 42: ten runs of 4, one of 2)
constexpr int kRunA = 4;   // horizontal adjoint: outputs per thread (kTw = 32 = 8 runs)
constexpr int kRunO = 2;   // vertical adjoint: rows per thread (kTh = 32 = 16 runs)
static_assert(kMw % kRunH == 0 && kTw % kRunA == 0 && kTh % kRunO == 0, "runs must tile the rows");

__device__ __forceinline__ void ssim_coefficients(const float (&m)[5], bool inside, float& a, float& b, float& c) {
    a = 0.0f;
    b = 0.0f;
    c = 0.0f;
    if (inside) {
        float mu_a = m[0], mu_b = m[1];
        float inverse_d = 1.0f / (mu_a * mu_a + mu_b * mu_b + 0.0001f);
        float inverse_e = 1.0f / (m[2] - mu_a * mu_a + m[3] - mu_b * mu_b + 0.0009f);
        float luminance = (2.0f * mu_a * mu_b + 0.0001f) * inverse_d;
        float contrast = (2.0f * (m[4] - mu_a * mu_b) + 0.0009f) * inverse_e;
        float mean_derivative = 2.0f * (mu_b - mu_a * luminance) * inverse_d * contrast;
        b = 2.0f * luminance * inverse_e;
        c = -luminance * contrast * inverse_e;
        a = mean_derivative - mu_b * b - 2.0f * mu_a * c;
    }
}

// Work items are (tile, channel) pairs, channel fastest, and each XCD runs a contiguous range of
// them (xcd_remap): the three channel workgroups of a tile, which read the same interleaved RGB
// lines, and neighbouring tiles, which share halo lines, then meet in one XCD's L2.
__global__ __launch_bounds__(kThreads) void image_gradients_kernel(const float* __restrict__ image,
    const uint8_t* __restrict__ target, float* __restrict__ gradients, int width, int height, int tiles_x,
    int items, Window win) {
    __shared__ SsimTile s;
    const int item = xcd_remap(static_cast<int>(blockIdx.x), items);
    const int channel = item % 3;
    const int tile = item / 3;
    const int origin_x = (tile % tiles_x) * kTw;
    const int origin_y = (tile / tiles_x) * kTh;
    const int t = threadIdx.x;
    // 1. Image and target with a 10-pixel halo (zero outside the image).
    for (int idx = t; idx < kIh * kIw; idx += kThreads) {
        int iy = idx / kIw, ix = idx - iy * kIw;
        int gx = origin_x - 10 + ix, gy = origin_y - 10 + iy;
        bool valid = gx >= 0 && gy >= 0 && gx < width && gy < height;
        int64_t index = (static_cast<int64_t>(gy) * width + gx) * 3 + channel;
        s.in[idx] = valid ? image[index] : 0.0f;
        s.in[kIh * kIw + idx] = valid ? static_cast<float>(target[index]) * (1.0f / 255.0f) : 0.0f;
    }
    __syncthreads();
    // 2. Horizontal pass of the five moments, kRunH adjacent columns per thread.
    for (int item = t; item < kIh * (kMw / kRunH); item += kThreads) {
        const int iy = item / (kMw / kRunH);
        const int column = (item - iy * (kMw / kRunH)) * kRunH;
        // The products of each input value are formed once and shared by the 11 taps that read it.
        float a[kRunH + 10], b[kRunH + 10], aa[kRunH + 10], bb[kRunH + 10], ab[kRunH + 10];
#pragma unroll
        for (int j = 0; j < kRunH + 10; ++j) {
            a[j] = s.in[iy * kIw + column + j];
            b[j] = s.in[kIh * kIw + iy * kIw + column + j];
            aa[j] = a[j] * a[j];
            bb[j] = b[j] * b[j];
            ab[j] = a[j] * b[j];
        }
#pragma unroll
        for (int g = 0; g < kRunH; ++g) {
            float m0 = 0.0f, m1 = 0.0f, m2 = 0.0f, m3 = 0.0f, m4 = 0.0f;
#pragma unroll
            for (int dx = 0; dx < 11; ++dx) {
                float w = win.w[dx];
                m0 += w * a[g + dx];
                m1 += w * b[g + dx];
                m2 += w * aa[g + dx];
                m3 += w * bb[g + dx];
                m4 += w * ab[g + dx];
            }
            const int idx = iy * kMw + column + g;
            s.h[0 * kIh * kMw + idx] = m0;
            s.h[1 * kIh * kMw + idx] = m1;
            s.h[2 * kIh * kMw + idx] = m2;
            s.h[3 * kIh * kMw + idx] = m3;
            s.h[4 * kIh * kMw + idx] = m4;
        }
    }
    __syncthreads();
    // 3. Vertical pass (kRunV rows per thread) and the per-position SSIM derivative coefficients
    //    (a, b, c); the coefficient maps reuse the input region, whose reads all ended above.
    float* coef = s.in;  // [3][kMh][kMw]
    constexpr int kRunsV = (kMh + kRunV - 1) / kRunV;
    for (int item = t; item < kMw * kRunsV; item += kThreads) {
        const int mx = item % kMw;
        const int row0 = (item / kMw) * kRunV;
        const int rows = min(kRunV, kMh - row0);
        float m[kRunV][5];
#pragma unroll
        for (int g = 0; g < kRunV; ++g) {
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                m[g][k] = 0.0f;
            }
        }
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            float v[kRunV + 10];
#pragma unroll
            for (int j = 0; j < kRunV + 10; ++j) {
                const int row = min(row0 + j, kIh - 1);  // rows past the region feed only unused outputs
                v[j] = s.h[k * kIh * kMw + row * kMw + mx];
            }
#pragma unroll
            for (int dy = 0; dy < 11; ++dy) {
                float w = win.w[dy];
#pragma unroll
                for (int g = 0; g < kRunV; ++g) {
                    m[g][k] += w * v[g + dy];
                }
            }
        }
        const int hx = origin_x - 5 + mx;
#pragma unroll
        for (int g = 0; g < kRunV; ++g) {
            if (g < rows) {
                const int my = row0 + g;
                const int hy = origin_y - 5 + my;
                const bool inside = hx >= 0 && hy >= 0 && hx < width && hy < height;
                float ca, cb, cc;
                ssim_coefficients(m[g], inside, ca, cb, cc);
                coef[0 * kMh * kMw + my * kMw + mx] = ca;
                coef[1 * kMh * kMw + my * kMw + mx] = cb;
                coef[2 * kMh * kMw + my * kMw + mx] = cc;
            }
        }
    }
    __syncthreads();
    // 4. Horizontal adjoint of the three coefficient maps, kRunA adjacent columns per thread.
    float* adjoint = s.h;  // [3][kMh][kTw]
    for (int item = t; item < kMh * (kTw / kRunA); item += kThreads) {
        const int my = item / (kTw / kRunA);
        const int column = (item - my * (kTw / kRunA)) * kRunA;
#pragma unroll
        for (int f = 0; f < 3; ++f) {
            float v[kRunA + 10];
#pragma unroll
            for (int j = 0; j < kRunA + 10; ++j) {
                v[j] = coef[f * kMh * kMw + my * kMw + column + j];
            }
#pragma unroll
            for (int g = 0; g < kRunA; ++g) {
                float sum = 0.0f;
#pragma unroll
                for (int dx = 0; dx < 11; ++dx) {
                    sum += win.w[dx] * v[g + dx];
                }
                adjoint[f * kMh * kTw + my * kTw + column + g] = sum;
            }
        }
    }
    __syncthreads();
    // 5. Vertical adjoint (kRunO rows per thread) and dL/dI.
    const float normalization = 1.0f / (3.0f * static_cast<float>(width) * static_cast<float>(height));
    for (int item = t; item < kTw * (kTh / kRunO); item += kThreads) {
        const int ox = item % kTw;
        const int row0 = (item / kTw) * kRunO;
        float f[kRunO][3];
#pragma unroll
        for (int m = 0; m < 3; ++m) {
            float v[kRunO + 10];
#pragma unroll
            for (int j = 0; j < kRunO + 10; ++j) {
                v[j] = adjoint[m * kMh * kTw + (row0 + j) * kTw + ox];
            }
#pragma unroll
            for (int g = 0; g < kRunO; ++g) {
                float sum = 0.0f;
#pragma unroll
                for (int dy = 0; dy < 11; ++dy) {
                    sum += win.w[dy] * v[g + dy];
                }
                f[g][m] = sum;
            }
        }
        const int x = origin_x + ox;
#pragma unroll
        for (int g = 0; g < kRunO; ++g) {
            const int y = origin_y + row0 + g;
            if (x >= width || y >= height) {
                continue;
            }
            int64_t pixel = (static_cast<int64_t>(y) * width + x) * 3 + channel;
            float render = image[pixel];
            float reference = static_cast<float>(target[pixel]) * (1.0f / 255.0f);
            float residual = render - reference;
            float l1_gradient = static_cast<float>(residual > 0.0f) - static_cast<float>(residual < 0.0f);
            float ssim_gradient = -(f[g][0] + reference * f[g][1] + 2.0f * render * f[g][2]);
            gradients[pixel] = (0.8f * l1_gradient + 0.2f * ssim_gradient) * normalization;
        }
    }
}

// Input region of a metrics tile: the outputs and the window's five pixels each side.
constexpr int kEw = kTw + 10;
constexpr int kEh = kTh + 10;
constexpr int kRunE = 4;  // horizontal moments: outputs per thread
constexpr int kRunF = 2;  // vertical moments: rows per thread
static_assert(kTw % kRunE == 0 && kTh % kRunF == 0, "runs must tile the rows");

// Per-block sums of (|I - T|, SSIM, (clamp(I, 0, 1) - T)^2) over the block's output pixels. The
// filters are register-blocked as in the gradient, over the outputs only (no second halo): bound by
// vector instructions and LDS reads, 41 KB of LDS, three workgroups per CU. 1332x876: 72 us with
// one output a thread over the halo twice, 41.5 us so.
__global__ __launch_bounds__(kThreads) void image_metrics_kernel(const float* __restrict__ image,
    const uint8_t* __restrict__ target, double* __restrict__ block_sums, int width, int height, Window win) {
    __shared__ float s_in[2][kEh * kEw];
    __shared__ float s_h[5][kEh * kTw];
    __shared__ double s_reduce[3][kThreads / 64];
    const int channel = blockIdx.z;
    const int origin_x = blockIdx.x * kTw;
    const int origin_y = blockIdx.y * kTh;
    const int t = threadIdx.x;
    float l1_sum = 0.0f, squared_sum = 0.0f, ssim_sum = 0.0f;
    for (int idx = t; idx < kEh * kEw; idx += kThreads) {
        const int iy = idx / kEw, ix = idx - iy * kEw;
        const int gx = origin_x - 5 + ix, gy = origin_y - 5 + iy;
        const bool valid = gx >= 0 && gy >= 0 && gx < width && gy < height;
        const int64_t index = (static_cast<int64_t>(gy) * width + gx) * 3 + channel;
        const float render = valid ? image[index] : 0.0f;
        const float reference = valid ? static_cast<float>(target[index]) * (1.0f / 255.0f) : 0.0f;
        s_in[0][idx] = render;
        s_in[1][idx] = reference;
        if (valid && ix >= 5 && ix < kTw + 5 && iy >= 5 && iy < kTh + 5) {
            l1_sum += fabsf(render - reference);
            const float clamped = fminf(fmaxf(render, 0.0f), 1.0f) - reference;
            squared_sum += clamped * clamped;
        }
    }
    __syncthreads();
    for (int item = t; item < kEh * (kTw / kRunE); item += kThreads) {
        const int iy = item / (kTw / kRunE);
        const int column = (item - iy * (kTw / kRunE)) * kRunE;
        float a[kRunE + 10], b[kRunE + 10];
#pragma unroll
        for (int j = 0; j < kRunE + 10; ++j) {
            a[j] = s_in[0][iy * kEw + column + j];
            b[j] = s_in[1][iy * kEw + column + j];
        }
#pragma unroll
        for (int g = 0; g < kRunE; ++g) {
            float m[5] = {0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int dx = 0; dx < 11; ++dx) {
                const float w = win.w[dx];
                const float wa = w * a[g + dx], wb = w * b[g + dx];
                m[0] += wa;
                m[1] += wb;
                m[2] += wa * a[g + dx];
                m[3] += wb * b[g + dx];
                m[4] += wa * b[g + dx];
            }
#pragma unroll
            for (int k = 0; k < 5; ++k) {
                s_h[k][iy * kTw + column + g] = m[k];
            }
        }
    }
    __syncthreads();
    for (int item = t; item < kTw * (kTh / kRunF); item += kThreads) {
        const int ox = item % kTw;
        const int row0 = item / kTw * kRunF;
        float m[kRunF][5];
#pragma unroll
        for (int k = 0; k < 5; ++k) {
            float v[kRunF + 10];
#pragma unroll
            for (int j = 0; j < kRunF + 10; ++j) {
                v[j] = s_h[k][(row0 + j) * kTw + ox];
            }
#pragma unroll
            for (int g = 0; g < kRunF; ++g) {
                float sum = 0.0f;
#pragma unroll
                for (int dy = 0; dy < 11; ++dy) {
                    sum += win.w[dy] * v[g + dy];
                }
                m[g][k] = sum;
            }
        }
#pragma unroll
        for (int g = 0; g < kRunF; ++g) {
            if (origin_x + ox < width && origin_y + row0 + g < height) {
                const float mu_a = m[g][0], mu_b = m[g][1];
                const float luminance = (2.0f * mu_a * mu_b + 0.0001f) / (mu_a * mu_a + mu_b * mu_b + 0.0001f);
                const float contrast = (2.0f * (m[g][4] - mu_a * mu_b) + 0.0009f) /
                                       (m[g][2] - mu_a * mu_a + m[g][3] - mu_b * mu_b + 0.0009f);
                ssim_sum += luminance * contrast;
            }
        }
    }
    // Fixed-order sums in FP64: within each wave, then over the waves.
    double sums[3] = {l1_sum, ssim_sum, squared_sum};
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            sums[k] += __shfl_xor(sums[k], offset);
        }
    }
    if ((t & 63) == 0) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            s_reduce[k][t >> 6] = sums[k];
        }
    }
    __syncthreads();
    if (t < 3) {
        double total = 0.0;
#pragma unroll
        for (int w = 0; w < kThreads / 64; ++w) {
            total += s_reduce[t][w];
        }
        int64_t block = (static_cast<int64_t>(blockIdx.z) * gridDim.y + blockIdx.y) * gridDim.x + blockIdx.x;
        block_sums[block * 3 + t] = total;
    }
}

const Window& window() {
    static const Window w = make_window();
    return w;
}

} // namespace
} // namespace gsn

extern "C" int gsn_image_gradients(gsn_context* context, int width, int height, const float* image,
    const uint8_t* target, float* image_gradients) {
    using namespace gsn;
    if (!context || width <= 0 || height <= 0 || !image || !target || !image_gradients) {
        return fail(GSN_ERROR_INVALID_ARGUMENT, "gsn_image_gradients: invalid arguments");
    }
    const int tiles_x = static_cast<int>(grid_for(width, kTw));
    const int64_t items = static_cast<int64_t>(tiles_x) * grid_for(height, kTh) * 3;
    if (items > 0x7fffffff) {
        return fail(GSN_ERROR_INVALID_ARGUMENT, "gsn_image_gradients: image too large");
    }
    StageScope scope(context, kStageImageGradients);
    image_gradients_kernel<<<static_cast<unsigned>(items), kThreads, 0, context->stream>>>(image, target,
        image_gradients, width, height, tiles_x, static_cast<int>(items), window());
    return check_launch("image_gradients_kernel");
}

namespace gsn {
namespace {

// Fixed-order finish of the per-block metric sums by one workgroup: thread t adds blocks t, t + 1024,
// ... in order, then the wave's lanes are combined by a butterfly and the waves in order, so every
// call with the same inputs returns the same bits (1,148 blocks: 15.5 us with 64 threads, 5 us so).
// out = {0.8 L1 + 0.2 (1 - SSIM), L1, SSIM, MSE}.
constexpr int kFinishThreads = 1024;

__global__ __launch_bounds__(kFinishThreads) void image_metrics_finish_kernel(const double* __restrict__ block_sums,
    int64_t blocks, double values, double* __restrict__ out) {
    __shared__ double s_sums[3][kFinishThreads / 64];
    double sums[3] = {0.0, 0.0, 0.0};
    for (int64_t b = threadIdx.x; b < blocks; b += kFinishThreads) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            sums[k] += block_sums[b * 3 + k];
        }
    }
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            sums[k] += __shfl_xor(sums[k], offset);
        }
    }
    if ((threadIdx.x & 63) == 0) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            s_sums[k][threadIdx.x >> 6] = sums[k];
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        double total[3] = {0.0, 0.0, 0.0};
        for (int w = 0; w < kFinishThreads / 64; ++w) {
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                total[k] += s_sums[k][w];
            }
        }
        const double l1 = total[0] / values;
        const double ssim = total[1] / values;
        out[0] = 0.8 * l1 + 0.2 * (1.0 - ssim);
        out[1] = l1;
        out[2] = ssim;
        out[3] = total[2] / values;
    }
}

} // namespace

int64_t image_metric_blocks(int width, int height) {
    return static_cast<int64_t>(grid_for(width, kTw)) * grid_for(height, kTh) * 3;
}

int launch_image_metrics(gsn_context* context, int width, int height, const float* image, const uint8_t* target,
    double* block_sums, double* out) {
    dim3 grid(grid_for(width, kTw), grid_for(height, kTh), 3);
    image_metrics_kernel<<<grid, kThreads, 0, context->stream>>>(image, target, block_sums, width, height, window());
    GSN_TRY(check_launch("image_metrics_kernel"));
    const double values = 3.0 * static_cast<double>(width) * height;
    image_metrics_finish_kernel<<<1, kFinishThreads, 0, context->stream>>>(block_sums, image_metric_blocks(width, height), values,
        out);
    return check_launch("image_metrics_finish_kernel");
}

} // namespace gsn

extern "C" int gsn_image_metrics(gsn_context* context, int width, int height, const float* image,
    const uint8_t* target, double* out) {
    using namespace gsn;
    if (!context || width <= 0 || height <= 0 || !image || !target || !out) {
        return fail(GSN_ERROR_INVALID_ARGUMENT, "gsn_image_metrics: invalid arguments");
    }
    const size_t blocks = static_cast<size_t>(image_metric_blocks(width, height));
    // Block sums followed by the four results.
    double* sums = static_cast<double*>(scratch(context, kSlotReduce, (blocks * 3 + 4) * sizeof(double)));
    if (!sums) {
        return GSN_ERROR_OUT_OF_MEMORY;
    }
    double* results = sums + blocks * 3;
    GSN_TRY(launch_image_metrics(context, width, height, image, target, sums, results));
    double* host = static_cast<double*>(context->pinned);
    GSN_HIP(hipMemcpyAsync(host, results, 4 * sizeof(double), hipMemcpyDeviceToHost, context->stream));
    GSN_HIP(hipStreamSynchronize(context->stream));
    for (int k = 0; k < 4; ++k) {
        out[k] = host[k];
    }
    return GSN_OK;
}
