// Held-out evaluation of a render (reference demo/render.cpp:107-155): the float image is clamped
// to [0, 1], scaled by 255 in FP32 and rounded half to even to 8 bits (OpenCV's convertTo to
// CV_8UC3 with scale 255), and compared with the 8-bit target by the sum of squared differences
// over all pixels and channels; PSNR = -10 log10(SSE / (3 W H 255^2)), infinite for SSE = 0.
// Integer work: the sum is exact, so the result does not depend on the summation order.
#include "gsn_internal.h"

#include <algorithm>
#include <cmath>

namespace gsn {
namespace {

// At most one workgroup per CU: each leaves one sum and the host adds them (integers, exact in any
// order). With 8,192 workgroups adding to one 64-bit address the atomics alone took 100 us.
constexpr int kEvalThreads = 1024;
constexpr unsigned kEvalGroups = 256;

__device__ __forceinline__ int quantize(float value) {
    const float v = fminf(fmaxf(value, 0.0f), 1.0f);
    return static_cast<int>(rintf(v * 255.0f));
}

// Bound by memory (18 bytes a pixel): groups of four values as one 16-byte and two 4-byte accesses
// where the caller's buffers are aligned for them (Wide), value by value otherwise and at the end.
// 1332x876: 102 us with one atomic sum and a value a thread, 6.3 us so.
template<bool Wide>
__global__ __launch_bounds__(kEvalThreads) void quantized_error_kernel(const float* __restrict__ image,
    const uint8_t* __restrict__ target, uint8_t* __restrict__ quantized, int64_t values,
    unsigned long long* __restrict__ sums) {
    __shared__ unsigned long long partial[kEvalThreads / 64];
    const int64_t thread = static_cast<int64_t>(blockIdx.x) * kEvalThreads + threadIdx.x;
    const int64_t threads = static_cast<int64_t>(gridDim.x) * kEvalThreads;
    unsigned long long sum = 0;
    auto one = [&](float value, int goal) {
        const int q = quantize(value);
        const int d = q - goal;
        sum += static_cast<unsigned long long>(d * d);
        return static_cast<uint8_t>(q);
    };
    int64_t done = 0;
    if (Wide) {
        const int64_t fours = values / 4;
        for (int64_t i = thread; i < fours; i += threads) {
            const float4 v = reinterpret_cast<const float4*>(image)[i];
            const uchar4 t = reinterpret_cast<const uchar4*>(target)[i];
            uchar4 q;
            q.x = one(v.x, t.x);
            q.y = one(v.y, t.y);
            q.z = one(v.z, t.z);
            q.w = one(v.w, t.w);
            if (quantized) {
                reinterpret_cast<uchar4*>(quantized)[i] = q;
            }
        }
        done = fours * 4;
    }
    // A value an access: several of a thread's loads in flight (5187x3361: 189 us one by one, 68 so).
    constexpr int kBatch = Wide ? 1 : 8;
    for (int64_t base = done + thread; base < values; base += kBatch * threads) {
        float v[kBatch];
        uint8_t t[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            const int64_t i = min(base + j * threads, values - 1);
            v[j] = image[i];
            t[j] = target[i];
        }
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            const int64_t i = base + j * threads;
            if (i < values) {
                const uint8_t q = one(v[j], static_cast<int>(t[j]));
                if (quantized) {
                    quantized[i] = q;
                }
            }
        }
    }
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) {
        sum += __shfl_xor(sum, offset);
    }
    if ((threadIdx.x & 63) == 0) {
        partial[threadIdx.x >> 6] = sum;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long block = 0;
        for (int w = 0; w < kEvalThreads / 64; ++w) {
            block += partial[w];
        }
        sums[blockIdx.x] = block;
    }
}

} // namespace
} // namespace gsn

extern "C" int gsn_image_quantized_error(gsn_context* context, int width, int height, const float* image,
    const uint8_t* target, uint8_t* quantized, double* out) {
    using namespace gsn;
    if (!context || width <= 0 || height <= 0 || !image || !target || !out) {
        return fail(GSN_ERROR_INVALID_ARGUMENT, "gsn_image_quantized_error: invalid arguments");
    }
    const int64_t values = static_cast<int64_t>(width) * height * 3;
    auto* sums = static_cast<unsigned long long*>(
        scratch(context, kSlotQuantizedError, kEvalGroups * sizeof(unsigned long long)));
    if (!sums) {
        return GSN_ERROR_OUT_OF_MEMORY;
    }
    const unsigned blocks = std::min(grid_for(values, 4 * kEvalThreads), kEvalGroups);
    const bool wide = reinterpret_cast<uintptr_t>(image) % 16 == 0 && reinterpret_cast<uintptr_t>(target) % 4 == 0 &&
                      reinterpret_cast<uintptr_t>(quantized) % 4 == 0;
    auto* kernel = wide ? quantized_error_kernel<true> : quantized_error_kernel<false>;
    kernel<<<blocks, kEvalThreads, 0, context->stream>>>(image, target, quantized, values, sums);
    GSN_TRY(check_launch("quantized_error_kernel"));
    static_assert(kPinnedSums + kEvalGroups * sizeof(unsigned long long) <= kPinnedBytes, "room for the sums");
    auto* host = reinterpret_cast<unsigned long long*>(static_cast<char*>(context->pinned) + kPinnedSums);
    GSN_HIP(hipMemcpyAsync(host, sums, blocks * sizeof(unsigned long long), hipMemcpyDeviceToHost, context->stream));
    GSN_HIP(hipStreamSynchronize(context->stream));
    unsigned long long sse = 0;
    for (unsigned b = 0; b < blocks; ++b) {
        sse += host[b];
    }
    const double total = static_cast<double>(sse);
    out[0] = total;
    out[1] = total == 0.0 ? INFINITY : -10.0 * std::log10(total / (3.0 * width * height * 255.0 * 255.0));
    return GSN_OK;
}
