// Learned densification proposal: a 16 -> 64 -> 64 -> 3 MLP (ReLU hidden layers, logits for
// keep / clone / split) with BF16 weights and FP32 accumulation on gfx950 MFMA
// (v_mfma_f32_32x32x16_bf16). No counterpart in the reference.
//
// A wave processes tiles of 32 samples with everything in registers. An operand of a 32x32x16
// product, A (rows) or B (columns), has the same form: lane l holds row (column) l & 31 and its K
// elements 8 * (l >> 5) .. + 7 of the 16-element chunk; the result has column l & 31 in lane l and
// row 8 (v >> 2) + 4 (l >> 5) + (v & 3) in register v. So mfma(weights, samples) gives samples in
// lanes and features in registers ("by sample"), mfma(samples, weights) the other way round ("by
// feature"), with the same bits; and a result whose lane is the next product's row becomes its
// operand by converting to BF16 and exchanging four-element pieces between the wave's halves
// (operand_chunk). No transposition through LDS, and weights stay in registers across tiles. (Staging
// both layouts of weights and activations in LDS took 58 KB per one-wave workgroup, two waves per CU.)
// Forward: Z1 = X W1^T + b1, A1 = relu(Z1); Z2 = A1 W2^T + b2, A2 = relu(Z2); Z3 = A2 W3^T + b3.
// Backward (softmax cross-entropy): dZ3 = w (softmax(Z3) - onehot) / sum(w); dW3 = dZ3^T A2;
// dA2 = dZ3 W3; dZ2 = dA2 [Z2 > 0]; dW2 = dZ2^T A1; dA1 = dZ2 W2; dZ1 = dA1 [Z1 > 0];
// dW1 = dZ1^T X; db = column sums of dZ. MFMA operands are BF16 (X, weights, A1, A2, dZ*),
// accumulation and the softmax are FP32. Weight gradients are accumulated per workgroup and
// reduced in a fixed order by the Adam kernel (deterministic).
#include "gsn_internal.h"

#include <algorithm>
#include <cmath>

namespace gsn {
namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

constexpr int kIn = 16;
constexpr int kHidden = 64;
constexpr int kClasses = 3;
// FP32 parameter block: W1[64][16], b1[64], W2[64][64], b2[64], W3[3][64], b3[3].
constexpr int kW1 = 0;
constexpr int kB1 = kW1 + kHidden * kIn;
constexpr int kW2 = kB1 + kHidden;
constexpr int kB2 = kW2 + kHidden * kHidden;
constexpr int kW3 = kB2 + kHidden;
constexpr int kB3 = kW3 + kClasses * kHidden;
constexpr int kParams = kB3 + kClasses;  // 5443
// BF16 weight block: W1[64][16], W2[64][64], W3 padded to [32][64].
constexpr int kBfW1 = 0;
constexpr int kBfW2 = kBfW1 + kHidden * kIn;
constexpr int kBfW3 = kBfW2 + kHidden * kHidden;
constexpr int kBfWeights = kBfW3 + 32 * kHidden;  // 7168

__device__ __forceinline__ f32x16 mfma(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ int d_row(int lane, int v) {
    return ((v >> 2) << 3) + ((lane >> 5) << 2) + (v & 3);
}

// Chunk c (0, 1) of the operand that continues a 32x32 result: K elements 16 c .. 16 c + 15 of the
// result's rows. Per half the lane holds rows 16 c + 4 h + (0..3) and 16 c + 8 + 4 h + (0..3); the
// swap gives half 0 the first eight and half 1 the last eight.
__device__ __forceinline__ bf16x8 operand_chunk(const float (&values)[16], int c) {
    union Pieces {
        __bf16 b[8];
        uint32_t u[4];
        bf16x8 v;
    } piece;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        piece.b[i] = static_cast<__bf16>(values[8 * c + i]);
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        auto swapped = __builtin_amdgcn_permlane32_swap(piece.u[i], piece.u[2 + i], false, false);
        piece.u[i] = swapped[0];
        piece.u[2 + i] = swapped[1];
    }
    return piece.v;
}

__device__ __forceinline__ bf16x8 zero_operand() {
    bf16x8 zero = {};
    return zero;
}

// Sixteen bytes from an address with no alignment beyond its elements' (the caller's buffers): one
// wide load, which global memory serves at any element address.
template<typename Wide, typename Element>
__device__ __forceinline__ Wide load_wide(const Element* address) {
    Wide value;
    __builtin_memcpy(&value, address, sizeof(value));
    return value;
}

// Operands of the weight matrices, one row of the matrix per lane.
struct ForwardWeights {
    bf16x8 w1[2];     // rows 32 b + l, K = the 16 inputs
    bf16x8 w2[2][4];  // rows 32 b + l, K chunks of the 64 hidden units
    bf16x8 w3[4];     // rows l (3..31 zero padding), K chunks
};

__device__ __forceinline__ ForwardWeights load_forward_weights(const __bf16* __restrict__ weights) {
    const int lane = threadIdx.x & 63;
    const int row = lane & 31, k8 = (lane >> 5) * 8;
    ForwardWeights w;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        w.w1[b] = load_wide<bf16x8>(weights + kBfW1 + (32 * b + row) * kIn + k8);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            w.w2[b][c] = load_wide<bf16x8>(weights + kBfW2 + (32 * b + row) * kHidden + 16 * c + k8);
        }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        w.w3[c] = load_wide<bf16x8>(weights + kBfW3 + row * kHidden + 16 * c + k8);
    }
    return w;
}

// A tile's inputs by sample: lane's sample, inputs 8 h .. + 7 (zero past the last sample).
struct TileInputs {
    float4 low, high;
};

__device__ __forceinline__ TileInputs load_inputs(const float* __restrict__ features, int64_t first, int count) {
    const int lane = threadIdx.x & 63;
    const int64_t sample = first + (lane & 31);
    TileInputs x;
    x.low = x.high = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    if (sample < count) {
        const float* row = features + sample * kIn + (lane >> 5) * 8;
        x.low = load_wide<float4>(row);
        x.high = load_wide<float4>(row + 4);
    }
    return x;
}

__device__ __forceinline__ bf16x8 input_operand(const TileInputs& x) {
    const float v[8] = {x.low.x, x.low.y, x.low.z, x.low.w, x.high.x, x.high.y, x.high.z, x.high.w};
    bf16x8 out;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        out[i] = static_cast<__bf16>(v[i]);
    }
    return out;
}

// values += bias of each row of a by-sample result (rows 32 b + d_row); bias is in LDS, four
// consecutive rows a read.
__device__ __forceinline__ void add_row_bias(float (&values)[16], const f32x16& acc, const float* bias, int b) {
    const int half = (threadIdx.x >> 5) & 1;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const float4 four = *reinterpret_cast<const float4*>(bias + 32 * b + 8 * g + 4 * half);
        values[4 * g] = acc[4 * g] + four.x;
        values[4 * g + 1] = acc[4 * g + 1] + four.y;
        values[4 * g + 2] = acc[4 * g + 2] + four.z;
        values[4 * g + 3] = acc[4 * g + 3] + four.w;
    }
}

__device__ __forceinline__ void relu(const float (&in)[16], float (&out)[16]) {
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        out[v] = fmaxf(in[v], 0.0f);
    }
}

// The by-sample hidden layers of a tile: pre-activations z (before the ReLU) of both layers and the
// operands of the activations.
struct HiddenLayers {
    bf16x8 a1[4], a2[4];
};

__device__ __forceinline__ void hidden_layers(const ForwardWeights& w, const float* bias1, const float* bias2, bf16x8 x,
    HiddenLayers& layers, float (&z2)[2][16]) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        float z[16], a[16];
        add_row_bias(z, mfma(w.w1[b], x, f32x16{}), bias1, b);
        relu(z, a);
        layers.a1[2 * b] = operand_chunk(a, 0);
        layers.a1[2 * b + 1] = operand_chunk(a, 1);
    }
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        f32x16 acc = {};
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            acc = mfma(w.w2[b][c], layers.a1[c], acc);
        }
        float a[16];
        add_row_bias(z2[b], acc, bias2, b);
        relu(z2[b], a);
        layers.a2[2 * b] = operand_chunk(a, 0);
        layers.a2[2 * b + 1] = operand_chunk(a, 1);
    }
}

// The logits of lane's sample: classes 0..2 in registers 0..2 of the lanes below 32.
__device__ __forceinline__ f32x16 output_layer(const ForwardWeights& w, const HiddenLayers& layers) {
    f32x16 acc = {};
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        acc = mfma(w.w3[c], layers.a2[c], acc);
    }
    return acc;
}

// The two hidden layers' biases in LDS; every wave of the workgroup reads them.
__device__ __forceinline__ void stage_biases(const float* __restrict__ biases, float* bias1, float* bias2) {
    if (threadIdx.x < kHidden) {
        bias1[threadIdx.x] = biases[kB1 + threadIdx.x];
        bias2[threadIdx.x] = biases[kB2 + threadIdx.x];
    }
    __syncthreads();
}

constexpr int kMlpWaves = 4;  // per workgroup

// 76 bytes and 10.6 kFLOP a sample: bound by memory once enough waves are in flight; the next tile's
// inputs are loaded while one is computed. 500K samples: 205 us with tiles
// staged through LDS by one wave per workgroup, 21 us so.
__global__ __launch_bounds__(64 * kMlpWaves) void mlp_forward_kernel(const float* __restrict__ features, int count,
    const __bf16* __restrict__ weights, const float* __restrict__ biases, float* __restrict__ logits) {
    __shared__ __align__(16) float bias1[kHidden], bias2[kHidden];
    stage_biases(biases, bias1, bias2);
    const ForwardWeights w = load_forward_weights(weights);
    const float bias3[kClasses] = {biases[kB3], biases[kB3 + 1], biases[kB3 + 2]};
    const int lane = threadIdx.x & 63;
    const int tiles = (count + 31) / 32;
    const int stride = static_cast<int>(gridDim.x) * kMlpWaves;
    int tile = static_cast<int>(blockIdx.x) * kMlpWaves + static_cast<int>(threadIdx.x >> 6);
    TileInputs next = load_inputs(features, static_cast<int64_t>(tile) * 32, count);
    for (; tile < tiles; tile += stride) {
        const bf16x8 x = input_operand(next);
        next = load_inputs(features, (static_cast<int64_t>(tile) + stride) * 32, count);
        HiddenLayers layers;
        float z2[2][16];
        hidden_layers(w, bias1, bias2, x, layers, z2);
        const f32x16 out = output_layer(w, layers);
        const int64_t sample = static_cast<int64_t>(tile) * 32 + lane;
        if (lane < 32 && sample < count) {
#pragma unroll
            for (int c = 0; c < kClasses; ++c) {
                logits[sample * kClasses + c] = out[c] + bias3[c];
            }
        }
    }
}

// Forward + backward over the workgroup's tiles; writes its gradient sums (parameter layout) and
// loss sum to partials[blockIdx.x]. A wave keeps its sums in registers (seven 32x32 results); at the
// end the workgroup adds its waves' sums through LDS, wave by wave, so that every order is fixed.
// Weight gradients sum over the samples, so their operands need samples as K: the by-feature
// results, computed by a second product of the same operands in the other order. Bound by the chain of
// products of a tile at four waves per CU; 65,536 samples: 75 us with the activations kept in LDS for
// the transposed reads, 29 us so.
__global__ __launch_bounds__(64 * kMlpWaves, 1) void mlp_gradient_kernel(const float* __restrict__ features,
    const int* __restrict__ labels, const float* __restrict__ sample_weights, int count, float weight_scale,
    const __bf16* __restrict__ weights, const float* __restrict__ biases, float* __restrict__ partials,
    float* __restrict__ loss_partials) {
    __shared__ __align__(16) float bias1[kHidden], bias2[kHidden];
    __shared__ __align__(16) __bf16 s_dz3[kMlpWaves][kClasses][32];  // [class][sample]
    __shared__ float s_sum[kParams + 1];                             // gradients, then the loss
    stage_biases(biases, bias1, bias2);
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    const int n = lane & 31;
    const int half = lane >> 5;
    const int k8 = half * 8;
    const ForwardWeights w = load_forward_weights(weights);
    // Operands of the transposed matrices: rows are the hidden units 32 b + n.
    bf16x8 w3t[2], w2t[2][4];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        w3t[b] = zero_operand();
        if (half == 0) {
#pragma unroll
            for (int c = 0; c < kClasses; ++c) {
                w3t[b][c] = weights[kBfW3 + c * kHidden + 32 * b + n];
            }
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                w2t[b][c][i] = weights[kBfW2 + (16 * c + k8 + i) * kHidden + 32 * b + n];
            }
        }
    }
    const float bias3[kClasses] = {biases[kB3], biases[kB3 + 1], biases[kB3 + 2]};
    const float own_bias1[2] = {bias1[n], bias1[32 + n]}, own_bias2[2] = {bias2[n], bias2[32 + n]};
    f32x16 gw1[2] = {}, gw2[4] = {}, gw3[2] = {};
    float gb1[2] = {0.0f, 0.0f}, gb2[2] = {0.0f, 0.0f}, gb3[kClasses] = {0.0f, 0.0f, 0.0f};
    float loss = 0.0f;
    const int tiles = (count + 31) / 32;
    for (int tile = blockIdx.x * kMlpWaves + wave; tile < tiles; tile += gridDim.x * kMlpWaves) {
        const int64_t first = static_cast<int64_t>(tile) * 32;
        const bf16x8 x = input_operand(load_inputs(features, first, count));
        // The inputs by feature (lane = input, 16..31 zero): samples 16 c + 8 h .. + 7.
        bf16x8 xt[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const int64_t sample = first + 16 * c + k8 + i;
                xt[c][i] = static_cast<__bf16>(n < kIn && sample < count ? features[sample * kIn + n] : 0.0f);
            }
        }
        HiddenLayers layers;
        float z2[2][16];
        hidden_layers(w, bias1, bias2, x, layers, z2);
        const f32x16 out = output_layer(w, layers);
        // Softmax cross-entropy, one lane per sample.
        bf16x8 dz3 = zero_operand();
        if (half == 0) {
            const bool valid = first + n < count;
            const float weight = valid ? (sample_weights ? sample_weights[first + n] : 1.0f) * weight_scale : 0.0f;
            const int label = valid ? labels[first + n] : 0;
            const float l0 = out[0] + bias3[0], l1 = out[1] + bias3[1], l2 = out[2] + bias3[2];
            const float top = fmaxf(l0, fmaxf(l1, l2));
            const float e0 = __expf(l0 - top), e1 = __expf(l1 - top), e2 = __expf(l2 - top);
            const float sum = e0 + e1 + e2;
            const float p[3] = {e0 / sum, e1 / sum, e2 / sum};
            const float chosen = label == 0 ? l0 : (label == 1 ? l1 : l2);
            if (valid) {
                loss += weight * (top + __logf(sum) - chosen);
            }
#pragma unroll
            for (int c = 0; c < kClasses; ++c) {
                dz3[c] = static_cast<__bf16>(weight * (p[c] - (c == label ? 1.0f : 0.0f)));
                s_dz3[wave][c][n] = dz3[c];
                gb3[c] += static_cast<float>(dz3[c]);
            }
        }
        wave_lds_fence();
        bf16x8 dz3t[2];
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            dz3t[c] = n < kClasses ? *reinterpret_cast<const bf16x8*>(&s_dz3[wave][n][16 * c + k8]) : zero_operand();
        }
        wave_lds_fence();
        // By feature: the activations of both layers, and dZ2 and dZ1 with them.
        bf16x8 dz2[4], dz2t[2][2], a1t[2][2];
        float z1t[2][16];
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const f32x16 first_layer = mfma(x, w.w1[b], f32x16{});
            f32x16 second_layer = {};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                second_layer = mfma(layers.a1[c], w.w2[b][c], second_layer);
            }
            float z2t[16], a[16];
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                z1t[b][v] = first_layer[v] + own_bias1[b];
                z2t[v] = second_layer[v] + own_bias2[b];
            }
            relu(z1t[b], a);
            a1t[b][0] = operand_chunk(a, 0);
            a1t[b][1] = operand_chunk(a, 1);
            relu(z2t, a);
            // dW3 (rows = class, columns = hidden, K = samples).
            gw3[b] = mfma(dz3t[0], operand_chunk(a, 0), gw3[b]);
            gw3[b] = mfma(dz3t[1], operand_chunk(a, 1), gw3[b]);
            // dA2 = dZ3 W3, masked by Z2 > 0: by sample for dA1, by feature for dW2.
            const f32x16 da2 = mfma(w3t[b], dz3, f32x16{});
            const f32x16 da2t = mfma(dz3, w3t[b], f32x16{});
            float g[16], gt[16], column = 0.0f;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                g[v] = z2[b][v] > 0.0f ? da2[v] : 0.0f;
                gt[v] = z2t[v] > 0.0f ? da2t[v] : 0.0f;
                column += static_cast<float>(static_cast<__bf16>(gt[v]));
            }
            gb2[b] += column;
            dz2[2 * b] = operand_chunk(g, 0);
            dz2[2 * b + 1] = operand_chunk(g, 1);
            dz2t[b][0] = operand_chunk(gt, 0);
            dz2t[b][1] = operand_chunk(gt, 1);
        }
        // dW2 (rows = out, columns = in, K = samples).
#pragma unroll
        for (int mb = 0; mb < 2; ++mb) {
#pragma unroll
            for (int nb = 0; nb < 2; ++nb) {
                gw2[mb * 2 + nb] = mfma(dz2t[mb][0], a1t[nb][0], gw2[mb * 2 + nb]);
                gw2[mb * 2 + nb] = mfma(dz2t[mb][1], a1t[nb][1], gw2[mb * 2 + nb]);
            }
        }
        // dA1 = dZ2 W2 by feature, masked by Z1 > 0; dW1 (rows = out, columns = input, K = samples).
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            f32x16 acc = {};
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                acc = mfma(dz2[c], w2t[b][c], acc);
            }
            float g[16], column = 0.0f;
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                g[v] = z1t[b][v] > 0.0f ? acc[v] : 0.0f;
                column += static_cast<float>(static_cast<__bf16>(g[v]));
            }
            gb1[b] += column;
            gw1[b] = mfma(operand_chunk(g, 0), xt[0], gw1[b]);
            gw1[b] = mfma(operand_chunk(g, 1), xt[1], gw1[b]);
        }
    }
    // Sums over the workgroup's waves, in wave order. A result's lane column is n, its register rows
    // d_row(lane, v); a bias's two halves of rows meet first.
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        gb1[b] += __shfl_xor(gb1[b], 32);
        gb2[b] += __shfl_xor(gb2[b], 32);
    }
#pragma unroll
    for (int offset = 16; offset > 0; offset >>= 1) {
        loss += __shfl_xor(loss, offset);
#pragma unroll
        for (int c = 0; c < kClasses; ++c) {
            gb3[c] += __shfl_xor(gb3[c], offset);
        }
    }
    for (int turn = 0; turn < kMlpWaves; ++turn) {
        if (wave == turn) {
            auto add = [&](int at, float value) { s_sum[at] = turn == 0 ? value : s_sum[at] + value; };
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const int row = d_row(lane, v);
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    if (n < kIn) {
                        add(kW1 + (32 * b + row) * kIn + n, gw1[b][v]);
                    }
                    add(kW2 + (32 * b + row) * kHidden + n, gw2[2 * b][v]);
                    add(kW2 + (32 * b + row) * kHidden + 32 + n, gw2[2 * b + 1][v]);
                    if (row < kClasses) {
                        add(kW3 + row * kHidden + 32 * b + n, gw3[b][v]);
                    }
                }
            }
            if (half == 0) {
#pragma unroll
                for (int b = 0; b < 2; ++b) {
                    add(kB1 + 32 * b + n, gb1[b]);
                    add(kB2 + 32 * b + n, gb2[b]);
                }
                if (n < kClasses) {
                    add(kB3 + n, n == 0 ? gb3[0] : (n == 1 ? gb3[1] : gb3[2]));
                }
                if (n == 0) {
                    add(kParams, loss);
                }
            }
        }
        __syncthreads();
    }
    float* out = partials + static_cast<int64_t>(blockIdx.x) * kParams;
    for (int i = threadIdx.x; i < kParams; i += 64 * kMlpWaves) {
        out[i] = s_sum[i];
    }
    if (threadIdx.x == 0) {
        loss_partials[blockIdx.x] = s_sum[kParams];
    }
}

// Sums the workgroups' gradients in a fixed order, applies Adam to the FP32 master parameters
// and refreshes the BF16 weight copy. gradients_out (optional) receives the summed gradients.
// A workgroup has kAdamParams parameters and kAdamSegments runs of the partials' rows; each run is
// added by its own threads (coalesced, many loads in flight), then the runs in order. (One thread
// per parameter over 1,024 rows one after another took 245 us; so, over 256 rows, 4.8.)
constexpr int kAdamParams = 32;
constexpr int kAdamSegments = 16;

__global__ __launch_bounds__(kAdamParams * kAdamSegments) void mlp_adam_kernel(const float* __restrict__ partials,
    int groups, float* __restrict__ params, float* __restrict__ first, float* __restrict__ second,
    __bf16* __restrict__ weights, float learning_rate, float first_correction, float second_correction,
    float* __restrict__ gradients_out) {
    __shared__ float s_sum[kAdamSegments][kAdamParams];
    const int segment = threadIdx.x / kAdamParams;
    const int p = blockIdx.x * kAdamParams + threadIdx.x % kAdamParams;
    const int rows = (groups + kAdamSegments - 1) / kAdamSegments;
    const int begin = min(segment * rows, groups), end = min(begin + rows, groups);
    float sum = 0.0f;
    if (p < kParams) {
#pragma unroll 8
        for (int row = begin; row < end; ++row) {
            sum += partials[static_cast<int64_t>(row) * kParams + p];
        }
    }
    s_sum[segment][threadIdx.x % kAdamParams] = sum;
    __syncthreads();
    if (segment != 0 || p >= kParams) {
        return;
    }
    float g = 0.0f;
#pragma unroll
    for (int k = 0; k < kAdamSegments; ++k) {
        g += s_sum[k][threadIdx.x];
    }
    if (gradients_out) {
        gradients_out[p] = g;
    }
    if (learning_rate > 0.0f) {
        float m = 0.9f * first[p] + 0.1f * g;
        float v = 0.999f * second[p] + 0.001f * g * g;
        first[p] = m;
        second[p] = v;
        params[p] -= learning_rate * (m * first_correction) / (sqrtf(v * second_correction) + 1e-8f);
    }
    float value = params[p];
    if (p < kB1) {
        weights[kBfW1 + p] = static_cast<__bf16>(value);
    }
    else if (p >= kW2 && p < kB2) {
        weights[kBfW2 + (p - kW2)] = static_cast<__bf16>(value);
    }
    else if (p >= kW3 && p < kB3) {
        weights[kBfW3 + (p - kW3)] = static_cast<__bf16>(value);
    }
}

__global__ void mlp_zero_padding_kernel(__bf16* weights) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < (32 - kClasses) * kHidden) {
        weights[kBfW3 + kClasses * kHidden + i] = static_cast<__bf16>(0.0f);
    }
}

// Workgroups of kMlpWaves tiles each, at most `most`; beyond that the waves take several tiles.
int mlp_groups(int count, int most) {
    const int64_t tiles = (static_cast<int64_t>(count) + 31) / 32;
    return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>((tiles + kMlpWaves - 1) / kMlpWaves, most)));
}

// Forward: four workgroups a CU hide the loads. Training: one a CU, whose waves' gradient sums take
// most of the registers; more would also mean more partials to add.
constexpr int kForwardGroups = 1024;
constexpr int kTrainingGroups = 256;

} // namespace
} // namespace gsn

extern "C" int gsn_mlp_sizes(int* parameters, int* bf16_weights) {
    if (!parameters || !bf16_weights) {
        return gsn::fail(GSN_ERROR_INVALID_ARGUMENT, "gsn_mlp_sizes: null output");
    }
    *parameters = gsn::kParams;
    *bf16_weights = gsn::kBfWeights;
    return GSN_OK;
}

extern "C" int gsn_mlp_sync_weights(gsn_context* context, const float* params, uint16_t* weights) {
    using namespace gsn;
    if (!context || !params || !weights) {
        return fail(GSN_ERROR_INVALID_ARGUMENT, "gsn_mlp_sync_weights: null argument");
    }
    mlp_zero_padding_kernel<<<grid_for((32 - kClasses) * kHidden, 256), 256, 0, context->stream>>>(
        reinterpret_cast<__bf16*>(weights));
    GSN_TRY(check_launch("mlp_zero_padding_kernel"));
    mlp_adam_kernel<<<grid_for(kParams, kAdamParams), kAdamParams * kAdamSegments, 0, context->stream>>>(nullptr, 0, const_cast<float*>(params),
        nullptr, nullptr, reinterpret_cast<__bf16*>(weights), 0.0f, 0.0f, 0.0f, nullptr);
    return check_launch("mlp_adam_kernel");
}

extern "C" int gsn_mlp_forward(gsn_context* context, const float* features, int count, const uint16_t* weights,
    const float* params, float* logits) {
    using namespace gsn;
    if (!context || count < 0 || (count > 0 && (!features || !weights || !params || !logits))) {
        return fail(GSN_ERROR_INVALID_ARGUMENT, "gsn_mlp_forward: invalid arguments");
    }
    if (count == 0) {
        return GSN_OK;
    }
    mlp_forward_kernel<<<mlp_groups(count, kForwardGroups), 64 * kMlpWaves, 0, context->stream>>>(features, count,
        reinterpret_cast<const __bf16*>(weights), params, logits);
    return check_launch("mlp_forward_kernel");
}

extern "C" int gsn_mlp_train_step(gsn_context* context, const float* features, const int32_t* labels,
    const float* sample_weights, int count, float* params, float* first, float* second, uint16_t* weights,
    float learning_rate, int step, float* gradients_out, double* loss_out) {
    using namespace gsn;
    if (!context || count <= 0 || !features || !labels || !params || !weights || step < 1 ||
        !(learning_rate >= 0.0f) || (learning_rate > 0.0f && (!first || !second))) {
        return fail(GSN_ERROR_INVALID_ARGUMENT, "gsn_mlp_train_step: invalid arguments");
    }
    int groups = mlp_groups(count, kTrainingGroups);
    float* partials = static_cast<float*>(scratch(context, kSlotMisc, static_cast<size_t>(groups) * (kParams + 1) * 4));
    if (!partials) {
        return GSN_ERROR_OUT_OF_MEMORY;
    }
    float* loss_partials = partials + static_cast<size_t>(groups) * kParams;
    float weight_scale = 1.0f / static_cast<float>(count);
    mlp_gradient_kernel<<<groups, 64 * kMlpWaves, 0, context->stream>>>(features, labels, sample_weights, count, weight_scale,
        reinterpret_cast<const __bf16*>(weights), params, partials, loss_partials);
    GSN_TRY(check_launch("mlp_gradient_kernel"));
    float c1 = static_cast<float>(1.0 / (1.0 - std::pow(0.9, step)));
    float c2 = static_cast<float>(1.0 / (1.0 - std::pow(0.999, step)));
    mlp_adam_kernel<<<grid_for(kParams, kAdamParams), kAdamParams * kAdamSegments, 0, context->stream>>>(partials, groups, params, first, second,
        reinterpret_cast<__bf16*>(weights), learning_rate, c1, c2, gradients_out);
    GSN_TRY(check_launch("mlp_adam_kernel"));
    if (loss_out) {
        float* host = new float[groups];
        GSN_HIP(hipMemcpyAsync(host, loss_partials, groups * sizeof(float), hipMemcpyDeviceToHost, context->stream));
        GSN_HIP(hipStreamSynchronize(context->stream));
        double total = 0.0;
        for (int b = 0; b < groups; ++b) {
            total += host[b];
        }
        delete[] host;
        *loss_out = total;
    }
    return GSN_OK;
}
