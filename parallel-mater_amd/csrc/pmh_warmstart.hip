// SPDX-License-Identifier: MIT
//
// Learned warm start (no counterpart in the reference, whose cold contacts
// start from lambda = 0 and the pair stiffness, geometry_constraints.slang:
// 1366-1373): a 16 -> 64 -> 64 -> 2 perceptron with ReLU, BF16 weights and
// activations on MFMA (v_mfma_f32_16x16x16_bf16) with FP32 accumulation,
// predicting the normal row's dual (lambda, penalty) of each cold contact
// point from 16 features computed at contact preparation.  Trained on the
// GPU by the kernels below from contact samples that plain AVBD logs.
//
// Every product is a 16x16 MFMA tile C += A(16 x K) B(K x 16).  The forward
// passes and training read both operands as padded rows along K, four values
// in one 8-byte LDS access (200000 rows forward: 143 us with 2-byte reads at
// strides whose rows share a bank, now 101); the gradients of one minibatch
// read transposed operands through strides.
// Lane l supplies A[l % 16][k0 + 4(l / 16) + j] and B[k0 + 4(l / 16) + j][l % 16]
// (j = 0..3) and receives C[4(l / 16) + e][l % 16] (e = 0..3).

#include "pmh_internal.hpp"
#include "pmh_warmstart.hpp"

#include <cmath>
#include <vector>

namespace pmh {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__host__ __device__ inline uint16_t to_bf16(float f) {
    uint32_t u;
    memcpy(&u, &f, 4);
    const uint32_t nan = (u >> 16) | 0x40u;                                    // NaN stays NaN
    const uint32_t even = (u + 0x7fffu + ((u >> 16) & 1u)) >> 16;              // round to nearest even
    return uint16_t((u & 0x7fffffffu) > 0x7f800000u ? nan : even);
}
__host__ __device__ inline float from_bf16(uint16_t h) {
    const uint32_t u = uint32_t(h) << 16;
    float f;
    memcpy(&f, &u, 4);
    return f;
}

__device__ __forceinline__ f32x4 mma_tile(const uint16_t *A, int sai, int sak, const uint16_t *B, int sbk, int sbj,
                                          int K, f32x4 acc) {
    const int l = threadIdx.x & 63, r = l & 15, q = (l >> 4) * 4;
    for (int k0 = 0; k0 < K; k0 += 16) {
        bf16x4 a, b;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            a[j] = short(A[r * sai + (k0 + q + j) * sak]);
            b[j] = short(B[(k0 + q + j) * sbk + r * sbj]);
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
    }
    return acc;
}

constexpr int kRow = 68;                       // halves per 64-wide row: 34 banks apart
constexpr int kNarrow = 20;                    // halves per 16-wide row
// One tile: rows of A and rows of B (the right operand transposed), both along K.
template <int K>
__device__ __forceinline__ f32x4 mma_rows(const uint16_t *A, int sa, const uint16_t *B, int sb, f32x4 acc) {
    const int l = threadIdx.x & 63, r = l & 15, q = (l >> 4) * 4;
#pragma unroll
    for (int k0 = 0; k0 < K; k0 += 16) {
        const bf16x4 a = *reinterpret_cast<const bf16x4 *>(A + r * sa + k0 + q);
        const bf16x4 b = *reinterpret_cast<const bf16x4 *>(B + r * sb + k0 + q);
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
    }
    return acc;
}
// Operands of one 64-sample pass, bf16 in LDS.
struct alignas(16) MlpShared {
    uint16_t w1[kMlpHidden * kNarrow];         // [out][in]
    uint16_t w2[kMlpHidden * kRow];            // [out][in]
    uint16_t w3[16 * kRow];                    // [out][in], rows 2..15 zero
    float b1[kMlpHidden], b2[kMlpHidden], b3[16];
    uint16_t x[64 * kNarrow];                  // [sample][feature]
    uint16_t h1[64 * kRow], h2[64 * kRow];
    uint16_t dy[64 * 16];                      // [sample][out], cols 2..15 zero
    uint16_t dz2[64 * kRow], dz1[64 * kRow];
    float y[64 * kMlpOut], t[64 * kMlpOut];
};

__device__ void load_weights(MlpShared &S, const float *p) {
    const int l = threadIdx.x;
    for (int k = l; k < kMlpHidden * kMlpIn; k += 64) S.w1[k / kMlpIn * kNarrow + k % kMlpIn] = to_bf16(p[kMlpW1 + k]);
    for (int k = l; k < kMlpHidden * kMlpHidden; k += 64) S.w2[k / kMlpHidden * kRow + k % kMlpHidden] = to_bf16(p[kMlpW2 + k]);
    for (int k = l; k < 16 * kMlpHidden; k += 64) S.w3[k / kMlpHidden * kRow + k % kMlpHidden] = k < kMlpOut * kMlpHidden ? to_bf16(p[kMlpW3 + k]) : 0;
    for (int k = l; k < kMlpHidden; k += 64) {
        S.b1[k] = p[kMlpB1 + k];
        S.b2[k] = p[kMlpB2 + k];
    }
    if (l < 16) S.b3[l] = l < kMlpOut ? p[kMlpB3 + l] : 0.0f;
}

// Forward pass of the 64 samples in S.x: h1, h2 (bf16, after ReLU) and y.
__device__ void forward(MlpShared &S) {
    const int l = threadIdx.x, r = l & 15, q = (l >> 4) * 4;
    for (int mi = 0; mi < 4; ++mi)
        for (int nj = 0; nj < 4; ++nj) {
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
            acc = mma_rows<kMlpIn>(S.x + mi * 16 * kNarrow, kNarrow, S.w1 + nj * 16 * kNarrow, kNarrow, acc);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int s = mi * 16 + q + e, o = nj * 16 + r;
                S.h1[s * kRow + o] = to_bf16(fmaxf(acc[e] + S.b1[o], 0.0f));
            }
        }
    __syncthreads();
    for (int mi = 0; mi < 4; ++mi)
        for (int nj = 0; nj < 4; ++nj) {
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
            acc = mma_rows<kMlpHidden>(S.h1 + mi * 16 * kRow, kRow, S.w2 + nj * 16 * kRow, kRow, acc);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int s = mi * 16 + q + e, o = nj * 16 + r;
                S.h2[s * kRow + o] = to_bf16(fmaxf(acc[e] + S.b2[o], 0.0f));
            }
        }
    __syncthreads();
    for (int mi = 0; mi < 4; ++mi) {
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        acc = mma_rows<kMlpHidden>(S.h2 + mi * 16 * kRow, kRow, S.w3, kRow, acc);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int s = mi * 16 + q + e;
            if (r < kMlpOut) S.y[s * kMlpOut + r] = acc[e] + S.b3[r];
        }
    }
    __syncthreads();
}

// Mean-squared-error gradients of the 64 samples (weights of `count` of
// them, the rest padding) into g[kMlpParams]; returns the summed squared
// error.  Bias gradients are FP32 sums, in sample order, of the bf16 deltas.
__device__ float backward(MlpShared &S, uint32_t count, float *g) {
    const int l = threadIdx.x, r = l & 15, q = (l >> 4) * 4;
    const float scale = 2.0f / float(count * kMlpOut);
    float sq = 0.0f;
    {   // dY, one sample per lane
        const int s = l;
        for (int o = 0; o < 16; ++o) {
            float d = 0.0f;
            if (o < kMlpOut && uint32_t(s) < count) {
                const float e = S.y[s * kMlpOut + o] - S.t[s * kMlpOut + o];
                sq += e * e;
                d = scale * e;
            }
            S.dy[s * 16 + o] = to_bf16(d);
        }
    }
    __syncthreads();
    // dW3 = dY^T H2, db3
    for (int nj = 0; nj < 4; ++nj) {
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        acc = mma_tile(S.dy, 1, 16, S.h2 + nj * 16, kRow, 1, 64, acc);
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (q + e < kMlpOut) g[kMlpW3 + (q + e) * kMlpHidden + nj * 16 + r] = acc[e];
    }
    if (l < kMlpOut) {
        float b = 0.0f;
        for (int s = 0; s < 64; ++s) b += from_bf16(S.dy[s * 16 + l]);
        g[kMlpB3 + l] = b;
    }
    // dZ2 = (dY W3) .* [H2 > 0]
    for (int mi = 0; mi < 4; ++mi)
        for (int nj = 0; nj < 4; ++nj) {
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
            acc = mma_tile(S.dy + mi * 16 * 16, 16, 1, S.w3 + nj * 16, kRow, 1, 16, acc);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int s = mi * 16 + q + e, o = nj * 16 + r;
                S.dz2[s * kRow + o] = from_bf16(S.h2[s * kRow + o]) > 0.0f ? to_bf16(acc[e]) : 0;
            }
        }
    __syncthreads();
    // dW2 = dZ2^T H1, db2
    for (int mi = 0; mi < 4; ++mi)
        for (int nj = 0; nj < 4; ++nj) {
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
            acc = mma_tile(S.dz2 + mi * 16, 1, kRow, S.h1 + nj * 16, kRow, 1, 64, acc);
#pragma unroll
            for (int e = 0; e < 4; ++e) g[kMlpW2 + (mi * 16 + q + e) * kMlpHidden + nj * 16 + r] = acc[e];
        }
    {
        float b = 0.0f;
        for (int s = 0; s < 64; ++s) b += from_bf16(S.dz2[s * kRow + l]);
        g[kMlpB2 + l] = b;
    }
    // dZ1 = (dZ2 W2) .* [H1 > 0]
    for (int mi = 0; mi < 4; ++mi)
        for (int nj = 0; nj < 4; ++nj) {
            f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
            acc = mma_tile(S.dz2 + mi * 16 * kRow, kRow, 1, S.w2 + nj * 16, kRow, 1, kMlpHidden, acc);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int s = mi * 16 + q + e, o = nj * 16 + r;
                S.dz1[s * kRow + o] = from_bf16(S.h1[s * kRow + o]) > 0.0f ? to_bf16(acc[e]) : 0;
            }
        }
    __syncthreads();
    // dW1 = dZ1^T X, db1
    for (int mi = 0; mi < 4; ++mi) {
        f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
        acc = mma_tile(S.dz1 + mi * 16, 1, kRow, S.x, kNarrow, 1, 64, acc);
#pragma unroll
        for (int e = 0; e < 4; ++e) g[kMlpW1 + (mi * 16 + q + e) * kMlpIn + r] = acc[e];
    }
    {
        float b = 0.0f;
        for (int s = 0; s < 64; ++s) b += from_bf16(S.dz1[s * kRow + l]);
        g[kMlpB1 + l] = b;
    }
    // summed squared error over the wave
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) sq += __shfl_xor(sq, d, 64);
    return sq;
}

// Samples [first, first + count) (count <= 64) into S.x / S.t.
__device__ void load_samples(MlpShared &S, const float *samples, uint32_t first, uint32_t count) {
    const int l = threadIdx.x;
    const bool live = uint32_t(l) < count;
    const float *row = samples + size_t(first + (live ? l : 0)) * kMlpSample;
    for (int f = 0; f < kMlpIn; ++f) S.x[l * kNarrow + f] = live ? to_bf16(row[f]) : 0;
    for (int o = 0; o < kMlpOut; ++o) S.t[l * kMlpOut + o] = live ? row[kMlpIn + o] : 0.0f;
    __syncthreads();
}

// Gradients of one minibatch (no update).
__global__ void __launch_bounds__(64) k_mlp_gradients(const float *samples, uint32_t count, const float *params,
                                                      float *grads, float *loss) {
    __shared__ MlpShared S;
    load_weights(S, params);
    load_samples(S, samples, 0, count);
    forward(S);
    const float sq = backward(S, count, grads);
    if (threadIdx.x == 0) *loss = sq / float(count * kMlpOut);
}

// Adam (beta 0.9, 0.999) over minibatches of 64 in the order given by
// `order`; loss[e] receives the mean loss of each epoch.
//
// The minibatches are a serial chain, so one workgroup of 16 wavefronts takes
// each as fast as it can: a wavefront per 16x16 tile, every operand also held
// transposed so that a lane reads its four values along K in one 8-byte LDS
// access, and the parameters with their Adam moments in the registers of the
// lanes that the gradient tiles arrive in, the bf16 weights only ever in LDS.
// What bounds it now is the chain of six stages and barriers and Adam's
// square roots and divisions on one CU.  One wavefront with strided 2-byte
// operands and the parameters in memory took 85 us per minibatch, this 7.1
// (8.3 with the samples' indices looked up in the stage that needs them and
// the bias corrections' powers after the update).
constexpr int kTrainThreads = 1024;
struct alignas(16) TrainShared {
    // weights: [out][in], and transposed where the backward pass reads them along out
    uint16_t w1[kMlpHidden * kNarrow], w2[kMlpHidden * kRow], w2t[kMlpHidden * kRow], w3[16 * kRow],
        w3t[kMlpHidden * kNarrow];
    // activations and deltas: [sample][unit], and [unit][sample]
    uint16_t x[2][64 * kNarrow], xt[2][16 * kRow];
    uint16_t h1[64 * kRow], h1t[64 * kRow], h2[64 * kRow], h2t[64 * kRow];
    uint16_t dy[64 * kNarrow], dyt[16 * kRow], dz2[64 * kRow], dz2t[64 * kRow], dz1t[64 * kRow];
    float b1[kMlpHidden], b2[kMlpHidden], b3[16];
    float t[2][64 * kMlpOut], e[64 * kMlpOut];
    float c1, c2;                              // Adam's bias corrections of the step
};

// Four values of a column (rows q .. q + 3) into [row][column] and, as one
// 8-byte store, into [column][row].
__device__ __forceinline__ void put_tile(uint16_t *rows, uint16_t *cols, int row, int col, const uint16_t *v) {
    bf16x4 four;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if (rows) rows[(row + e) * kRow + col] = v[e];
        four[e] = short(v[e]);
    }
    *reinterpret_cast<bf16x4 *>(cols + col * kRow + row) = four;
}
// Sum of a row of 64 deltas in sample order.
__device__ __forceinline__ float row_sum(const uint16_t *row) {
    float b = 0.0f;
    for (int s = 0; s < 64; s += 4) {
        const bf16x4 v = *reinterpret_cast<const bf16x4 *>(row + s);
#pragma unroll
        for (int e = 0; e < 4; ++e) b += from_bf16(uint16_t(v[e]));
    }
    return b;
}

struct AdamState {
    float p = 0.0f, m = 0.0f, v = 0.0f;
    __device__ __forceinline__ void step(float g, float lr, float c1, float c2) {
        m = 0.9f * m + 0.1f * g;
        v = 0.999f * v + 0.001f * g * g;
        p -= lr * (m / c1) / (sqrtf(v / c2) + 1.0e-8f);
    }
};

__global__ void __launch_bounds__(kTrainThreads) k_mlp_train(const float *samples, uint32_t n, const uint32_t *order,
                                                             uint32_t epochs, float lr, float *params, float *loss) {
    __shared__ TrainShared S;
    const int tid = threadIdx.x, wave = tid >> 6, l = tid & 63, r = l & 15, q = (l >> 4) * 4;
    const int mi = wave >> 2, nj = wave & 3;
    const uint32_t batches = (n + 63) / 64;
    // Parameters: W2 by tile over all wavefronts, W1 on 0-3, W3 on 4-7, the
    // biases on 8, 9 and 10.
    AdamState w2[4], w1[4], w3[2], bias;
    for (int k = tid; k < 64 * kNarrow; k += kTrainThreads) S.dy[k] = 0;
    for (int k = tid; k < 16 * kRow; k += kTrainThreads) S.dyt[k] = S.w3[k] = 0;
    for (int k = tid; k < kMlpHidden * kNarrow; k += kTrainThreads) S.w3t[k] = 0;
    if (tid < 16) S.b3[tid] = 0.0f;
    __syncthreads();
    const int row2 = mi * 16 + q, col = nj * 16 + r;      // W2[row2 + e][col]
    const int row1 = wave * 16 + q;                        // W1[row1 + e][r] on wavefronts 0-3
    const int col3 = (wave & 3) * 16 + r;                  // W3[e][col3] on wavefronts 4-7, q = 0
    auto put_w2 = [&]() {
        uint16_t v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = to_bf16(w2[e].p);
        put_tile(S.w2, S.w2t, row2, col, v);
    };
    auto put_w1 = [&]() {
#pragma unroll
        for (int e = 0; e < 4; ++e) S.w1[(row1 + e) * kNarrow + r] = to_bf16(w1[e].p);
    };
    auto put_w3 = [&]() {
#pragma unroll
        for (int e = 0; e < 2; ++e) S.w3[e * kRow + col3] = S.w3t[col3 * kNarrow + e] = to_bf16(w3[e].p);
    };
    const bool has_w1 = wave < 4, has_w3 = wave >= 4 && wave < 8 && q == 0;
    const bool has_b = wave == 8 || wave == 9 || (wave == 10 && l < kMlpOut);
    const int bias_at = wave == 8 ? kMlpB1 + l : wave == 9 ? kMlpB2 + l : kMlpB3 + l;
    auto put_bias = [&]() {
        if (wave == 8) S.b1[l] = bias.p;
        else if (wave == 9) S.b2[l] = bias.p;
        else S.b3[l] = bias.p;
    };
#pragma unroll
    for (int e = 0; e < 4; ++e) w2[e].p = params[kMlpW2 + (row2 + e) * kMlpHidden + col];
    put_w2();
    if (has_w1) {
#pragma unroll
        for (int e = 0; e < 4; ++e) w1[e].p = params[kMlpW1 + (row1 + e) * kMlpIn + r];
        put_w1();
    }
    if (has_w3) {
#pragma unroll
        for (int e = 0; e < 2; ++e) w3[e].p = params[kMlpW3 + e * kMlpHidden + col3];
        put_w3();
    }
    if (has_b) {
        bias.p = params[bias_at];
        put_bias();
    }
    // A minibatch's samples are fetched one ahead, and their indices two
    // ahead: value k of it is feature k % 18 of its sample k / 18.
    float held[2];
    uint32_t index[2] = {0, 0};                // of the next fetch
    uint32_t ahead_ep = 0, ahead_bi = 0;       // the minibatch they are of
    auto lookup = [&]() {
        const uint32_t first = ahead_bi * 64, count = min(64u, n - first);
        if (ahead_ep < epochs)
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const uint32_t s = (tid + h * kTrainThreads) / kMlpSample;
                index[h] = s < count ? order[size_t(ahead_ep) * n + first + s] : ~0u;
            }
    };
    auto fetch = [&]() {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t f = (tid + h * kTrainThreads) % kMlpSample;
            held[h] = index[h] != ~0u ? samples[size_t(index[h]) * kMlpSample + f] : 0.0f;
        }
        if (++ahead_bi == batches) {
            ahead_bi = 0;
            ++ahead_ep;
        }
        lookup();
    };
    auto store = [&](int buf) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const uint32_t k = tid + h * kTrainThreads, s = k / kMlpSample, f = k % kMlpSample;
            if (s >= 64u) continue;
            if (f < uint32_t(kMlpIn)) S.x[buf][s * kNarrow + f] = S.xt[buf][f * kRow + s] = to_bf16(held[h]);
            else S.t[buf][s * kMlpOut + f - kMlpIn] = held[h];
        }
    };
    lookup();
    fetch();
    store(0);
    __syncthreads();
    const f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    uint32_t t = 0;
    int buf = 0;
    for (uint32_t ep = 0; ep < epochs; ++ep) {
        float total = 0.0f;
        for (uint32_t bi = 0; bi < batches; ++bi, buf ^= 1) {
            const uint32_t count = min(64u, n - bi * 64);
            const bool more = bi + 1 < batches || ep + 1 < epochs;
            if (more) fetch();
            uint16_t v[4];
            {   // hidden 1
                const f32x4 acc = mma_rows<kMlpIn>(S.x[buf] + mi * 16 * kNarrow, kNarrow, S.w1 + nj * 16 * kNarrow,
                                                   kNarrow, zero);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = to_bf16(fmaxf(acc[e] + S.b1[col], 0.0f));
                put_tile(S.h1, S.h1t, row2, col, v);
            }
            __syncthreads();
            {   // hidden 2
                const f32x4 acc = mma_rows<kMlpHidden>(S.h1 + mi * 16 * kRow, kRow, S.w2 + nj * 16 * kRow, kRow, zero);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = to_bf16(fmaxf(acc[e] + S.b2[col], 0.0f));
                put_tile(S.h2, S.h2t, row2, col, v);
            }
            __syncthreads();
            if (wave < 4) {   // outputs, their errors and deltas
                const f32x4 acc = mma_rows<kMlpHidden>(S.h2 + wave * 16 * kRow, kRow, S.w3, kRow, zero);
                const float scale = 2.0f / float(count * kMlpOut);
                if (r < kMlpOut) {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int s = wave * 16 + q + e;
                        const float err = uint32_t(s) < count ? (acc[e] + S.b3[r]) - S.t[buf][s * kMlpOut + r] : 0.0f;
                        const uint16_t d = to_bf16(uint32_t(s) < count ? scale * err : 0.0f);
                        S.e[s * kMlpOut + r] = err;
                        S.dy[s * kNarrow + r] = S.dyt[r * kRow + s] = d;
                    }
                }
            }
            ++t;
            if (tid == kTrainThreads - 1) {   // on a wavefront without outputs
                S.c1 = 1.0f - powf(0.9f, float(t));
                S.c2 = 1.0f - powf(0.999f, float(t));
            }
            __syncthreads();
            f32x4 g3 = zero;
            float gb = 0.0f;
            {   // dZ2 = (dY W3) .* [H2 > 0]; dW3 = dY^T H2
                const f32x4 acc = mma_rows<16>(S.dy + mi * 16 * kNarrow, kNarrow, S.w3t + nj * 16 * kNarrow, kNarrow, zero);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[e] = from_bf16(S.h2[(row2 + e) * kRow + col]) > 0.0f ? to_bf16(acc[e]) : 0;
                put_tile(S.dz2, S.dz2t, row2, col, v);
                if (wave >= 4 && wave < 8)
                    g3 = mma_rows<64>(S.dyt, kRow, S.h2t + (wave & 3) * 16 * kRow, kRow, zero);
                if (wave == 10 && l < kMlpOut) gb = row_sum(S.dyt + l * kRow);
                if (wave == 15) {   // the summed squared error
                    float sq = 0.0f;
#pragma unroll
                    for (int o = 0; o < kMlpOut; ++o) {
                        const float err = S.e[l * kMlpOut + o];
                        if (uint32_t(l) < count) sq += err * err;
                    }
#pragma unroll
                    for (int d = 32; d >= 1; d >>= 1) sq += __shfl_xor(sq, d, 64);
                    total += sq;
                }
            }
            __syncthreads();
            f32x4 g2;
            {   // dW2 = dZ2^T H1; dZ1 = (dZ2 W2) .* [H1 > 0]
                const f32x4 acc = mma_rows<64>(S.dz2 + mi * 16 * kRow, kRow, S.w2t + nj * 16 * kRow, kRow, zero);
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    v[e] = from_bf16(S.h1[(row2 + e) * kRow + col]) > 0.0f ? to_bf16(acc[e]) : 0;
                put_tile(nullptr, S.dz1t, row2, col, v);
                g2 = mma_rows<64>(S.dz2t + mi * 16 * kRow, kRow, S.h1t + nj * 16 * kRow, kRow, zero);
                if (wave == 9) gb = row_sum(S.dz2t + l * kRow);
                if (more) store(buf ^ 1);
            }
            const float c1 = S.c1, c2 = S.c2;
            __syncthreads();
            // dW1 = dZ1^T X, and the update.  W2 is read by nobody until the
            // next barrier.
            if (has_w1) {
                const f32x4 g1 = mma_rows<64>(S.dz1t + wave * 16 * kRow, kRow, S.xt[buf], kRow, zero);
#pragma unroll
                for (int e = 0; e < 4; ++e) w1[e].step(g1[e], lr, c1, c2);
                put_w1();
            }
            if (has_w3) {
#pragma unroll
                for (int e = 0; e < 2; ++e) w3[e].step(g3[e], lr, c1, c2);
                put_w3();
            }
            if (has_b) {
                if (wave == 8) gb = row_sum(S.dz1t + l * kRow);
                bias.step(gb, lr, c1, c2);
                put_bias();
            }
#pragma unroll
            for (int e = 0; e < 4; ++e) w2[e].step(g2[e], lr, c1, c2);
            put_w2();
            __syncthreads();
        }
        if (wave == 15 && l == 0) loss[ep] = total / float(n * kMlpOut);
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) params[kMlpW2 + (row2 + e) * kMlpHidden + col] = w2[e].p;
    if (has_w1) {
#pragma unroll
        for (int e = 0; e < 4; ++e) params[kMlpW1 + (row1 + e) * kMlpIn + r] = w1[e].p;
    }
    if (has_w3) {
#pragma unroll
        for (int e = 0; e < 2; ++e) params[kMlpW3 + e * kMlpHidden + col3] = w3[e].p;
    }
    if (has_b) params[bias_at] = bias.p;
}

// Inference for listed cold points: y0 = log10(1 + lambda / (m_eff |g|)),
// y1 = log10(k / k0); lambda >= 0, k0 <= k <= the penalty cap.
__global__ void __launch_bounds__(64) k_mlp_infer(const uint32_t *count_ptr, const uint32_t *list, const float *feat,
                                                  const float *scale, const float *params, float4 *c_lam,
                                                  float4 *c_pen, uint32_t cap, uint32_t policy) {
    __shared__ MlpShared S;
    load_weights(S, params);
    const uint32_t total = min(*count_ptr, cap);
    const int l = threadIdx.x;
    for (uint32_t first = blockIdx.x * 64; first < total; first += gridDim.x * 64) {
        const uint32_t count = min(64u, total - first);
        const bool live = uint32_t(l) < count;
        for (int f = 0; f < kMlpIn; ++f) S.x[l * kNarrow + f] = live ? to_bf16(feat[size_t(first + l) * kMlpIn + f]) : 0;
        __syncthreads();
        forward(S);
        if (live) {
            const uint32_t c = list[first + l];
            const float lam_scale = scale[2 * size_t(first + l)], k0 = scale[2 * size_t(first + l) + 1];
            // predictions stay within the range of the training targets
            const float y0 = fminf(fmaxf(S.y[l * kMlpOut], 0.0f), params[kMlpBound]);
            const float y1 = fminf(fmaxf(S.y[l * kMlpOut + 1], 0.0f), params[kMlpBound + 1]);
            const float lam = (exp10f(y0) - 1.0f) * lam_scale;
            const float k = fminf(k0 * exp10f(y1), kMaxPenalty);
            // The penalty always; lambda only where the contact starts in
            // violation (initial normal error > 0, feature 5), i.e. where it
            // is active from the first iteration anyway.
            if (policy & kWarmPenalty) {
                float4 b = c_pen[c];
                b.x = fmaxf(k, k0);
                c_pen[c] = b;
            }
            if ((policy & kWarmLambda) && feat[size_t(first + l) * kMlpIn + 5] > 0.0f) {
                float4 a = c_lam[c];
                a.x = lam;
                c_lam[c] = a;
            }
        }
        __syncthreads();
    }
}

PmhResult mlp_infer(hipStream_t s, const uint32_t *count, const uint32_t *list, const float *feat,
                    const float *scale, const float *params, float4 *c_lam, float4 *c_pen, uint32_t cap,
                    uint32_t policy) {
    const uint32_t blocks = std::max<uint32_t>(1, std::min<uint32_t>((cap + 63) / 64, 1024));
    k_mlp_infer<<<blocks, 64, 0, s>>>(count, list, feat, scale, params, c_lam, c_pen, cap, policy);
    PMH_CHECK(hipGetLastError());
    return PMH_SUCCESS;
}

// Forward pass of `n` feature rows (16 floats each) into y (2 floats each).
__global__ void __launch_bounds__(64) k_mlp_forward(const float *x, uint32_t n, const float *params, float *y) {
    __shared__ MlpShared S;
    load_weights(S, params);
    const int l = threadIdx.x;
    for (uint32_t first = blockIdx.x * 64; first < n; first += gridDim.x * 64) {
        const uint32_t count = min(64u, n - first);
        const bool live = uint32_t(l) < count;
        for (int f = 0; f < kMlpIn; ++f) S.x[l * kNarrow + f] = live ? to_bf16(x[size_t(first + l) * kMlpIn + f]) : 0;
        __syncthreads();
        forward(S);
        if (live)
            for (int o = 0; o < kMlpOut; ++o) y[size_t(first + l) * kMlpOut + o] = S.y[l * kMlpOut + o];
        __syncthreads();
    }
}

}  // namespace pmh

using namespace pmh;

extern "C" {

void pmhWarmstartInit(uint32_t seed, float *params) {
    // He-uniform weights, zero biases, from a 32-bit LCG.
    uint32_t st = seed * 2654435761u + 12345u;
    auto uni = [&]() { st = st * 1664525u + 1013904223u; return (st >> 8) * (1.0f / 16777216.0f); };
    for (int k = 0; k < kMlpParams; ++k) params[k] = 0.0f;
    const float a1 = std::sqrt(6.0f / kMlpIn), a2 = std::sqrt(6.0f / kMlpHidden), a3 = std::sqrt(3.0f / kMlpHidden);
    for (int k = 0; k < kMlpHidden * kMlpIn; ++k) params[kMlpW1 + k] = (2.0f * uni() - 1.0f) * a1;
    for (int k = 0; k < kMlpHidden * kMlpHidden; ++k) params[kMlpW2 + k] = (2.0f * uni() - 1.0f) * a2;
    for (int k = 0; k < kMlpOut * kMlpHidden; ++k) params[kMlpW3 + k] = (2.0f * uni() - 1.0f) * a3;
    params[kMlpBound] = params[kMlpBound + 1] = 0.0f;
}

PmhResult pmhWarmstartForward(const float *params, const float *features, uint32_t n, float *outputs) {
    if (!params || !features || !outputs || n == 0) return PMH_ERROR_INVALID_ARGUMENT;
    DBuf<float> dx, dp, dy;
    PmhResult r;
    if ((r = dx.reserve(size_t(n) * kMlpIn)) || (r = dp.reserve(kMlpParams)) || (r = dy.reserve(size_t(n) * kMlpOut)))
        return r;
    PMH_CHECK(hipMemcpy(dx.p, features, sizeof(float) * n * kMlpIn, hipMemcpyHostToDevice));
    PMH_CHECK(hipMemcpy(dp.p, params, sizeof(float) * kMlpParams, hipMemcpyHostToDevice));
    k_mlp_forward<<<std::max<uint32_t>(1, std::min<uint32_t>((n + 63) / 64, 1024)), 64>>>(dx.p, n, dp.p, dy.p);
    PMH_CHECK(hipGetLastError());
    PMH_CHECK(hipMemcpy(outputs, dy.p, sizeof(float) * n * kMlpOut, hipMemcpyDeviceToHost));
    dx.release(); dp.release(); dy.release();
    return PMH_SUCCESS;
}

PmhResult pmhWarmstartGradients(const float *samples, uint32_t count, const float *params, float *grads,
                                float *loss) {
    if (!samples || !params || !grads || !loss || count == 0 || count > 64) return PMH_ERROR_INVALID_ARGUMENT;
    DBuf<float> ds, dp, dg, dl;
    PmhResult r;
    if ((r = ds.reserve(size_t(count) * kMlpSample)) || (r = dp.reserve(kMlpParams)) || (r = dg.reserve(kMlpParams)) ||
        (r = dl.reserve(1)))
        return r;
    PMH_CHECK(hipMemcpy(ds.p, samples, sizeof(float) * count * kMlpSample, hipMemcpyHostToDevice));
    PMH_CHECK(hipMemcpy(dp.p, params, sizeof(float) * kMlpParams, hipMemcpyHostToDevice));
    PMH_CHECK(hipMemset(dg.p, 0, sizeof(float) * kMlpParams));
    k_mlp_gradients<<<1, 64>>>(ds.p, count, dp.p, dg.p, dl.p);
    PMH_CHECK(hipGetLastError());
    PMH_CHECK(hipMemcpy(grads, dg.p, sizeof(float) * kMlpParams, hipMemcpyDeviceToHost));
    PMH_CHECK(hipMemcpy(loss, dl.p, sizeof(float), hipMemcpyDeviceToHost));
    ds.release(); dp.release(); dg.release(); dl.release();
    return PMH_SUCCESS;
}

PmhResult pmhWarmstartTrain(const float *samples, uint32_t n, uint32_t epochs, float learning_rate, uint32_t seed,
                            float *params, float *epoch_loss) {
    if (!samples || !params || !epoch_loss || n == 0 || epochs == 0 || !(learning_rate > 0.0f))
        return PMH_ERROR_INVALID_ARGUMENT;
    // Epoch permutations from the seed (Fisher-Yates with an LCG).
    std::vector<uint32_t> order(size_t(epochs) * n);
    uint32_t st = seed * 747796405u + 2891336453u;
    for (uint32_t ep = 0; ep < epochs; ++ep) {
        uint32_t *o = order.data() + size_t(ep) * n;
        for (uint32_t k = 0; k < n; ++k) o[k] = k;
        for (uint32_t k = n - 1; k > 0; --k) {
            st = st * 1664525u + 1013904223u;
            const uint32_t j = uint32_t((uint64_t(st) * (k + 1)) >> 32);
            const uint32_t t = o[k];
            o[k] = o[j];
            o[j] = t;
        }
    }
    DBuf<float> ds, dp, dl;
    DBuf<uint32_t> dorder;
    PmhResult r;
    if ((r = ds.reserve(size_t(n) * kMlpSample)) || (r = dp.reserve(kMlpParams)) || (r = dl.reserve(epochs)) ||
        (r = dorder.reserve(order.size())))
        return r;
    PMH_CHECK(hipMemcpy(ds.p, samples, sizeof(float) * size_t(n) * kMlpSample, hipMemcpyHostToDevice));
    PMH_CHECK(hipMemcpy(dp.p, params, sizeof(float) * kMlpParams, hipMemcpyHostToDevice));
    PMH_CHECK(hipMemcpy(dorder.p, order.data(), sizeof(uint32_t) * order.size(), hipMemcpyHostToDevice));
    k_mlp_train<<<1, kTrainThreads>>>(ds.p, n, dorder.p, epochs, learning_rate, dp.p, dl.p);
    PMH_CHECK(hipGetLastError());
    PMH_CHECK(hipMemcpy(params, dp.p, sizeof(float) * kMlpParams, hipMemcpyDeviceToHost));
    PMH_CHECK(hipMemcpy(epoch_loss, dl.p, sizeof(float) * epochs, hipMemcpyDeviceToHost));
    for (int o = 0; o < kMlpOut; ++o) {
        float hi = 0.0f;
        for (uint32_t k = 0; k < n; ++k) hi = std::max(hi, samples[size_t(k) * kMlpSample + kMlpIn + o]);
        params[kMlpBound + o] = hi;
    }
    ds.release(); dp.release(); dl.release(); dorder.release();
    return PMH_SUCCESS;
}

}  // extern "C"
