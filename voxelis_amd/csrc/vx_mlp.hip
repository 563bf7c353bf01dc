// vx_mlp.hip -- the node-growth predictor: an FP32 MLP 16 -> 64 -> 64 -> 1 (ReLU),
// forward, backward and Adam kernels.
//
// Parameters, packed float32 (kMlpParams):
//   W1 [64][16] | b1 [64] | W2 [64][64] | b2 [64] | W3 [64] | b3
// Loss: mean squared error over the batch, L = (1/n) sum_s (y_s - t_s)^2.
//
// Forward, backward and the gradients are matrix products over the batch (K = 16, 64 or
// the samples), so they run on the f32 matrix unit (v_mfma_f32_16x16x4_f32: f32 inputs and
// accumulation) in one pass over the samples: nothing per sample goes to memory but y.
// Partial gradients per block are added in block order, so results do not depend on
// scheduling.
#include <hip/hip_runtime.h>

#include <cstdint>

namespace vx {

constexpr int kIn = 16, kHid = 64;
constexpr int kOffW1 = 0, kOffB1 = kOffW1 + kHid * kIn, kOffW2 = kOffB1 + kHid,
              kOffB2 = kOffW2 + kHid * kHid, kOffW3 = kOffB2 + kHid, kOffB3 = kOffW3 + kHid;
constexpr int kMlpParams = kOffB3 + 1;  // 5313
constexpr int kMlpTile = 64;            // samples of one tile: 16 per wavefront
constexpr int kMlpPart = 5376;          // floats of one block's partial gradients (loss at kMlpParams)

typedef float MlpAcc __attribute__((ext_vector_type(4)));

// A 16 x 16 product over 4 k: lane l gives A[l % 16][l / 16] and B[l / 16][l % 16] and holds
// rows 4 * (l / 16) + r, column l % 16 of the result.
__device__ inline MlpAcc mlp_mma(float a, float b, MlpAcc c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

struct MlpLds {  // odd row lengths: a column walk meets every bank
    float x[kMlpTile][kIn + 1];
    float w1[kHid][kIn + 1];
    float w2[kHid][kHid + 1];
    float h1[kMlpTile][kHid + 1];
    float d1[kMlpTile][kHid + 1];
    float d2[kMlpTile][kHid + 1];
    float sum[4][4][kHid];  // per wavefront: b1, b2, W3; [3]: b3 and the loss
};

// Blocks take tiles of 64 samples: a1 = x W1^T + b1, a2 = relu(a1) W2^T + b2,
// y = relu(a2) . W3 + b3.  BACK: also dL/da2, dL/da1 and the block's share of every
// parameter's gradient, accumulated in registers over its tiles and written to
// part[block][kMlpPart] (or, by a single block, to grad and loss).
//
// The tile is 64 samples: a row block of the products for each wavefront, 224 products of it
// per tile (about 7.2 k cycles of its SIMD's matrix unit), and 128 blocks for a batch of 8192.
// The form it replaces wrote 1 KB per sample to memory and reduced it with one lane per
// parameter, a chain of n dependent loads: a training step of 8192 rows (gradient and Adam)
// took 2067 us and takes 24 us now, which is the host's time to call it.  The sums are shorter
// so: the gradient's error against 64 bits (2-norm, mean of 12 seeds) is 6e-8 for 64 rows,
// 4e-8 for 1000 and 7e-7 for 8192, where the one chain had 1.1e-7, 4e-7 and 1.7e-6.
template <bool BACK>
__global__ __launch_bounds__(256) void k_mlp(const float* P, const float* x, uint32_t n, float* y,
                                             const float* target, float* part, float* grad, float* loss) {
    __shared__ MlpLds S;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, c = lane & 15, q = lane >> 4;
    for (int e = tid; e < kHid * kIn; e += 256) S.w1[e / kIn][e % kIn] = P[kOffW1 + e];
    for (int e = tid; e < kHid * kHid; e += 256) S.w2[e / kHid][e % kHid] = P[kOffW2 + e];
    float b1[4], b2[4], w3[4];
#pragma unroll
    for (int t = 0; t < 4; t++) {
        b1[t] = P[kOffB1 + 16 * t + c];
        b2[t] = P[kOffB2 + 16 * t + c];
        w3[t] = P[kOffW3 + 16 * t + c];
    }
    const float b3 = P[kOffB3];
    MlpAcc g1 = {0.f, 0.f, 0.f, 0.f}, g2[4];
    float gb1[4], gb2[4], g3[4], gb3 = 0.f, gl = 0.f;
#pragma unroll
    for (int t = 0; t < 4; t++) {
        g2[t] = MlpAcc{0.f, 0.f, 0.f, 0.f};
        gb1[t] = gb2[t] = g3[t] = 0.f;
    }
    for (uint64_t s0 = (uint64_t)blockIdx.x * kMlpTile; s0 < n; s0 += (uint64_t)gridDim.x * kMlpTile) {
        __syncthreads();  // the previous tile's rows were read
        for (int e = tid; e < kMlpTile * kIn; e += 256) {
            const uint64_t s = s0 + e / kIn;
            S.x[e / kIn][e % kIn] = s < n ? x[s * kIn + e % kIn] : 0.f;
        }
        __syncthreads();
        const int r0 = 16 * w;  // this wavefront's samples of the tile
        bool ok[4];             // row 4q + r of them
#pragma unroll
        for (int r = 0; r < 4; r++) ok[r] = s0 + r0 + 4 * q + r < n;
#pragma unroll
        for (int t = 0; t < 4; t++) {
            MlpAcc a = {b1[t], b1[t], b1[t], b1[t]};
#pragma unroll
            for (int k = 0; k < kIn; k += 4) a = mlp_mma(S.x[r0 + c][k + q], S.w1[16 * t + c][k + q], a);
#pragma unroll
            for (int r = 0; r < 4; r++) S.h1[r0 + 4 * q + r][16 * t + c] = ok[r] && a[r] > 0.f ? a[r] : 0.f;
        }
        __syncthreads();
        MlpAcc a2[4];
        MlpAcc out = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 4; t++) {
            a2[t] = MlpAcc{b2[t], b2[t], b2[t], b2[t]};
#pragma unroll
            for (int k = 0; k < kHid; k += 4) a2[t] = mlp_mma(S.h1[r0 + c][k + q], S.w2[16 * t + c][k + q], a2[t]);
#pragma unroll
            for (int r = 0; r < 4; r++) {
                a2[t][r] = a2[t][r] > 0.f ? a2[t][r] : 0.f;
                out[r] = fmaf(w3[t], a2[t][r], out[r]);
            }
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) out[r] += __shfl_xor(out[r], o);
            out[r] += b3;
            if (ok[r] && c == 0 && y) y[s0 + r0 + 4 * q + r] = out[r];
        }
        if constexpr (BACK) {
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const float e = ok[r] ? out[r] - target[s0 + r0 + 4 * q + r] : 0.f;
                const float dy = 2.f * e / (float)n;
                if (c == 0) {
                    gb3 += dy;
                    gl = fmaf(e, e, gl);
                }
#pragma unroll
                for (int t = 0; t < 4; t++) {
                    const float d = ok[r] && a2[t][r] > 0.f ? dy * w3[t] : 0.f;
                    S.d2[r0 + 4 * q + r][16 * t + c] = d;
                    gb2[t] += d;
                    if (ok[r]) g3[t] = fmaf(dy, a2[t][r], g3[t]);
                }
            }
            __syncthreads();
#pragma unroll
            for (int t = 0; t < 4; t++) {
                MlpAcc a = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int k = 0; k < kHid; k += 4) a = mlp_mma(S.d2[r0 + c][k + q], S.w2[k + q][16 * t + c], a);
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float d = S.h1[r0 + 4 * q + r][16 * t + c] > 0.f ? a[r] : 0.f;
                    S.d1[r0 + 4 * q + r][16 * t + c] = d;
                    gb1[t] += d;
                }
            }
            __syncthreads();
            // the tile's products over its samples: rows j = 16 w + ..
#pragma unroll
            for (int k = 0; k < kMlpTile; k += 4) {
                const float dj = S.d2[k + q][r0 + c];
#pragma unroll
                for (int t = 0; t < 4; t++) g2[t] = mlp_mma(dj, S.h1[k + q][16 * t + c], g2[t]);
                g1 = mlp_mma(S.d1[k + q][r0 + c], S.x[k + q][c], g1);
            }
        }
    }
    if constexpr (BACK) {
        const bool one = gridDim.x == 1;
        float* G = one ? grad : part + (size_t)blockIdx.x * kMlpPart;
#pragma unroll
        for (int t = 0; t < 4; t++) {
#pragma unroll
            for (int o = 16; o < 64; o <<= 1) {
                gb1[t] += __shfl_xor(gb1[t], o);
                gb2[t] += __shfl_xor(gb2[t], o);
                g3[t] += __shfl_xor(g3[t], o);
            }
            if (q == 0) {
                S.sum[w][0][16 * t + c] = gb1[t];
                S.sum[w][1][16 * t + c] = gb2[t];
                S.sum[w][2][16 * t + c] = g3[t];
            }
        }
#pragma unroll
        for (int o = 16; o < 64; o <<= 1) {
            gb3 += __shfl_xor(gb3, o);
            gl += __shfl_xor(gl, o);
        }
        if (lane == 0) {
            S.sum[w][3][0] = gb3;
            S.sum[w][3][1] = gl;
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const int j = 16 * w + 4 * q + r;
#pragma unroll
            for (int t = 0; t < 4; t++) G[kOffW2 + j * kHid + 16 * t + c] = g2[t][r];
            G[kOffW1 + j * kIn + c] = g1[r];
        }
        __syncthreads();
        if (tid < 3 * kHid) {
            const int v = tid / kHid, j = tid % kHid;
            const float t = (S.sum[0][v][j] + S.sum[1][v][j]) + (S.sum[2][v][j] + S.sum[3][v][j]);
            G[(v == 0 ? kOffB1 : v == 1 ? kOffB2 : kOffW3) + j] = t;
        } else if (tid < 3 * kHid + 2) {
            const int v = tid - 3 * kHid;
            const float t = (S.sum[0][3][v] + S.sum[1][3][v]) + (S.sum[2][3][v] + S.sum[3][3][v]);
            if (v == 0) G[kOffB3] = t;
            else if (!one) G[kMlpParams] = t;
            else if (loss) *loss = t / (float)n;
        }
    }
}

// The blocks' partial gradients added in a fixed order: 64 parameters per block, four
// lanes each (block b of the first pass goes to lane b % 4).
__global__ __launch_bounds__(256) void k_mlp_reduce(const float* part, uint32_t blocks, uint32_t n, float* grad,
                                                    float* loss) {
    __shared__ float s[4][64];
    const uint32_t i = threadIdx.x & 63u, g = threadIdx.x >> 6, p = blockIdx.x * 64 + i;
    float v = 0.f;
#pragma unroll 8
    for (uint32_t b = g; b < blocks; b += 4) v += part[(size_t)b * kMlpPart + p];
    s[g][i] = v;
    __syncthreads();
    if (g == 0 && p <= (uint32_t)kMlpParams) {
        v = (s[0][i] + s[1][i]) + (s[2][i] + s[3][i]);
        if (p < (uint32_t)kMlpParams) grad[p] = v;
        else if (loss) *loss = v / (float)n;
    }
}

// Adam (Kingma & Ba, 2015) with bias correction; step counts from 1.
__global__ void k_mlp_adam(float* P, const float* grad, float* m, float* v, uint32_t step, float lr, float b1,
                           float b2, float eps) {
    uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= (uint32_t)kMlpParams) return;
    float g = grad[p];
    float mm = b1 * m[p] + (1.f - b1) * g;
    float vv = b2 * v[p] + (1.f - b2) * g * g;
    m[p] = mm;
    v[p] = vv;
    float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
    P[p] -= lr * (mm / c1) / (sqrtf(vv / c2) + eps);
}

}  // namespace vx
