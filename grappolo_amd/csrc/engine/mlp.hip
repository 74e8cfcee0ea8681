// mlp.hip -- training and inference kernels of the active-set MLP on the
// gfx950 matrix cores (see mlp.hpp for the network and the loss, and
// mlp_device.hpp for the operand layout).
//
// Backward pass of one tile of 16 samples (dz = c_s (sigmoid(z) - y) / B):
//   dZ2 = relu'(z2) * w3 dz                      FP32, then BF16 for the matrix cores
//   dH1 = W2 dZ2                                 MFMA, A = W2 tiles, B = dZ2 (as produced)
//   dZ1 = relu'(z1) * dH1                        FP32, then BF16
//   gW2 = H1 dZ2^T,  gW1 = X dZ1^T               MFMA with the samples as the K dimension:
//                                                 H1, dZ2, dZ1 are transposed through LDS
//   gb1 = sum dZ1, gb2 = sum dZ2, gw3 = sum dz h2, gb3 = sum dz   FP32 (unrounded)
// The wavefronts of a workgroup add their gradients in LDS, every workgroup
// writes its sum to its own row, and the rows are summed in a fixed order, so a
// gradient is deterministic.
#include <math.h>

#include "mlp_device.hpp"

namespace glv {

namespace {

constexpr int kMlpBlock = 256;  // 4 wavefronts
constexpr int kWpb = kMlpBlock / kWave;

__device__ inline u64 mix64(u64 z) {
    z += 0x9E3779B97F4A7C15ULL;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

// B operand of layer 1 for the tile starting at sample `base` (index map idx()).
__device__ inline mlp_s4 load_x(const uint16_t *feats, i64 sample, bool ok) {
    const int lane = threadIdx.x % kWave, g = lane >> 4;
    mlp_s4 x = {0, 0, 0, 0};
    if (ok && g < 2) {
        const uint2 raw = *reinterpret_cast<const uint2 *>(feats + sample * kMlpIn + 4 * g);
        x[0] = (short)(raw.x & 0xffffu);
        x[1] = (short)(raw.x >> 16);
        x[2] = (short)(raw.y & 0xffffu);
        x[3] = (short)(raw.y >> 16);
    }
    return x;
}

// Transposes of D-layout 16x16 BF16 tiles through a wavefront's private LDS:
// all tiles of a turn are stored, then read back, so that the turn waits for
// LDS once.  Rows of 20 (16 used) keep the stores of the four lane groups in
// different banks.
constexpr int kTileRow = 20;
constexpr int kTileWords = 16 * kTileRow;
__device__ inline void store_tile(mlp_s4 x, uint16_t *buf) {
    const int lane = threadIdx.x % kWave, g = lane >> 4, r = lane & 15;
#pragma unroll
    for (int i = 0; i < 4; i++) buf[(4 * g + i) * kTileRow + r] = (uint16_t)x[i];
}
// lane returns M[r][4g .. 4g+3] of the matrix M whose D layout was stored
__device__ inline mlp_s4 load_tile(const uint16_t *buf) {
    const int lane = threadIdx.x % kWave, g = lane >> 4, r = lane & 15;
    const uint2 raw = *reinterpret_cast<const uint2 *>(buf + r * kTileRow + 4 * g);
    mlp_s4 y;
    y[0] = (short)(raw.x & 0xffffu);
    y[1] = (short)(raw.x >> 16);
    y[2] = (short)(raw.y & 0xffffu);
    y[3] = (short)(raw.y >> 16);
    return y;
}

// The gradient kernel's weights, in LDS but for layer 1's: a lane's bytes of an
// operand together.  With them in registers (394) a SIMD holds one wavefront.
struct MlpLds {
    mlp_s4 w2t[16][kWave], w2[16][kWave];  // layer 2 [4u + t]; dH1 = W2 dZ2 [4t + u]: W2[16t + r][16u + 4g + i]
    mlp_f4 b1[16], b2[16], w3[16];         // units 4x .. 4x + 3; w3 BF16-rounded
};
struct MlpLdsView {
    const MlpLds &S;
    mlp_s4 w1[4];
    float b3;
    int lane, g;
    __device__ mlp_s4 in(int t) const { return w1[t]; }
    __device__ mlp_s4 mid(int u, int t) const { return S.w2t[4 * u + t][lane]; }
    __device__ mlp_s4 back(int t, int u) const { return S.w2[4 * t + u][lane]; }
    __device__ mlp_f4 bias1(int t) const { return S.b1[4 * t + g]; }
    __device__ mlp_f4 bias2(int u) const { return S.b2[4 * u + g]; }
    __device__ mlp_f4 out(int u) const { return S.w3[4 * u + g]; }
};

// A lane's share of the gradient (per-unit sums already over the 16 samples'
// lanes), and its place in the parameter vector
struct MlpSums {
    mlp_f4 gW2[4][4], gW1[4], gb1[4], gb2[4], gw3[4];
    float gb3, loss;
    // x = f(place, x) for each value x that the lane holds
    template <class F>
    __device__ void each(F f) {
        const int lane = threadIdx.x % kWave, g = lane >> 4, r = lane & 15;
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int u = 0; u < 4; u++)
#pragma unroll
                for (int i = 0; i < 4; i++) gW2[t][u][i] = f(kMlpW2 + (16 * t + 4 * g + i) * kMlpHidden + 16 * u + r, gW2[t][u][i]);
        if (g < 2) {
#pragma unroll
            for (int u = 0; u < 4; u++)
#pragma unroll
                for (int i = 0; i < 4; i++) gW1[u][i] = f(kMlpW1 + (4 * g + i) * kMlpHidden + 16 * u + r, gW1[u][i]);
        }
        if (r == 0) {
#pragma unroll
            for (int t = 0; t < 4; t++)
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    gb1[t][i] = f(kMlpB1 + 16 * t + 4 * g + i, gb1[t][i]);
                    gb2[t][i] = f(kMlpB2 + 16 * t + 4 * g + i, gb2[t][i]);
                    gw3[t][i] = f(kMlpW3 + 16 * t + 4 * g + i, gw3[t][i]);
                }
        }
        if (lane == 0) {
            gb3 = f(kMlpB3, gb3);
            loss = f(kMlpParams, loss);
        }
    }
};

__global__ __launch_bounds__(kMlpBlock) void k_mlp_forward(const float *P, const uint16_t *feats, i64 n,
                                                           float *logits) {
    MlpW W;
    mlp_load(P, W);
    const int lane = threadIdx.x % kWave, r = lane & 15;
    const i64 wave = (i64)blockIdx.x * kWpb + threadIdx.x / kWave;
    const i64 nwaves = (i64)gridDim.x * kWpb;
    for (i64 base = wave * 16; base < n; base += nwaves * 16) {
        const i64 smp = base + r;
        const bool ok = smp < n;
        MlpAct A;
        mlp_forward_tile(W, load_x(feats, smp, ok), A);
        if (ok && lane < 16) logits[smp] = A.z;
    }
}

// Bound by the chain of one tile (four dependent MFMA layers, the logistic, 13
// transposes) at the two wavefronts per SIMD that its registers allow:
// 262,144 samples take 50 us on 512 workgroups.  155 us with the weights in
// registers (one wavefront a SIMD), on 128 workgroups, with a wait for
// LDS per transpose and the features loaded a second time for gW1.
__global__ __launch_bounds__(kMlpBlock, 2) void k_mlp_grad(const float *P, MlpBatch B, float *gpart) {
    constexpr int kTiles = 13;  // per wavefront: x, dZ2, dZ1, H1
    constexpr size_t kTileBytes = sizeof(uint16_t) * kWpb * kTiles * kTileWords;
    constexpr size_t kSumBytes = sizeof(float) * 2 * kMlpStride;  // after the tiles: two wavefronts' sums
    __shared__ MlpLds s_w;
    __shared__ alignas(16) unsigned char s_mem[kTileBytes > kSumBytes ? kTileBytes : kSumBytes];
    static_assert(kWpb == 4, "the sums of four wavefronts are added in two steps");
    const int wv = threadIdx.x / kWave;
    uint16_t *buf = reinterpret_cast<uint16_t *>(s_mem) + wv * kTiles * kTileWords;
    const int lane = threadIdx.x % kWave, g = lane >> 4, r = lane & 15;
    const i64 wave = (i64)blockIdx.x * kWpb + wv;
    const i64 nwaves = (i64)gridDim.x * kWpb;
    // wavefront t fills row t of the tiles
#pragma unroll
    for (int u = 0; u < 4; u++) {
        mlp_s4 a, b;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            a[i] = (short)bf16_bits(P[kMlpW2 + (16 * wv + 4 * g + i) * kMlpHidden + 16 * u + r]);
            b[i] = (short)bf16_bits(P[kMlpW2 + (16 * wv + r) * kMlpHidden + 16 * u + 4 * g + i]);
        }
        s_w.w2t[4 * u + wv][lane] = a;
        s_w.w2[4 * wv + u][lane] = b;
    }
    if (threadIdx.x < 16)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int h = 4 * threadIdx.x + i;
            s_w.b1[threadIdx.x][i] = P[kMlpB1 + h];
            s_w.b2[threadIdx.x][i] = P[kMlpB2 + h];
            s_w.w3[threadIdx.x][i] = bf16_round(P[kMlpW3 + h]);
        }
    MlpLdsView W{s_w, {}, P[kMlpB3], lane, g};
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int i = 0; i < 4; i++)
            W.w1[t][i] = g < 2 ? (short)bf16_bits(P[kMlpW1 + (4 * g + i) * kMlpHidden + 16 * t + r]) : (short)0;
    __syncthreads();
    MlpSums S;
    const mlp_f4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int t = 0; t < 4; t++) {
        S.gW1[t] = zero;
        S.gb1[t] = zero;
        S.gb2[t] = zero;
        S.gw3[t] = zero;
#pragma unroll
        for (int u = 0; u < 4; u++) S.gW2[t][u] = zero;
    }
    S.gb3 = 0.f;
    S.loss = 0.f;
    const float inv_b = 1.0f / (float)B.batch;
    for (i64 base = wave * 16; base < B.batch; base += nwaves * 16) {
        const i64 j = base + r;  // position of lane's sample in the batch
        const bool ok = j < B.batch;
        i64 smp = j;
        if (B.random) smp = (i64)(mix64(B.seed + (u64)(B.step * B.batch + j)) % (u64)B.n);
        MlpAct A;
        const mlp_s4 x = load_x(B.feats, smp, ok);
        mlp_forward_tile(W, x, A);
        float dz = 0.f;
        if (ok) {
            const float y = B.labels[smp] ? 1.0f : 0.0f;
            const float c = (y > 0.5f ? B.pos_weight : 1.0f) * inv_b;
            const float z = A.z;
            const float p = 1.0f / (1.0f + expf(-z));
            dz = c * (p - y);
            // softplus(z) - y z, stable for either sign of z
            const float sp = fmaxf(z, 0.0f) + log1pf(expf(-fabsf(z)));
            if (g == 0) {
                S.loss += c * (sp - y * z);
                S.gb3 += dz;
            }
        }
        // layer 3 and layer 2 deltas
        mlp_s4 dz2b[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            const mlp_f4 w3 = W.out(u);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float zz = A.z2[u][i];
                const float d = zz > 0.f ? w3[i] * dz : 0.f;
                S.gw3[u][i] += dz * fmaxf(zz, 0.f);
                S.gb2[u][i] += d;
                dz2b[u][i] = (short)bf16_of(d);
            }
        }
        // dH1 = W2 dZ2, then layer-1 deltas
        mlp_s4 dz1b[4];
#pragma unroll
        for (int t = 0; t < 4; t++) {
            mlp_f4 d = zero;
#pragma unroll
            for (int u = 0; u < 4; u++) d = mfma16(W.back(t, u), dz2b[u], d);
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float v = A.z1[t][i] > 0.f ? d[i] : 0.f;
                S.gb1[t][i] += v;
                dz1b[t][i] = (short)bf16_of(v);
            }
        }
        // weight gradients: samples along K; X^T is x transposed
        store_tile(x, buf);
#pragma unroll
        for (int t = 0; t < 4; t++) {
            store_tile(dz2b[t], buf + (1 + t) * kTileWords);
            store_tile(dz1b[t], buf + (5 + t) * kTileWords);
            store_tile(A.h1[t], buf + (9 + t) * kTileWords);
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        const mlp_s4 xa = load_tile(buf);
        mlp_s4 dz2T[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            dz2T[u] = load_tile(buf + (1 + u) * kTileWords);
            S.gW1[u] = mfma16(xa, load_tile(buf + (5 + u) * kTileWords), S.gW1[u]);
        }
#pragma unroll
        for (int t = 0; t < 4; t++) {
            const mlp_s4 h1T = load_tile(buf + (9 + t) * kTileWords);
#pragma unroll
            for (int u = 0; u < 4; u++) S.gW2[t][u] = mfma16(h1T, dz2T[u], S.gW2[t][u]);
        }
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");  // read before the next tile's stores
    }
    // reduce the per-sample sums over the 16 lanes of each group
#pragma unroll
    for (int t = 0; t < 4; t++)
#pragma unroll
        for (int i = 0; i < 4; i++) {
            float a = S.gb1[t][i], b = S.gb2[t][i], c = S.gw3[t][i];
#pragma unroll
            for (int o = 1; o < 16; o <<= 1) {
                a += __shfl_xor(a, o);
                b += __shfl_xor(b, o);
                c += __shfl_xor(c, o);
            }
            S.gb1[t][i] = a;
            S.gb2[t][i] = b;
            S.gw3[t][i] = c;
        }
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
        S.gb3 += __shfl_xor(S.gb3, o);
        S.loss += __shfl_xor(S.loss, o);
    }
    // the workgroup's sum: (wavefront 0 + 2) + (1 + 3)
    float *sums = reinterpret_cast<float *>(s_mem);
    float *mine = sums + (wv & 1) * kMlpStride;
    float *row = gpart + (i64)blockIdx.x * kMlpStride;
    __syncthreads();  // every wavefront is past its tiles
    if (wv >= 2) S.each([&](int p, float x) { return mine[p] = x; });
    __syncthreads();
    if (wv < 2) S.each([&](int p, float x) { return x + mine[p]; });
    if (wv == 1) S.each([&](int p, float x) { return mine[p] = x; });  // its own half, read by itself above
    __syncthreads();
    if (wv == 0) S.each([&](int p, float x) { return row[p] = x + sums[kMlpStride + p]; });
}

// Column p of the partial rows, summed by kRedParts threads, each a strided part
// of the rows with kRedFlight loads in flight, then the parts in order (thread
// part 0 holds the sum).  512 rows (10 MB) with a thread per column, one load
// after the other, took 110 us; 4 us so.
constexpr int kRedCols = 64, kRedParts = 16, kRedFlight = 8;
__device__ inline float column_sum(const float *gpart, i64 nrows, int p, float (*sh)[kRedCols]) {
    const int c = threadIdx.x % kRedCols, part = threadIdx.x / kRedCols;
    float s = 0.f;
    if (p <= kMlpParams)
        for (i64 w0 = part; w0 < nrows; w0 += kRedParts * kRedFlight) {
            float x[kRedFlight];
#pragma unroll
            for (int k = 0; k < kRedFlight; k++) {
                const i64 w = w0 + k * kRedParts;
                x[k] = w < nrows ? gpart[w * kMlpStride + p] : 0.f;
            }
#pragma unroll
            for (int k = 0; k < kRedFlight; k++) s += x[k];
        }
    sh[part][c] = s;
    __syncthreads();
    if (part == 0)
        for (int q = 1; q < kRedParts; q++) s += sh[q][c];
    return s;
}

__global__ __launch_bounds__(kRedCols *kRedParts) void k_mlp_reduce(const float *gpart, i64 nrows, float *grad) {
    __shared__ float sh[kRedParts][kRedCols];
    const int p = blockIdx.x * kRedCols + threadIdx.x % kRedCols;
    const float s = column_sum(gpart, nrows, p, sh);
    if (threadIdx.x < kRedCols && p <= kMlpParams) grad[p] = s;
}

__global__ __launch_bounds__(kRedCols *kRedParts) void k_mlp_adam(float *P, float *m, float *v, const float *gpart,
                                                                  i64 nrows, float lr, float b1, float b2, float eps,
                                                                  float c1, float c2, float *loss) {
    __shared__ float sh[kRedParts][kRedCols];
    const int p = blockIdx.x * kRedCols + threadIdx.x % kRedCols;
    const float g = column_sum(gpart, nrows, p, sh);
    if (threadIdx.x >= kRedCols || p > kMlpParams) return;
    if (p == kMlpParams) {
        if (loss) *loss = g;
        return;
    }
    const float mm = b1 * m[p] + (1.0f - b1) * g;
    const float vv = b2 * v[p] + (1.0f - b2) * g * g;
    m[p] = mm;
    v[p] = vv;
    P[p] -= lr * (mm * c1) / (sqrtf(vv * c2) + eps);
}

}  // namespace

#define GLV_LAUNCH_CHECK() GLV_HIP(hipGetLastError())

void launch_mlp_forward(const float *P, const uint16_t *feats, i64 n, float *logits, hipStream_t s) {
    if (n <= 0) return;
    const i64 tiles = (n + 15) / 16;
    const unsigned blocks = (unsigned)std::min<i64>((tiles + kWpb - 1) / kWpb, 8192);
    k_mlp_forward<<<blocks, kMlpBlock, 0, s>>>(P, feats, n, logits);
    GLV_LAUNCH_CHECK();
}

i64 mlp_grad_rows(i64 batch) {
    const i64 tiles = (batch + 15) / 16;
    return std::min<i64>((tiles + kWpb - 1) / kWpb, kMlpMaxRows);
}

void launch_mlp_grad_partials(const float *P, const MlpBatch &B, float *gpart, hipStream_t s) {
    if (B.batch <= 0) return;
    if (B.random && B.n <= 0) fail(GLV_E_INVALID_ARG, "empty sample set");
    k_mlp_grad<<<(unsigned)mlp_grad_rows(B.batch), kMlpBlock, 0, s>>>(P, B, gpart);
    GLV_LAUNCH_CHECK();
}

constexpr unsigned kRedGrid = (kMlpParams + 1 + kRedCols - 1) / kRedCols;
void launch_mlp_reduce(const float *gpart, i64 nrows, float *grad, hipStream_t s) {
    k_mlp_reduce<<<kRedGrid, kRedCols * kRedParts, 0, s>>>(gpart, nrows, grad);
    GLV_LAUNCH_CHECK();
}

void launch_mlp_adam(float *P, float *m, float *v, const float *gpart, i64 nrows, float lr, float beta1,
                     float beta2, float eps, float c1, float c2, float *loss, hipStream_t s) {
    k_mlp_adam<<<kRedGrid, kRedCols * kRedParts, 0, s>>>(P, m, v, gpart, nrows, lr, beta1, beta2, eps, c1, c2, loss);
    GLV_LAUNCH_CHECK();
}

}  // namespace glv
