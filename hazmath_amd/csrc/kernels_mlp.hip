// kernels_mlp.hip -- the per-aggregate parameter network: an MLP
// 12 -> 64 -> 64 -> 2 with GELU, FP32, forward and backward on the FP32
// matrix cores (v_mfma_f32_16x16x4f32), full-precision FP32 Adam.
//
// Parameters live in one FP32 vector (row-major):
//   W1 [16][64] (inputs 12..15 are zero padding), b1 [64],
//   W2 [64][64], b2 [64], W3 [64][16] (outputs 2..15 are padding), b3 [16].
// Batches are padded to a multiple of 64 rows; padded rows carry zero weight in
// the loss, so they contribute nothing to gradients.
// Loss: mean squared error over the two outputs and the valid rows.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include <mutex>

#include "hz_internal.h"

// Scratch memory of hz_mlp_forward_noalloc: the padded inputs and the two
// hidden layers and padded outputs of up to kNoAllocRows rows (160 floats a
// row, 10 MiB).  Each GPU holds its own copy for the life of the process; host
// code reaches it only through the address hipGetSymbolAddress returns for the
// current device, never through this name.
constexpr int kNoAllocRows = HZ_MLP_NOALLOC_MAX_ROWS;
constexpr size_t kNoAllocFloats = (size_t)kNoAllocRows * (16 + 64 + 64 + 16);
static __device__ __align__(256) float scratch[kNoAllocFloats];

namespace hz {

namespace {

constexpr int kIn = 16, kHid = 64, kOut = 16;
constexpr int kOffW1 = 0, kOffB1 = kOffW1 + kIn * kHid, kOffW2 = kOffB1 + kHid, kOffB2 = kOffW2 + kHid * kHid,
              kOffW3 = kOffB2 + kHid, kOffB3 = kOffW3 + kHid * kOut, kParams = kOffB3 + kOut;
static_assert(kParams == HZ_MLP_PARAMS, "parameter layout");
constexpr int kRows = 64;   // batch rows per tile

typedef float f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }

enum Epi { kEpiNone = 0, kEpiGelu = 1 };

// C[M x N] = A[M x K] B + bias, K <= 64, N <= 64 (the forward pass).  One
// workgroup (4 wavefronts) per 64-row tile; wavefront w owns rows 16w..16w+15
// and all N columns as 16x16 MFMA blocks.  Epilogue kEpiGelu: C = gelu(C).
// MFMA f32 16x16x4 lanes: A[lane % 16][k + lane / 16], B[k + lane / 16][lane % 16],
// accumulator element r = D[4 (lane / 16) + r][lane % 16].
template <int kEpi>
__global__ __launch_bounds__(256) void k_mlp_gemm(int M, int N, int K, const float *__restrict__ A,
                                                  const float *__restrict__ B, const float *__restrict__ bias,
                                                  float *__restrict__ C) {
    __shared__ float As[kRows][65];
    __shared__ float Bs[64][65];
    const int r0 = blockIdx.x * kRows;
    const int tid = threadIdx.x;
    for (int e = tid; e < kRows * 64; e += 256) {
        const int r = e / 64, k = e % 64;
        As[r][k] = (r0 + r < M && k < K) ? A[(size_t)(r0 + r) * K + k] : 0.0f;
    }
    for (int e = tid; e < 64 * 64; e += 256) {
        const int k = e / 64, c = e % 64;
        Bs[k][c] = k < K && c < N ? B[(size_t)k * N + c] : 0.0f;
    }
    __syncthreads();
    const int w = tid / kWave, lane = tid % kWave;
    const int nb = (N + 15) / 16;
    f4 acc[4];
    for (int j = 0; j < 4; ++j) acc[j] = f4{0.0f, 0.0f, 0.0f, 0.0f};
    const int kpad = (K + 3) & ~3;
    for (int ks = 0; ks < kpad; ks += 4) {
        const float a = As[16 * w + lane % 16][ks + lane / 16];
        for (int j = 0; j < nb; ++j) {
            const float b = Bs[ks + lane / 16][16 * j + lane % 16];
            acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc[j], 0, 0, 0);
        }
    }
    for (int j = 0; j < nb; ++j)
        for (int r = 0; r < 4; ++r) {
            const int row = r0 + 16 * w + 4 * (lane / 16) + r;
            const int col = 16 * j + lane % 16;
            if (row >= M || col >= N) continue;
            const float v = acc[j][r] + bias[col];
            C[(size_t)row * N + col] = kEpi == kEpiGelu ? gelu(v) : v;
        }
}

// Loss and gradient partials of the network in one pass over the batch.
//
// Layer by layer this read and wrote eight 64-column activations a row (2 KB of
// traffic for 56 bytes of input) in eleven launches, and the sums over partials
// ran on 17 blocks and one thread.  The whole network is 25 KB, so a workgroup
// keeps it in LDS and takes its 64-row tiles through forward and backward
// there: only inputs and targets are read, and a workgroup's 6,288 gradient
// sums, held in MFMA accumulators over its tiles, are written once.  96 KB of
// LDS: one workgroup a CU, eight wavefronts to cover each other's LDS reads
// and erf chains (four took 104 us).  84,400 rows: 877 -> 82 us of kernels.
//
// Wavefront wave = w + 4 half owns rows 16w..16w+15 and the column half `half`
// of a tile's activations and of gW2; gW1 (columns 16w..) and the outputs go to
// half 0, gW3 (rows 16w..) to half 1.  G1, G2 first hold gelu'(Z) and then dZ.
// Rows past the batch have dY = 0 and add nothing.  MFMA lanes as in k_mlp_gemm.
constexpr int kGradThreads = 512;
struct GradTile {
    float W1[kIn][kHid + 1], W2[kHid][kHid + 1], W3[kHid][kOut + 1];
    float b1[kHid], b2[kHid], b3[kOut];
    float X[kRows][kIn + 1], D[kRows][kOut + 1];
    float H1[kRows][kHid + 1], H2[kRows][kHid + 1], G1[kRows][kHid + 1], G2[kRows][kHid + 1];
};

// gelu(z) and its derivative from one erf: 0.5 z (1 + e) and 0.5 (1 + e) + z pdf
__device__ __forceinline__ void gelu_both(float z, float &h, float &g) {
    const float cdf = 0.5f * (1.0f + erff(z * 0.70710678118654752f));
    h = z * cdf;
    g = cdf + z * (0.39894228040143268f * expf(-0.5f * z * z));
}

__global__ __launch_bounds__(kGradThreads) void k_mlp_grad(int B, const float *__restrict__ theta, const float *__restrict__ x,
                                                  const float *__restrict__ t, const int *__restrict__ idx,
                                                  float *__restrict__ part, double *__restrict__ lpart) {
    extern __shared__ double s_tile[];
    GradTile &S = *reinterpret_cast<GradTile *>(s_tile);
    __shared__ double sh[kGradThreads / kWave];
    const int tid = threadIdx.x, wave = tid / kWave, lane = tid % kWave;
    const int w = wave % 4, half = wave / 4, j0 = 2 * half;
    const int lm = lane % 16, lk = lane / 16;
    for (int e = tid; e < kIn * kHid; e += kGradThreads) S.W1[e / kHid][e % kHid] = theta[kOffW1 + e];
    for (int e = tid; e < kHid * kHid; e += kGradThreads) S.W2[e / kHid][e % kHid] = theta[kOffW2 + e];
    for (int e = tid; e < kHid * kOut; e += kGradThreads) S.W3[e / kOut][e % kOut] = theta[kOffW3 + e];
    if (tid < kHid) {
        S.b1[tid] = theta[kOffB1 + tid];
        S.b2[tid] = theta[kOffB2 + tid];
    }
    if (tid < kOut) S.b3[tid] = theta[kOffB3 + tid];
    const f4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
    f4 gW1 = zero, gW3 = zero, gW2[2] = {zero, zero};
    // bias gradients: thread's column tid % 64 (tid % 16), rows of its part
    float gb1 = 0.0f, gb2 = 0.0f, gb3 = 0.0f;
    double loss = 0.0;
    const float scale = 1.0f / (2.0f * (float)B);
    const int ntiles = (B + kRows - 1) / kRows;
    for (int tile = blockIdx.x; tile < ntiles; tile += gridDim.x) {
        const int r0 = tile * kRows;
        __syncthreads();   // weights are there; the last tile's readers of X and G1 are done
        for (int e = tid; e < kRows * kIn; e += kGradThreads) {
            const int r = e / kIn, c = e % kIn;
            float v = 0.0f;
            if (r0 + r < B && c < HZ_MLP_INPUTS) v = x[(size_t)(idx ? idx[r0 + r] : r0 + r) * HZ_MLP_INPUTS + c];
            S.X[r][c] = v;
        }
        float tv[4] = {0.0f, 0.0f, 0.0f, 0.0f};   // targets of this lane's outputs
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = r0 + 16 * w + 4 * lk + r;
            if (row < B && lm < HZ_MLP_OUTPUTS) tv[r] = t[(size_t)(idx ? idx[row] : row) * HZ_MLP_OUTPUTS + lm];
        }
        __syncthreads();
        f4 acc[2];
        // layer 1
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[j] = zero;
#pragma unroll
        for (int ks = 0; ks < kIn; ks += 4) {
            const float a = S.X[16 * w + lm][ks + lk];
#pragma unroll
            for (int j = 0; j < 2; ++j)
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, S.W1[ks + lk][16 * (j0 + j) + lm], acc[j], 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 16 * w + 4 * lk + r, col = 16 * (j0 + j) + lm;
                gelu_both(acc[j][r] + S.b1[col], S.H1[row][col], S.G1[row][col]);
            }
        __syncthreads();
        // layer 2
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[j] = zero;
#pragma unroll 4
        for (int ks = 0; ks < kHid; ks += 4) {
            const float a = S.H1[16 * w + lm][ks + lk];
#pragma unroll
            for (int j = 0; j < 2; ++j)
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, S.W2[ks + lk][16 * (j0 + j) + lm], acc[j], 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 16 * w + 4 * lk + r, col = 16 * (j0 + j) + lm;
                gelu_both(acc[j][r] + S.b2[col], S.H2[row][col], S.G2[row][col]);
            }
        __syncthreads();
        // layer 3, dY = 2 (Y - T) / (2 B)
        if (half == 0) {
            acc[0] = zero;
#pragma unroll 4
            for (int ks = 0; ks < kHid; ks += 4)
                acc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(S.H2[16 * w + lm][ks + lk], S.W3[ks + lk][lm], acc[0], 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int row = 16 * w + 4 * lk + r;
                float g = 0.0f;
                if (r0 + row < B && lm < HZ_MLP_OUTPUTS) {
                    const float d = acc[0][r] + S.b3[lm] - tv[r];
                    g = 2.0f * d * scale;
                    loss += (double)d * (double)d;
                }
                S.D[row][lm] = g;
            }
        }
        __syncthreads();
        // gW3 += H2^T dY;  dZ2 = (dY W3^T) gelu'(Z2), own rows of G2
        if (half == 1)
#pragma unroll 4
            for (int ks = 0; ks < kRows; ks += 4)
                gW3 = __builtin_amdgcn_mfma_f32_16x16x4f32(S.H2[ks + lk][16 * w + lm], S.D[ks + lk][lm], gW3, 0, 0, 0);
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[j] = zero;
#pragma unroll
        for (int ks = 0; ks < kOut; ks += 4) {
            const float a = S.D[16 * w + lm][ks + lk];
#pragma unroll
            for (int j = 0; j < 2; ++j)
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, S.W3[16 * (j0 + j) + lm][ks + lk], acc[j], 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) S.G2[16 * w + 4 * lk + r][16 * (j0 + j) + lm] *= acc[j][r];
        if (tid < 4 * kOut)
            for (int r = 0; r < kRows / 4; ++r) gb3 += S.D[tid / kOut * (kRows / 4) + r][tid % kOut];
        __syncthreads();
        // gW2 += H1^T dZ2;  dZ1 = (dZ2 W2^T) gelu'(Z1), own rows of G1
#pragma unroll 4
        for (int ks = 0; ks < kRows; ks += 4) {
            const float a = S.H1[ks + lk][16 * w + lm];
#pragma unroll
            for (int j = 0; j < 2; ++j)
                gW2[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, S.G2[ks + lk][16 * (j0 + j) + lm], gW2[j], 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[j] = zero;
#pragma unroll 4
        for (int ks = 0; ks < kHid; ks += 4) {
            const float a = S.G2[16 * w + lm][ks + lk];
#pragma unroll
            for (int j = 0; j < 2; ++j)
                acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a, S.W2[16 * (j0 + j) + lm][ks + lk], acc[j], 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) S.G1[16 * w + 4 * lk + r][16 * (j0 + j) + lm] *= acc[j][r];
#pragma unroll 4
        for (int r = 0; r < kRows / 8; ++r) gb2 += S.G2[wave * (kRows / 8) + r][lane];
        __syncthreads();
        // gW1 += X^T dZ1
        if (half == 0)
#pragma unroll 4
            for (int ks = 0; ks < kRows; ks += 4)
                gW1 = __builtin_amdgcn_mfma_f32_16x16x4f32(S.X[ks + lk][lm], S.G1[ks + lk][16 * w + lm], gW1, 0, 0, 0);
#pragma unroll 4
        for (int r = 0; r < kRows / 8; ++r) gb1 += S.G1[wave * (kRows / 8) + r][lane];
    }
    float *out = part + (size_t)blockIdx.x * kParams;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (half == 0) out[kOffW1 + (4 * lk + r) * kHid + 16 * w + lm] = gW1[r];
        else out[kOffW3 + (16 * w + 4 * lk + r) * kOut + lm] = gW3[r];
#pragma unroll
        for (int j = 0; j < 2; ++j) out[kOffW2 + (16 * w + 4 * lk + r) * kHid + 16 * (j0 + j) + lm] = gW2[j][r];
    }
    // the bias sums' parts meet in LDS
    __syncthreads();
    S.H1[wave][lane] = gb1;
    S.H2[wave][lane] = gb2;
    if (tid < 4 * kOut) S.D[tid / kOut][tid % kOut] = gb3;
    __syncthreads();
    if (tid < kHid) {
        float v1 = 0.0f, v2 = 0.0f;
        for (int q = 0; q < kGradThreads / kWave; ++q) {
            v1 += S.H1[q][tid];
            v2 += S.H2[q][tid];
        }
        out[kOffB1 + tid] = v1;
        out[kOffB2 + tid] = v2;
    }
    if (tid < kOut) out[kOffB3 + tid] = S.D[0][tid] + S.D[1][tid] + S.D[2][tid] + S.D[3][tid];
    const double bs = block_sum<kGradThreads>(loss, sh);
    if (tid == 0) lpart[blockIdx.x] = bs;
}

// grad[e] = sum over the G partials, a wavefront per quarter of them and 64
// entries a workgroup; the last workgroup forms the loss.
__global__ __launch_bounds__(256) void k_mlp_reduce(int G, int nvalid, const float *__restrict__ part,
                                                    const double *__restrict__ lpart, float *__restrict__ out,
                                                    float *__restrict__ loss) {
    __shared__ float s[4][kWave];
    __shared__ double sh[256 / kWave];
    const int w = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    if (blockIdx.x == gridDim.x - 1) {
        const double tot = final_sum<256>(lpart, G, sh);
        if (threadIdx.x == 0) *loss = (float)(tot / (2.0 * nvalid));
        return;
    }
    const int e = blockIdx.x * kWave + lane;
    const int per = (G + 3) / 4, g1 = min(G, (w + 1) * per);
    float v = 0.0f;
    constexpr int U = 16;
    if (e < kParams)
        for (int g = w * per; g < g1; g += U) {
            float a[U];
#pragma unroll
            for (int u = 0; u < U; ++u) a[u] = g + u < g1 ? part[(size_t)(g + u) * kParams + e] : 0.0f;
#pragma unroll
            for (int u = 0; u < U; ++u) v += a[u];
        }
    s[w][lane] = v;
    __syncthreads();
    if (w == 0 && e < kParams) out[e] = s[0][lane] + s[1][lane] + s[2][lane] + s[3][lane];
}

__global__ void k_mlp_adam(int n, float *__restrict__ th, const float *__restrict__ g, float *__restrict__ m,
                           float *__restrict__ v, float lr, float b1, float b2, float eps, float c1, float c2) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        const float gi = g[i];
        const float mi = b1 * m[i] + (1.0f - b1) * gi;
        const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
        m[i] = mi;
        v[i] = vi;
        th[i] -= lr * (mi / c1) / (sqrtf(vi / c2) + eps);
    }
}

// padded input rows: x[b][0..11], zeros in 12..15 and in padded rows
__global__ void k_mlp_pad_inputs(int B, int M, const float *__restrict__ x, float *__restrict__ X) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < M * kIn; i += gridDim.x * blockDim.x) {
        const int row = i / kIn, c = i % kIn;
        float v = 0.0f;
        if (row < B && c < HZ_MLP_INPUTS) v = x[(size_t)row * HZ_MLP_INPUTS + c];
        X[i] = v;
    }
}

__global__ void k_mlp_take_outputs(int B, const float *__restrict__ Y, float *__restrict__ y) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < B * HZ_MLP_OUTPUTS; i += gridDim.x * blockDim.x)
        y[i] = Y[(i / HZ_MLP_OUTPUTS) * kOut + i % HZ_MLP_OUTPUTS];
}

inline int gsz(long n) { return (int)std::max(1L, std::min<long>((n + 255) / 256, 4096)); }

}  // namespace

MlpWork mlp_work(int capacity) {
    MlpWork w;
    w.cap = (capacity + kRows - 1) / kRows * kRows;
    const size_t M = (size_t)w.cap;
    w.X = arena().alloc_n<float>(M * kIn);
    w.H1 = arena().alloc_n<float>(M * kHid);
    w.H2 = arena().alloc_n<float>(M * kHid);
    w.Y = arena().alloc_n<float>(M * kOut);
    return w;
}

void mlp_forward(const float *theta, const MlpWork &w, int B) {
    hipStream_t st = stream();
    const int M = (B + kRows - 1) / kRows * kRows;
    const int g = M / kRows;
    k_mlp_gemm<kEpiGelu><<<g, 256, 0, st>>>(M, kHid, kIn, w.X, theta + kOffW1, theta + kOffB1, w.H1);
    k_mlp_gemm<kEpiGelu><<<g, 256, 0, st>>>(M, kHid, kHid, w.H1, theta + kOffW2, theta + kOffB2, w.H2);
    k_mlp_gemm<kEpiNone><<<g, 256, 0, st>>>(M, kOut, kHid, w.H2, theta + kOffW3, theta + kOffB3, w.Y);
    HZ_LAUNCH_CHECK();
}

void mlp_inputs(const float *x, int B, const MlpWork &w) {
    const int M = (B + kRows - 1) / kRows * kRows;
    k_mlp_pad_inputs<<<gsz((long)M * kIn), 256, 0, stream()>>>(B, M, x, w.X);
    HZ_LAUNCH_CHECK();
}

void mlp_outputs(int B, const MlpWork &w, float *y) {
    k_mlp_take_outputs<<<gsz((long)B * 2), 256, 0, stream()>>>(B, w.Y, y);
    HZ_LAUNCH_CHECK();
}

MlpGradWork mlp_grad_work() {
    MlpGradWork w;
    w.part = arena().alloc_n<float>((size_t)kMlpGradBlocks * kParams);
    w.lpart = arena().alloc_n<double>(kMlpGradBlocks);
    return w;
}

void mlp_loss_grad(const float *theta, const float *x, const float *t, const int *idx, int B, const MlpGradWork &w,
                   float *grad, float *loss) {
    static const bool ready = [] {
        HZ_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_mlp_grad),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)sizeof(GradTile)));
        return true;
    }();
    (void)ready;
    const int G = std::min(kMlpGradBlocks, (B + kRows - 1) / kRows);
    k_mlp_grad<<<G, kGradThreads, sizeof(GradTile), stream()>>>(B, theta, x, t, idx, w.part, w.lpart);
    HZ_LAUNCH_CHECK();
    k_mlp_reduce<<<(kParams + kWave - 1) / kWave + 1, 256, 0, stream()>>>(G, B, w.part, w.lpart, grad, loss);
    HZ_LAUNCH_CHECK();
}

// The device address of `scratch` on the current device, looked up once per
// device (nullptr when the lookup fails).
static float *noalloc_scratch() {
    static std::mutex mu;
    static float *addr[64] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return nullptr;
    std::lock_guard<std::mutex> lock(mu);
    if (!addr[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) {
            std::fprintf(stderr, "hazmath_mi355x: hipGetSymbolAddress(scratch) failed: %s\n", hipGetErrorString(e));
            return nullptr;
        }
        addr[dev] = static_cast<float *>(p);
    }
    return addr[dev];
}

int mlp_forward_noalloc(const float *theta, const float *x, int B, float *y, hipStream_t st) {
    float *base = noalloc_scratch();
    if (!base) return HZ_ERROR_DEVICE;
    float *X = base;
    float *H1 = X + (size_t)kNoAllocRows * kIn;
    float *H2 = H1 + (size_t)kNoAllocRows * kHid;
    float *Y = H2 + (size_t)kNoAllocRows * kHid;
    const int M = (B + kRows - 1) / kRows * kRows;
    const int g = M / kRows;
    k_mlp_pad_inputs<<<gsz((long)M * kIn), 256, 0, st>>>(B, M, x, X);
    k_mlp_gemm<kEpiGelu><<<g, 256, 0, st>>>(M, kHid, kIn, X, theta + kOffW1, theta + kOffB1, H1);
    k_mlp_gemm<kEpiGelu><<<g, 256, 0, st>>>(M, kHid, kHid, H1, theta + kOffW2, theta + kOffB2, H2);
    k_mlp_gemm<kEpiNone><<<g, 256, 0, st>>>(M, kOut, kHid, H2, theta + kOffW3, theta + kOffB3, Y);
    k_mlp_take_outputs<<<gsz((long)B * 2), 256, 0, st>>>(B, Y, y);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        std::fprintf(stderr, "hazmath_mi355x: hz_mlp_forward_noalloc launch failed: %s\n", hipGetErrorString(e));
        return HZ_ERROR_DEVICE;
    }
    return HZ_SUCCESS;
}

void mlp_adam(float *theta, const float *grad, float *m, float *v, float lr, int step) {
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    const float c1 = 1.0f - std::pow(b1, (float)step), c2 = 1.0f - std::pow(b2, (float)step);
    k_mlp_adam<<<gsz(kParams), 256, 0, stream()>>>(kParams, theta, grad, m, v, lr, b1, b2, eps, c1, c2);
    HZ_LAUNCH_CHECK();
}

}  // namespace hz
