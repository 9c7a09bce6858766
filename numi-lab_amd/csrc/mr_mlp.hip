// Warm-start MLP training kernels (gfx950): forward with recorded
// activations, MSE loss gradient, backward (matrix-core GEMMs over the batch)
// and Adam. All matrix products take BF16 operands and accumulate in FP32 on
// v_mfma_f32_16x16x32_bf16; every reduction runs in a fixed order, so a
// training run repeats bit for bit.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "mr_mlp_host.h"
#include "mr_mlp_tile.h"

namespace {

using mr::kMlpHidden;
using mr::kMlpIn;
using mr::kMlpOut;
using mr::kMlpRows;
using mr::mlp_bf16x8;
using mr::mlp_f32x4;
using mr::MlpView;

// Forward pass over tiles of 16 rows, four wavefronts a workgroup, each owning 64
// of the 256 hidden columns: its slice of W2 (64 x 256 BF16, 128 registers a lane)
// is read once and stays in registers while the workgroup walks its tiles, so a
// row costs no weight traffic. (One wavefront per tile streamed the 128 KB of W2
// from L2 for every 16 rows: 800 MB for 100,003 rows.) What is left is the
// activations, 512 a row. The tile's h1 and h2 pass through LDS; the four
// wavefronts take turns at the small output layer. Two workgroups share a CU, one
// in its products while the other evaluates GELU.
// Measured, 100,003 rows: 160 -> 84 us; 8192 rows with trace: 48 -> 21 us.
constexpr uint32_t kForwardGroups = 512u;  // two per CU

template <bool kTrace>
__global__ void __launch_bounds__(256, 2) mlp_forward_kernel(MlpView m, const float* x, uint32_t n, float* y_hat,
                                                             mr::MlpTrace trace) {
    __shared__ float s_x[kMlpRows * kMlpIn];
    __shared__ __align__(16) __bf16 s_h1[kMlpRows * mr::kMlpHStride];
    __shared__ __align__(16) __bf16 s_h2[kMlpRows * mr::kMlpHStride];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t ar = lane & 15u, kg = lane >> 4;
    mlp_bf16x8 w1[4], w2[4][8];
    float b1[4], b2[4];
#pragma unroll
    for (uint32_t t = 0; t < 4u; ++t) {
        const uint32_t col = wave * 64u + t * 16u + ar;
        b1[t] = m.b1[col];
        b2[t] = m.b2[col];
#pragma unroll
        for (uint32_t e = 0; e < 8u; ++e) w1[t][e] = kg == 0u ? m.w1[(size_t)col * kMlpIn + e] : (__bf16)0.0f;
#pragma unroll
        for (uint32_t kb = 0; kb < 8u; ++kb)
            w2[t][kb] = *reinterpret_cast<const mlp_bf16x8*>(m.w2 + (size_t)col * kMlpHidden + kb * 32u + kg * 8u);
    }
    const uint32_t f = threadIdx.x % kMlpIn;
    const float shift = m.in_shift[f], scale = m.in_scale[f];
    const uint32_t tiles = (n + kMlpRows - 1u) / kMlpRows;
    uint32_t turn = 0u;
    for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x, ++turn) {
        const uint32_t row0 = tile * kMlpRows;
        const uint32_t rows = n - row0 < kMlpRows ? n - row0 : kMlpRows;
        if (threadIdx.x < kMlpRows * kMlpIn) {
            const uint32_t row = threadIdx.x / kMlpIn;
            const float xn = row < rows ? (x[(size_t)row0 * kMlpIn + threadIdx.x] - shift) * scale : 0.0f;
            s_x[threadIdx.x] = xn;
            if (kTrace && row < rows) trace.xq[(size_t)row0 * kMlpIn + threadIdx.x] = (__bf16)xn;
        }
        __syncthreads();
        mlp_bf16x8 a;
#pragma unroll
        for (uint32_t e = 0; e < 8u; ++e) a[e] = kg == 0u ? (__bf16)s_x[ar * kMlpIn + e] : (__bf16)0.0f;
        const auto activate = [&](const mlp_f32x4& acc, float bias, uint32_t t, __bf16* dst, float* z_out, __bf16* h_out) {
            const uint32_t col = wave * 64u + t * 16u + ar;
#pragma unroll
            for (uint32_t r = 0; r < 4u; ++r) {
                const uint32_t row = kg * 4u + r;
                const float z = acc[r] + bias;
                const __bf16 h = (__bf16)mr::mlp_gelu(z);
                dst[row * mr::kMlpHStride + col] = h;
                if (kTrace && row < rows) {
                    z_out[(size_t)(row0 + row) * kMlpHidden + col] = z;
                    h_out[(size_t)(row0 + row) * kMlpHidden + col] = h;
                }
            }
        };
#pragma unroll
        for (uint32_t t = 0; t < 4u; ++t) {
            const mlp_f32x4 zero = {0.0f, 0.0f, 0.0f, 0.0f};
            activate(__builtin_amdgcn_mfma_f32_16x16x32_bf16(a, w1[t], zero, 0, 0, 0), b1[t], t, s_h1, trace.z1, trace.h1);
        }
        __syncthreads();
        mlp_f32x4 acc[4] = {};
#pragma unroll
        for (uint32_t kb = 0; kb < 8u; ++kb) {
            const mlp_bf16x8 h = *reinterpret_cast<const mlp_bf16x8*>(s_h1 + ar * mr::kMlpHStride + kb * 32u + kg * 8u);
#pragma unroll
            for (uint32_t t = 0; t < 4u; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(h, w2[t][kb], acc[t], 0, 0, 0);
        }
#pragma unroll
        for (uint32_t t = 0; t < 4u; ++t) activate(acc[t], b2[t], t, s_h2, trace.z2, trace.h2);
        __syncthreads();
        if (wave == (turn & 3u)) {
            float y[4];
            mr::mlp_output_layer(s_h2, m, lane, y);
            if (ar < kMlpOut) {
#pragma unroll
                for (uint32_t r = 0; r < 4u; ++r) {
                    const uint32_t row = kg * 4u + r;
                    if (row < rows) y_hat[(size_t)(row0 + row) * kMlpOut + ar] = y[r];
                }
            }
        }
    }
}

// d = y_hat - t / out_scale. With delta = 0 the loss is mean(d^2) and
// dy = 2 d / (3 n); with delta > 0 it is the Huber loss, mean(h(d)) with
// h(d) = d^2 / 2 for |d| <= delta, delta (|d| - delta / 2) beyond, and
// dy = clamp(d, -delta, delta) / (3 n). Per-block partial sums of the loss
// terms are summed by mr_mlp_sum_kernel in block order.
extern "C" __global__ void __launch_bounds__(256) mr_mlp_mse_kernel(const float* y_hat, const float* t,
                                                                    const float* out_scale, uint32_t n, float delta,
                                                                    float* dy, float* partial) {
    __shared__ float red[256];
    const uint32_t total = n * kMlpOut;
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    float se = 0.0f;
    if (i < total) {
        const float d = y_hat[i] - t[i] / out_scale[i % kMlpOut];
        if (delta > 0.0f) {
            const float ad = fabsf(d);
            const float g = ad <= delta ? d : (d > 0.0f ? delta : -delta);
            dy[i] = g / (float)total;
            se = ad <= delta ? 0.5f * d * d : delta * (ad - 0.5f * delta);
        } else {
            dy[i] = 2.0f * d / (float)total;
            se = d * d;
        }
    }
    red[threadIdx.x] = se;
    __syncthreads();
    for (uint32_t w = 128u; w > 0u; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0u) partial[blockIdx.x] = red[0];
}

extern "C" __global__ void __launch_bounds__(256) mr_mlp_sum_kernel(const float* partial, uint32_t count,
                                                                    float scale, float* out) {
    __shared__ float red[256];
    float acc = 0.0f;
    for (uint32_t i = threadIdx.x; i < count; i += 256u) acc += partial[i];
    red[threadIdx.x] = acc;
    __syncthreads();
    for (uint32_t w = 128u; w > 0u; w >>= 1) {
        if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0u) *out = red[0] * scale;
}

// Hidden-layer backward over tiles of 16 rows:
//   dz2[m][j] = (sum_o dy[m][o] W3[o][j]) * gelu'(z2[m][j])
//   dz1[m][i] = (sum_j dz2[m][j] W2[j][i]) * gelu'(z1[m][i])
// laid out like the forward kernel: each of four wavefronts holds its 64 columns
// of W2 (now by input) in registers, dz2 of the tile goes to memory in FP32 and
// to LDS as the BF16 operand of the second product.
// Measured, 8192 rows: 6.7 + 69 us (elementwise pass, strided GEMM) -> 25 us.
__global__ void __launch_bounds__(256, 2) mlp_hidden_backward_kernel(MlpView m, const float* dy, const float* z2,
                                                                     const float* z1, uint32_t n, float* dz2,
                                                                     float* dz1) {
    __shared__ __align__(16) __bf16 s_d[kMlpRows * mr::kMlpHStride];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t ar = lane & 15u, kg = lane >> 4;
    const uint32_t j = threadIdx.x;
    // the first tile's activations are on their way before the weights are asked for
    float zb[kMlpRows];
    const auto load_z2 = [&](uint32_t row0, uint32_t rows) {
#pragma unroll
        for (uint32_t r = 0; r < kMlpRows; ++r)
            zb[r] = r < rows ? z2[(size_t)(row0 + r) * kMlpHidden + j] : 0.0f;
    };
    load_z2(blockIdx.x * kMlpRows, n - blockIdx.x * kMlpRows);
    mlp_bf16x8 w2[4][8];
#pragma unroll
    for (uint32_t t = 0; t < 4u; ++t)
#pragma unroll
        for (uint32_t kb = 0; kb < 8u; ++kb)
#pragma unroll
            for (uint32_t e = 0; e < 8u; ++e)
                w2[t][kb][e] = m.w2[(size_t)(kb * 32u + kg * 8u + e) * kMlpHidden + wave * 64u + t * 16u + ar];
    float w3[kMlpOut];
#pragma unroll
    for (uint32_t o = 0; o < kMlpOut; ++o) w3[o] = (float)m.w3[(size_t)o * kMlpHidden + j];
    const uint32_t tiles = (n + kMlpRows - 1u) / kMlpRows;
    for (uint32_t tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
        const uint32_t row0 = tile * kMlpRows;
        const uint32_t rows = n - row0 < kMlpRows ? n - row0 : kMlpRows;
        if (tile != blockIdx.x) load_z2(row0, rows);
        float za[4][4];
#pragma unroll
        for (uint32_t t = 0; t < 4u; ++t)
#pragma unroll
            for (uint32_t r = 0; r < 4u; ++r) {
                const uint32_t row = kg * 4u + r;
                za[t][r] = row < rows ? z1[(size_t)(row0 + row) * kMlpHidden + wave * 64u + t * 16u + ar] : 0.0f;
            }
#pragma unroll
        for (uint32_t r = 0; r < kMlpRows; ++r) {
            float v = 0.0f;
            if (r < rows) {
                const size_t at = (size_t)(row0 + r);
                float g = 0.0f;
#pragma unroll
                for (uint32_t o = 0; o < kMlpOut; ++o) g += dy[at * kMlpOut + o] * w3[o];
                v = g * mr::mlp_gelu_grad(zb[r]);
                dz2[at * kMlpHidden + j] = v;
            }
            s_d[r * mr::kMlpHStride + j] = (__bf16)v;
        }
        __syncthreads();
        mlp_f32x4 acc[4] = {};
#pragma unroll
        for (uint32_t kb = 0; kb < 8u; ++kb) {
            const mlp_bf16x8 d = *reinterpret_cast<const mlp_bf16x8*>(s_d + ar * mr::kMlpHStride + kb * 32u + kg * 8u);
#pragma unroll
            for (uint32_t t = 0; t < 4u; ++t) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(d, w2[t][kb], acc[t], 0, 0, 0);
        }
#pragma unroll
        for (uint32_t t = 0; t < 4u; ++t) {
            const uint32_t col = wave * 64u + t * 16u + ar;
#pragma unroll
            for (uint32_t r = 0; r < 4u; ++r) {
                const uint32_t row = kg * 4u + r;
                if (row < rows) dz1[(size_t)(row0 + row) * kMlpHidden + col] = acc[t][r] * mr::mlp_gelu_grad(za[t][r]);
            }
        }
        __syncthreads();
    }
}

// Weight gradient C[i][j] = sum_p A[p][i] B[p][j] over a long row axis p
// (the batch): A FP32 [K][M], B BF16 [K][N], both fed to the matrix cores as
// BF16 with FP32 accumulation. One workgroup of 16 wavefronts per 16x16 output
// tile: wavefront w takes the 32-row chunks w, w + 16, w + 32, ... of p, and the
// 16 partial tiles are summed through LDS in wavefront order, so the result does
// not depend on scheduling. The workgroups of the first column tile also return
// bias[i] = sum_p A[p][i] from the FP32 values (the bias gradient), summed in
// the same fixed order. Whole chunks are loaded four at a time without row
// checks, so that 64 loads are in flight a lane: the pass is bound by their
// latency (one chunk at a time, with checks, took twice as long).
constexpr uint32_t kWgradWaves = 16u;

struct WgradShared {
    float tile[kWgradWaves][16][17];
    float bias[kWgradWaves][4][16];
};

__device__ __forceinline__ void wgrad_tile(WgradShared& s, uint32_t M, uint32_t N, uint32_t K, const float* A,
                                           const __bf16* B, float* C, float* bias, uint32_t i0, uint32_t j0) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t ar = lane & 15u, kg = lane >> 4;
    const bool in_a = i0 + ar < M, in_b = j0 + ar < N;
    // columns past the edge read column 0 and count as zero
    const float* ap = A + (in_a ? i0 + ar : 0u);
    const __bf16* bp = B + (in_b ? j0 + ar : 0u);
    const __bf16 zero = (__bf16)0.0f;
    mlp_f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    float bsum = 0.0f;
    constexpr uint32_t kStep = kWgradWaves * 32u, kDeep = 4u;
    uint32_t p0 = wave * 32u;
    const auto product = [&](const float (&av)[8], const __bf16 (&bv)[8]) {
        mlp_bf16x8 a, b;
#pragma unroll
        for (uint32_t e = 0; e < 8u; ++e) {
            bsum += av[e];
            a[e] = (__bf16)av[e];
            b[e] = bv[e];
        }
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
    };
    for (; p0 + (kDeep - 1u) * kStep + 32u <= K; p0 += kDeep * kStep) {
        float av[kDeep][8];
        __bf16 bv[kDeep][8];
#pragma unroll
        for (uint32_t d = 0; d < kDeep; ++d)
#pragma unroll
            for (uint32_t e = 0; e < 8u; ++e) {
                const size_t p = p0 + d * kStep + kg * 8u + e;
                av[d][e] = ap[p * M];
                bv[d][e] = bp[p * N];
            }
#pragma unroll
        for (uint32_t d = 0; d < kDeep; ++d) {
#pragma unroll
            for (uint32_t e = 0; e < 8u; ++e) {
                av[d][e] = in_a ? av[d][e] : 0.0f;
                bv[d][e] = in_b ? bv[d][e] : zero;
            }
            product(av[d], bv[d]);
        }
    }
    for (; p0 < K; p0 += kStep) {
        float av[8];
        __bf16 bv[8];
#pragma unroll
        for (uint32_t e = 0; e < 8u; ++e) {
            const size_t p = p0 + kg * 8u + e;
            av[e] = in_a && p < K ? ap[p * M] : 0.0f;
            bv[e] = in_b && p < K ? bp[p * N] : zero;
        }
        product(av, bv);
    }
#pragma unroll
    for (uint32_t r = 0; r < 4u; ++r) s.tile[wave][kg * 4u + r][ar] = acc[r];
    s.bias[wave][kg][ar] = bsum;
    __syncthreads();
    if (threadIdx.x < 256u) {
        const uint32_t row = threadIdx.x >> 4, col = threadIdx.x & 15u;
        float v = 0.0f;
        for (uint32_t w = 0; w < kWgradWaves; ++w) v += s.tile[w][row][col];
        const uint32_t i = i0 + row, j = j0 + col;
        if (i < M && j < N) C[(size_t)i * N + j] = v;
    } else if (j0 == 0u && threadIdx.x < 272u) {
        const uint32_t row = threadIdx.x - 256u;
        float v = 0.0f;
        for (uint32_t w = 0; w < kWgradWaves; ++w)
            for (uint32_t g = 0; g < 4u; ++g) v += s.bias[w][g][row];
        if (i0 + row < M) bias[i0 + row] = v;
    }
}

// The same for the 256 x 256 gradient, 32x32 outputs a workgroup: a lane loads two
// neighbouring columns of A and of B at once (fragment f holds the columns of
// parity f), so that every 128-byte line of A is used whole and half of each of
// B's. With 16x16 tiles the lines fetched, 540 MB for 8192 rows, bound the pass.
// Each output keeps the order of its sum.
struct WgradWide {
    float tile[kWgradWaves][32][33];
    float bias[kWgradWaves][4][32];
};

typedef float mlp_f32x2 __attribute__((ext_vector_type(2), aligned(4)));
typedef __bf16 mlp_bf16x2 __attribute__((ext_vector_type(2), aligned(2)));

__device__ __forceinline__ void wgrad_wide_tile(WgradWide& s, uint32_t K, const float* A, const __bf16* B, float* C,
                                                float* bias, uint32_t i0, uint32_t j0) {
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t ar = lane & 15u, kg = lane >> 4;
    const float* ap = A + i0 + 2u * ar;
    const __bf16* bp = B + j0 + 2u * ar;
    mlp_f32x4 acc[2][2] = {};
    float bsum[2] = {0.0f, 0.0f};
    constexpr uint32_t kStep = kWgradWaves * 32u, kDeep = 2u;
    const auto product = [&](const mlp_f32x2 (&av)[8], const mlp_bf16x2 (&bv)[8]) {
        mlp_bf16x8 a[2], b[2];
#pragma unroll
        for (uint32_t e = 0; e < 8u; ++e)
#pragma unroll
            for (uint32_t f = 0; f < 2u; ++f) {
                bsum[f] += av[e][f];
                a[f][e] = (__bf16)av[e][f];
                b[f][e] = bv[e][f];
            }
#pragma unroll
        for (uint32_t fa = 0; fa < 2u; ++fa)
#pragma unroll
            for (uint32_t fb = 0; fb < 2u; ++fb)
                acc[fa][fb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[fa], b[fb], acc[fa][fb], 0, 0, 0);
    };
    uint32_t p0 = wave * 32u;
    for (; p0 + (kDeep - 1u) * kStep + 32u <= K; p0 += kDeep * kStep) {
        mlp_f32x2 av[kDeep][8];
        mlp_bf16x2 bv[kDeep][8];
#pragma unroll
        for (uint32_t d = 0; d < kDeep; ++d)
#pragma unroll
            for (uint32_t e = 0; e < 8u; ++e) {
                const size_t p = (size_t)(p0 + d * kStep + kg * 8u + e) * kMlpHidden;
                av[d][e] = *reinterpret_cast<const mlp_f32x2*>(ap + p);
                bv[d][e] = *reinterpret_cast<const mlp_bf16x2*>(bp + p);
            }
#pragma unroll
        for (uint32_t d = 0; d < kDeep; ++d) product(av[d], bv[d]);
    }
    for (; p0 < K; p0 += kStep) {
        mlp_f32x2 av[8] = {};
        mlp_bf16x2 bv[8] = {};
#pragma unroll
        for (uint32_t e = 0; e < 8u; ++e) {
            const uint32_t row = p0 + kg * 8u + e;
            if (row < K) {
                av[e] = *reinterpret_cast<const mlp_f32x2*>(ap + (size_t)row * kMlpHidden);
                bv[e] = *reinterpret_cast<const mlp_bf16x2*>(bp + (size_t)row * kMlpHidden);
            }
        }
        product(av, bv);
    }
#pragma unroll
    for (uint32_t fa = 0; fa < 2u; ++fa) {
#pragma unroll
        for (uint32_t fb = 0; fb < 2u; ++fb)
#pragma unroll
            for (uint32_t r = 0; r < 4u; ++r) s.tile[wave][2u * (kg * 4u + r) + fa][2u * ar + fb] = acc[fa][fb][r];
        s.bias[wave][kg][2u * ar + fa] = bsum[fa];
    }
    __syncthreads();
    const uint32_t row = threadIdx.x >> 5, col = threadIdx.x & 31u;
    float v = 0.0f;
    for (uint32_t w = 0; w < kWgradWaves; ++w) v += s.tile[w][row][col];
    C[(size_t)(i0 + row) * kMlpHidden + j0 + col] = v;
    if (j0 == 0u && threadIdx.x < 32u) {
        float b = 0.0f;
        for (uint32_t w = 0; w < kWgradWaves; ++w)
            for (uint32_t g = 0; g < 4u; ++g) b += s.bias[w][g][threadIdx.x];
        bias[i0 + threadIdx.x] = b;
    }
}

// All weight and bias gradients in one launch: workgroups 0-63 the tiles of
// dW2 = dz2^T h1, 64-79 the 16 tiles of dW3 = dy^T h2, 80-95 those of
// dW1 = dz1^T xq. As launches of their own each of the thin products kept 16 of
// 256 CUs busy for as long as the large one took.
// Measured, 8192 rows: 3 x 23.5 us -> 36 us.
constexpr uint32_t kWgradTiles = 64u + 16u + 16u;

__global__ void __launch_bounds__(1024) mlp_wgrad_kernel(uint32_t n, const float* dy, const float* dz2,
                                                         const float* dz1, mr::MlpTrace tr, MRMlpGradsC g) {
    __shared__ union {
        WgradWide wide;
        WgradShared thin;
    } s;
    const uint32_t b = blockIdx.x;
    if (b < 64u)
        wgrad_wide_tile(s.wide, n, dz2, tr.h1, g.w2, g.b2, (b >> 3) * 32u, (b & 7u) * 32u);
    else if (b < 80u)
        wgrad_tile(s.thin, kMlpOut, kMlpHidden, n, dy, tr.h2, g.w3, g.b3, 0u, (b - 64u) * 16u);
    else
        wgrad_tile(s.thin, kMlpHidden, kMlpIn, n, dz1, tr.xq, g.w1, g.b1, (b - 80u) * 16u, 0u);
}

// One Adam step on up to kAdamTensors tensors: workgroup b works on the tensor
// whose range of workgroups [first, next first) holds b. The network's six
// parameters took six launches of a few microseconds each for 67,587 values.
// A tensor of more than 2^31 values enters as several, and a launch stays below 2^32 threads.
constexpr uint32_t kAdamTensors = 8u;
constexpr uint32_t kAdamValues = 1u << 31;
constexpr uint32_t kAdamGroups = 1u << 23;

struct AdamArgs {
    MRMlpAdamTensorC tensor[kAdamTensors];
    uint32_t first[kAdamTensors];  // first workgroup of each tensor
    uint32_t tensors;
};

extern "C" __global__ void __launch_bounds__(256) mr_mlp_adam_kernel(AdamArgs args, float lr, float beta1, float beta2,
                                                                     float eps, float c1, float c2) {
    uint32_t k = 0u;
    while (k + 1u < args.tensors && args.first[k + 1u] <= blockIdx.x) ++k;
    const MRMlpAdamTensorC t = args.tensor[k];
    const uint32_t i = (blockIdx.x - args.first[k]) * 256u + threadIdx.x;
    if (i >= t.count) return;
    const float gi = t.grad[i];
    const float a = beta1 * t.m1[i] + (1.0f - beta1) * gi;
    const float b = beta2 * t.m2[i] + (1.0f - beta2) * gi * gi;
    t.m1[i] = a;
    t.m2[i] = b;
    const float ahat = a / c1, bhat = b / c2;
    const float wi = t.param[i] - lr * ahat / (sqrtf(bhat) + eps);
    t.param[i] = wi;
    if (t.param_bf16 != nullptr) reinterpret_cast<__bf16*>(t.param_bf16)[i] = (__bf16)wi;
}

MlpView view_of(const MRMlpWeightsC& w) {
    MlpView m;
    m.w1 = reinterpret_cast<const __bf16*>(w.w1);
    m.b1 = w.b1;
    m.w2 = reinterpret_cast<const __bf16*>(w.w2);
    m.b2 = w.b2;
    m.w3 = reinterpret_cast<const __bf16*>(w.w3);
    m.b3 = w.b3;
    m.in_shift = w.in_shift;
    m.in_scale = w.in_scale;
    m.out_scale = w.out_scale;
    return m;
}

mr::MlpTrace trace_of(const MRMlpTraceC& t) {
    mr::MlpTrace r;
    r.xq = reinterpret_cast<__bf16*>(t.xq);
    r.z1 = t.z1;
    r.h1 = reinterpret_cast<__bf16*>(t.h1);
    r.z2 = t.z2;
    r.h2 = reinterpret_cast<__bf16*>(t.h2);
    return r;
}

} // namespace

namespace mr {

hipError_t mlp_forward(const MRMlpWeightsC& w, const float* x, uint32_t n, float* y_hat, const MRMlpTraceC* trace,
                       hipStream_t st) {
    const MlpView m = view_of(w);
    const uint32_t tiles = (n + kMlpRows - 1u) / kMlpRows;
    const dim3 grid(tiles < kForwardGroups ? tiles : kForwardGroups);
    if (trace != nullptr)
        hipLaunchKernelGGL((mlp_forward_kernel<true>), grid, dim3(256), 0, st, m, x, n, y_hat, trace_of(*trace));
    else
        hipLaunchKernelGGL((mlp_forward_kernel<false>), grid, dim3(256), 0, st, m, x, n, y_hat, MlpTrace{});
    return hipGetLastError();
}

uint32_t mlp_loss_scratch_floats(uint32_t n) { return (n * kMlpOut + 255u) / 256u; }

hipError_t mlp_loss(const float* y_hat, const float* t, const float* out_scale, uint32_t n, float delta, float* dy,
                    float* loss, float* scratch, hipStream_t st) {
    const uint32_t blocks = mlp_loss_scratch_floats(n);
    hipLaunchKernelGGL(mr_mlp_mse_kernel, dim3(blocks), dim3(256), 0, st, y_hat, t, out_scale, n, delta, dy,
                       scratch);
    hipLaunchKernelGGL(mr_mlp_sum_kernel, dim3(1), dim3(256), 0, st, scratch, blocks, 1.0f / (float)(n * kMlpOut),
                       loss);
    return hipGetLastError();
}

hipError_t mlp_backward(const MRMlpWeightsC& w, const MRMlpTraceC& trc, const float* dy, uint32_t n, float* dz2,
                        float* dz1, const MRMlpGradsC& g, hipStream_t st) {
    const MlpView m = view_of(w);
    const MlpTrace tr = trace_of(trc);
    const uint32_t tiles = (n + kMlpRows - 1u) / kMlpRows;
    hipLaunchKernelGGL(mlp_hidden_backward_kernel, dim3(tiles < kForwardGroups ? tiles : kForwardGroups), dim3(256), 0,
                       st, m, dy, tr.z2, tr.z1, n, dz2, dz1);
    hipLaunchKernelGGL(mlp_wgrad_kernel, dim3(kWgradTiles), dim3(64u * kWgradWaves), 0, st, n, dy, dz2, dz1, tr, g);
    return hipGetLastError();
}

hipError_t mlp_adam(const MRMlpAdamTensorC* tensors, uint32_t tensor_count, float lr, float beta1, float beta2,
                    float eps, uint32_t step, hipStream_t st) {
    float c1 = 1.0f, c2 = 1.0f;
    for (uint32_t k = 0; k < step; ++k) {
        c1 *= beta1;
        c2 *= beta2;
    }
    c1 = 1.0f - c1;
    c2 = 1.0f - c2;
    AdamArgs args{};
    uint32_t groups = 0u;
    const auto launch = [&] {
        if (groups > 0u)
            hipLaunchKernelGGL(mr_mlp_adam_kernel, dim3(groups), dim3(256), 0, st, args, lr, beta1, beta2, eps, c1, c2);
        args.tensors = 0u;
        groups = 0u;
    };
    for (uint32_t k = 0; k < tensor_count; ++k) {
        MRMlpAdamTensorC rest = tensors[k];
        while (rest.count > 0u) {
            const uint32_t n = rest.count < kAdamValues ? rest.count : kAdamValues;
            const uint32_t own = (n + 255u) / 256u;
            if (args.tensors == kAdamTensors || groups + own > kAdamGroups) launch();
            args.tensor[args.tensors] = rest;
            args.tensor[args.tensors].count = n;
            args.first[args.tensors++] = groups;
            groups += own;
            rest.param += n;
            rest.param_bf16 += rest.param_bf16 != nullptr ? n : 0u;
            rest.grad += n;
            rest.m1 += n;
            rest.m2 += n;
            rest.count -= n;
        }
    }
    launch();
    return hipGetLastError();
}

} // namespace mr
