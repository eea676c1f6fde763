// Kernels of the warm-start MLP (in -> hid -> hid -> out, GELU): an FP32
// matrix-core GEMM with fused bias/GELU, GELU-gradient, affine and row-sum
// epilogues, the MSE gradient, Adam, and row normalisation / gathering.
// Weights are read as FP32 (training) or bfloat16 (inference); arithmetic is
// FP32.  Every output element is summed in a fixed order, so results are
// run-to-run deterministic.
#include "ccd_kernels.h"

#include <algorithm>

namespace ccd {
namespace {

constexpr int BLOCK = 256;
constexpr int WAVE = 64;
constexpr int KSTEP = 16;  // K values of a fragment: four per lane

using f32x4 = __attribute__((__vector_size__(4 * sizeof(float)))) float;
// four floats (or four bfloat16) of any alignment that the element type has
struct __attribute__((packed, aligned(4))) Loose4 {
    float v[4];
};
struct __attribute__((packed, aligned(2))) Loose4h {
    uint16_t v[4];
};

template <class T>
__device__ __forceinline__ float ld(const T* p, size_t i) {
    if constexpr (sizeof(T) == 2) return __uint_as_float((uint32_t)p[i] << 16);
    else return p[i];
}

__device__ __forceinline__ float gelu(float z) { return 0.5f * z * (1.0f + erff(z * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_grad(float z) {
    return 0.5f * (1.0f + erff(z * 0.70710678118654752f)) + z * expf(-0.5f * z * z) * 0.39894228040143268f;
}

// Four K values k0 .. k0 + 3 of row i of an operand (element (i, p) at
// X[i si + p sp]); K values from ke on read as zero.  KF: sp == 1.
template <class T, bool KF>
__device__ __forceinline__ f32x4 fragment(const T* __restrict__ X, uint64_t si, uint64_t sp, uint32_t i, uint32_t k0,
                                          uint32_t ke) {
    if (k0 + 4 <= ke) {
        if constexpr (KF && sizeof(T) == 4) {
            const Loose4 x = *reinterpret_cast<const Loose4*>(X + (size_t)i * si + k0);
            return f32x4{x.v[0], x.v[1], x.v[2], x.v[3]};
        } else if constexpr (KF) {
            const Loose4h x = *reinterpret_cast<const Loose4h*>(X + (size_t)i * si + k0);
            return f32x4{ld(x.v, 0), ld(x.v, 1), ld(x.v, 2), ld(x.v, 3)};
        } else {
            const T* q = X + (size_t)i * si + (size_t)k0 * sp;
            return f32x4{ld(q, 0), ld(q, sp), ld(q, 2 * sp), ld(q, 3 * sp)};
        }
    }
    f32x4 r = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (uint32_t u = 0; u < 4; ++u)
        if (k0 + u < ke) r[u] = ld(X, (size_t)i * si + (size_t)(k0 + u) * sp);
    return r;
}

// C(i, j) = sum_p A(i, p) B(p, j), A(i, p) = A[i sai + p sap], B(p, j) = B[p sbp + j sbj]
// on v_mfma_f32_16x16x4_f32 (FP32 products and sums).  A wave computes RT x
// CT tiles of 16 x 16; lane l loads A(i0 + l % 16, k .. k + 3) and
// B(k .. k + 3, j0 + l % 16) with k = 4 (l / 16) of each step of 16 K values,
// one 16-byte load where K is the operand's unit stride, straight into the
// registers of four matrix instructions (which take value u of every lane
// together: a permutation of the step's K values common to both operands).
// The next step's fragments are loaded while a step multiplies; nothing is
// staged in LDS, the operands' rereads are L2 hits (the weights are 0.4 MB).
// AK, BK: K is the operand's unit stride.
// KW > 1: the KW waves of a block share its RT x CT tiles, wave w taking
// steps w, w + KW, ...; their sums are added in wave order through LDS.  For
// few output tiles (a minibatch, a weight gradient) this is what fills the
// chip.  KW == 1: the block's four waves take four row groups.
// blockIdx.z: slice of K when the product is split further (partials to
// g.part).
template <class TB, bool AK, bool BK, int EPI, int RT, int CT, int KW>
__global__ __launch_bounds__(KW > 1 ? KW * WAVE : BLOCK) void gemm_kernel(GemmArgs g, const TB* __restrict__ B) {
    extern __shared__ __align__(16) float gemm_lds[];
    const uint32_t lane = threadIdx.x & (WAVE - 1), wv = threadIdx.x / WAVE, row = lane % 16, sub = lane / 16;
    const uint32_t i0 = (KW > 1 ? blockIdx.y : blockIdx.y * (BLOCK / WAVE) + wv) * (16 * RT);
    const uint32_t j0 = blockIdx.x * (16 * CT);
    const uint32_t kc = (g.K + gridDim.z - 1) / gridDim.z;
    const uint32_t kb = min(g.K, blockIdx.z * kc), ke = min(g.K, kb + kc);
    if (KW == 1 && i0 >= g.M) return;
    f32x4 acc[RT][CT];
    float rs[RT];
    const bool sums = EPI == GEMM_STORE && g.rowsum && blockIdx.x == 0;
#pragma unroll
    for (int r = 0; r < RT; ++r) {
        rs[r] = 0.0f;
#pragma unroll
        for (int c = 0; c < CT; ++c) acc[r][c] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    auto load = [&](uint32_t k, f32x4(&a)[RT], f32x4(&b)[CT]) {
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            a[r] = fragment<float, AK>(g.A, g.sai, g.sap, min(i0 + 16 * r + row, g.M - 1), k + 4 * sub, ke);
            if (AK && g.asub) {
                const f32x4 s = fragment<float, true>(g.asub, 0, 1, 0, k + 4 * sub, ke);
                const f32x4 m = fragment<float, true>(g.amul, 0, 1, 0, k + 4 * sub, ke);
#pragma unroll
                for (int u = 0; u < 4; ++u) a[r][u] = (a[r][u] - s[u]) * m[u];
            }
        }
#pragma unroll
        for (int c = 0; c < CT; ++c)
            b[c] = fragment<TB, BK>(B, g.sbj, g.sbp, min(j0 + 16 * c + row, g.N - 1), k + 4 * sub, ke);
    };
    const uint32_t w = KW > 1 ? wv : 0u;
    f32x4 a[RT], b[CT];
    uint32_t k = kb + w * KSTEP;
    if (k < ke) load(k, a, b);
    while (k < ke) {
        const uint32_t kn = k + (KW > 1 ? KW : 1) * KSTEP;
        f32x4 an[RT], bn[CT];
        if (kn < ke) load(kn, an, bn);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int r = 0; r < RT; ++r)
#pragma unroll
                for (int c = 0; c < CT; ++c)
                    acc[r][c] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[r][u], b[c][u], acc[r][c], 0, 0, 0);
        if (sums) {
#pragma unroll
            for (int r = 0; r < RT; ++r) rs[r] += (a[r][0] + a[r][1]) + (a[r][2] + a[r][3]);
        }
#pragma unroll
        for (int r = 0; r < RT; ++r) a[r] = an[r];
#pragma unroll
        for (int c = 0; c < CT; ++c) b[c] = bn[c];
        k = kn;
    }
    auto finish = [&](uint32_t i, uint32_t j, float v) {
        if (i >= g.M || j >= g.N) return;
        if (gridDim.z > 1) {  // split K: partial of this slice
            g.part[((size_t)blockIdx.z * g.M + i) * g.N + j] = v;
            return;
        }
        const size_t o = (size_t)i * g.ldc + j;
        if constexpr (EPI == GEMM_STORE) {
            float z = g.bias ? v + ld<TB>(static_cast<const TB*>(g.bias), j) : v;
            if (g.csub) z = (z - g.csub[j]) * g.cmul[j];
            g.C[o] = z;
        } else if constexpr (EPI == GEMM_BIAS_GELU) {
            const float z = v + ld<TB>(static_cast<const TB*>(g.bias), j);
            if (g.C) g.C[o] = z;
            g.C2[o] = gelu(z);
        } else {  // GEMM_GELU_GRAD
            g.C[o] = v * gelu_grad(g.aux[o]);
        }
    };
    if constexpr (KW == 1) {
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
            for (int c = 0; c < CT; ++c)
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    finish(i0 + 16 * r + 4 * sub + q, j0 + 16 * c + row, acc[r][c][q]);
        return;
    }
    constexpr uint32_t PER = RT * CT * 4;  // values a lane holds
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int c = 0; c < CT; ++c)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                gemm_lds[(wv * PER + (r * CT + c) * 4 + q) * WAVE + lane] = acc[r][c][q];
    float* rsum = gemm_lds + KW * PER * WAVE;  // [KW][16 RT]
    if (sums) {
#pragma unroll
        for (int r = 0; r < RT; ++r) {
            rs[r] += __shfl_xor(rs[r], 16);
            rs[r] += __shfl_xor(rs[r], 32);
            if (sub == 0) rsum[wv * 16 * RT + 16 * r + row] = rs[r];
        }
    }
    __syncthreads();
    for (uint32_t e = threadIdx.x; e < PER * WAVE; e += KW * WAVE) {
        float v = 0.0f;
#pragma unroll
        for (uint32_t x = 0; x < KW; ++x) v += gemm_lds[x * PER * WAVE + e];
        const uint32_t ln = e % WAVE, t = e / WAVE;
        finish(i0 + 16 * (t / 4 / CT) + 4 * (ln / 16) + t % 4, j0 + 16 * (t / 4 % CT) + ln % 16, v);
    }
    if (sums && threadIdx.x < 16 * RT) {
        float v = 0.0f;
        for (uint32_t x = 0; x < KW; ++x) v += rsum[x * 16 * RT + threadIdx.x];
        const uint32_t i = i0 + threadIdx.x;
        if (i < g.M) {
            if (gridDim.z > 1) g.part[(size_t)gridDim.z * g.M * g.N + (size_t)blockIdx.z * g.M + i] = v;
            else g.rowsum[i] = v;
        }
    }
}

// C[i][j] = sum over slices z (in order) of part[z][i][j]; the row sums, if
// any, lie behind the slices
__global__ __launch_bounds__(BLOCK) void splitk_reduce_kernel(GemmArgs g, uint32_t slices) {
    const uint64_t total = (uint64_t)g.M * g.N;
    for (uint64_t q = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; q < total; q += (uint64_t)gridDim.x * BLOCK) {
        float s = 0.0f;
        for (uint32_t z = 0; z < slices; ++z) s += g.part[(size_t)z * total + q];
        g.C[(q / g.N) * g.ldc + q % g.N] = s;
    }
    if (!g.rowsum) return;
    for (uint64_t q = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; q < g.M; q += (uint64_t)gridDim.x * BLOCK) {
        float s = 0.0f;
        for (uint32_t z = 0; z < slices; ++z) s += g.part[(size_t)slices * total + (size_t)z * g.M + q];
        g.rowsum[q] = s;
    }
}

// dY = 2 (Y - T) / count; per-block FP64 sums of (Y - T)^2
__global__ __launch_bounds__(BLOCK) void mse_kernel(const float* __restrict__ Y, const float* __restrict__ T,
                                                    uint64_t count, float* __restrict__ dY, double* __restrict__ part) {
    __shared__ double sh[BLOCK];
    double s = 0.0;
    const float scale = 2.0f / (float)count;
    for (uint64_t q = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; q < count; q += (uint64_t)gridDim.x * BLOCK) {
        const float d = Y[q] - T[q];
        dY[q] = d * scale;
        s += (double)d * (double)d;
    }
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int off = BLOCK / 2; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) sh[threadIdx.x] += sh[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) part[blockIdx.x] = sh[0];
}

// *out = (sum of n <= MSE_PARTS partials) / count, one block
__global__ __launch_bounds__(BLOCK) void sum_parts_kernel(const double* __restrict__ part, uint32_t n, uint64_t count,
                                                          double* __restrict__ out) {
    __shared__ double sh[BLOCK];
    double s = 0.0;
    for (uint32_t q = threadIdx.x; q < n; q += BLOCK) s += part[q];
    sh[threadIdx.x] = s;
    __syncthreads();
    for (int off = BLOCK / 2; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) sh[threadIdx.x] += sh[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = sh[0] / (double)count;
}

__global__ __launch_bounds__(BLOCK) void adam_kernel(AdamArgs a) {
    for (uint64_t q = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; q < a.count; q += (uint64_t)gridDim.x * BLOCK) {
        const float g = a.grad[q];
        const float m = a.beta1 * a.m[q] + (1.0f - a.beta1) * g;
        const float v = a.beta2 * a.v[q] + (1.0f - a.beta2) * g * g;
        a.m[q] = m;
        a.v[q] = v;
        a.param[q] -= a.lr * (m / a.bc1) / (sqrtf(v / a.bc2) + a.eps);
    }
}

// Y[i][j] = (X[src_row(i)][j] - sub[j]) * mul[j]   (src_row: rows[i] or i)
__global__ __launch_bounds__(BLOCK) void affine_rows_kernel(const float* __restrict__ X, const uint32_t* __restrict__ rows,
                                                            uint32_t M, uint32_t N, const float* __restrict__ sub,
                                                            const float* __restrict__ mul, float* __restrict__ Y) {
    const uint64_t total = (uint64_t)M * N;
    for (uint64_t q = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; q < total; q += (uint64_t)gridDim.x * BLOCK) {
        const uint64_t i = q / N, j = q % N;
        const uint64_t si = rows ? rows[i] : i;
        const float x = X[si * N + j];
        Y[q] = sub ? (x - sub[j]) * mul[j] : x;
    }
}

uint32_t grid_for(uint64_t count) {
    uint64_t b = (count + BLOCK - 1) / BLOCK;
    if (b > 8192) b = 8192;
    return (uint32_t)(b ? b : 1);
}

}  // namespace

namespace {

template <class TB, bool AK, bool BK, int EPI, int RT, int CT, int KW>
hipError_t gemm_run(const GemmArgs& g, const TB* B, uint32_t slices, hipStream_t s) {
    const uint32_t rows = 16 * RT * (KW > 1 ? 1 : BLOCK / WAVE);
    const dim3 grid((g.N + 16 * CT - 1) / (16 * CT), (g.M + rows - 1) / rows, slices);
    if (grid.y > 65535u) return hipErrorInvalidValue;
    const size_t lds = KW > 1 ? sizeof(float) * KW * (RT * CT * 4 * WAVE + 16 * RT) : 0;
    hipLaunchKernelGGL((gemm_kernel<TB, AK, BK, EPI, RT, CT, KW>), grid, dim3(KW > 1 ? KW * WAVE : BLOCK), lds, s, g, B);
    return hipGetLastError();
}

// 64 x 64 outputs a wave where that leaves every SIMD one (1,024); else 32 x
// 32 shared by the four waves of a block, or, for a long K (a weight
// gradient over a minibatch), by 16.  1,024 x 256 x 256: 46 -> 8 us; 48,019
// x 256 x 256: 190 us in three chunks -> 89 us in one launch.
template <class TB, bool AK, bool BK, int EPI>
hipError_t gemm_pick(const GemmArgs& g, const TB* B, hipStream_t s) {
    const uint64_t t64 = (uint64_t)((g.M + 63) / 64) * ((g.N + 63) / 64);
    if (t64 >= 1024 && !g.rowsum) return gemm_run<TB, AK, BK, EPI, 4, 4, 1>(g, B, 1, s);
    if constexpr (EPI == GEMM_STORE && !AK) {
        if (g.K >= 512) {
            // further slices of K while each keeps 2,048 values and the chip has room
            const uint64_t t32 = (uint64_t)((g.M + 31) / 32) * ((g.N + 31) / 32);
            uint64_t slices = 1;
            if (g.part) {
                slices = std::min<uint64_t>(std::min<uint64_t>(g.K / 2048u, 512u / t32),
                                            g.part_cap / ((uint64_t)g.M * (g.N + 1)));
                slices = std::max<uint64_t>(std::min<uint64_t>(slices, 16u), 1u);
            }
            const hipError_t e = gemm_run<TB, AK, BK, EPI, 2, 2, 16>(g, B, (uint32_t)slices, s);
            if (e != hipSuccess || slices == 1) return e;
            hipLaunchKernelGGL(splitk_reduce_kernel, dim3(grid_for((uint64_t)g.M * g.N)), dim3(BLOCK), 0, s, g,
                               (uint32_t)slices);
            return hipGetLastError();
        }
    }
    return gemm_run<TB, AK, BK, EPI, 2, 2, 4>(g, B, 1, s);
}

}  // namespace

hipError_t launch_gemm(const GemmArgs& g, const void* B, bool bf16_b, int epi, hipStream_t s) {
    if (g.M == 0 || g.N == 0) return hipSuccess;
    const float* F = static_cast<const float*>(B);
    // the products the network makes: K is the unit stride of both operands
    // (forward), of the left one (gradient of a layer's input) or of neither
    // (weight gradient, with row sums)
    if (bf16_b) {
        const bf16* H = static_cast<const bf16*>(B);
        if (g.sap != 1 || g.sbp != 1 || g.rowsum) return hipErrorInvalidValue;
        if (epi == GEMM_STORE) return gemm_pick<bf16, true, true, GEMM_STORE>(g, H, s);
        if (epi == GEMM_BIAS_GELU) return gemm_pick<bf16, true, true, GEMM_BIAS_GELU>(g, H, s);
        return hipErrorInvalidValue;
    }
    if (g.rowsum) return epi == GEMM_STORE ? gemm_pick<float, false, false, GEMM_STORE>(g, F, s) : hipErrorInvalidValue;
    if (g.sap != 1) return hipErrorInvalidValue;
    if (epi == GEMM_GELU_GRAD) return gemm_pick<float, true, false, GEMM_GELU_GRAD>(g, F, s);
    if (g.sbp != 1) return hipErrorInvalidValue;
    if (epi == GEMM_STORE) return gemm_pick<float, true, true, GEMM_STORE>(g, F, s);
    if (epi == GEMM_BIAS_GELU) return gemm_pick<float, true, true, GEMM_BIAS_GELU>(g, F, s);
    return hipErrorInvalidValue;
}

hipError_t launch_mse(const float* Y, const float* T, uint64_t count, float* dY, double* part, double* out,
                      hipStream_t s) {
    if (count == 0) return hipSuccess;
    uint32_t g = grid_for(count);
    if (g > MSE_PARTS) g = MSE_PARTS;
    hipLaunchKernelGGL(mse_kernel, dim3(g), dim3(BLOCK), 0, s, Y, T, count, dY, part);
    hipLaunchKernelGGL(sum_parts_kernel, dim3(1), dim3(BLOCK), 0, s, part, g, count, out);
    return hipGetLastError();
}

hipError_t launch_adam(const AdamArgs& a, hipStream_t s) {
    if (a.count == 0) return hipSuccess;
    hipLaunchKernelGGL(adam_kernel, dim3(grid_for(a.count)), dim3(BLOCK), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_affine_rows(const float* X, const uint32_t* rows, uint32_t M, uint32_t N, const float* sub,
                              const float* mul, float* Y, hipStream_t s) {
    const uint64_t total = (uint64_t)M * N;
    if (total == 0) return hipSuccess;
    hipLaunchKernelGGL(affine_rows_kernel, dim3(grid_for(total)), dim3(BLOCK), 0, s, X, rows, M, N, sub, mul, Y);
    return hipGetLastError();
}

}  // namespace ccd
