// Fold-in of new rows against fixed item factors H (the learned warm-start
// extension; the reference has no fold-in).  Folding in a row is CCD++ with
// the item side frozen: per sweep and rank t,
//   a = r^ + w_t h_t,  w_t = sum a h_t / (lambda |row| + sum h_t^2),  r^ = a - w_t h_t
// (the u-side update of src/cdmf_ref.cpp:7-17 on one row).
//
// computed on the row's normal equations (below).  The features and the
// sweeps take a launch for the long rows, listed by the host, and one for
// the others.  Per-row sums are reduced in a fixed order: deterministic.
#include "ccd_kernels.h"

#include <algorithm>

namespace ccd {

// old with lane `lane` (constant) replaced by the uniform x: the compiler's
// own lane write, which it keeps two wait states behind the lane read that x
// comes from.  (It does not look into inline assembly.)
__device__ int write_lane(int x, int lane, int old) __asm("llvm.amdgcn.writelane.i32");

namespace {

constexpr int WAVE = 64;
constexpr int BLOCK = 256;
constexpr int LBLOCK = 1024;
constexpr int LWAVES = LBLOCK / WAVE;
constexpr int FEAT_U = 32;   // H-row loads in flight per feature step
// Feature sums of a row's elements s .. e - 1 for rank t, over the chunks
// of 64 elements c0, c0 + cstep, ...: S = sum r, m = sum r h, v = sum r h^2
// (FP64, in element order within each chunk, chunks in order).  A chunk's
// ratings and indices come in with one coalesced, non-temporal load each
// (so that they do not push the item rows of HT, reread for every rating
// of the item, out of L2); each element's index and rating are then read
// from its lane (v_readlane) and the H rows of 32 elements are loaded
// together.  Lanes past k load rank 0's entry and drop it, so there is no
// branch around the loads.
__device__ __forceinline__ void feature_sums(const FoldArgs& a, uint32_t s, uint32_t e, uint32_t c0, uint32_t cstep,
                                             uint32_t t, bool tok, double& S, double& m, double& v) {
    const uint32_t tt = tok ? t : 0u;
    const int lane = threadIdx.x & (WAVE - 1);
    for (uint32_t base = s + c0 * WAVE; base < e; base += cstep * WAVE) {
        const uint32_t p = base + (uint32_t)lane;
        const bool okp = p < e;
        const uint32_t cv = okp ? __builtin_nontemporal_load(a.idx + p) : 0u;
        const float rv = okp ? __builtin_nontemporal_load(a.val + p) : 0.0f;
        const uint32_t n = e - base < (uint32_t)WAVE ? e - base : (uint32_t)WAVE;
#pragma unroll
        for (int half = 0; half < WAVE / FEAT_U; ++half) {
            if ((uint32_t)(FEAT_U * half) >= n) break;
            float h[FEAT_U];
#pragma unroll
            for (int u = 0; u < FEAT_U; ++u) {
                const uint32_t c = (uint32_t)__builtin_amdgcn_readlane((int)cv, FEAT_U * half + u);
                h[u] = a.HT[(size_t)c * a.ld + tt];
            }
#pragma unroll
            for (int u = 0; u < FEAT_U; ++u) {
                if ((uint32_t)(FEAT_U * half + u) < n) {
                    const float r = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(rv), FEAT_U * half + u));
                    const float hu = tok ? h[u] : 0.0f;
                    S += r;
                    m += (double)r * hu;
                    v += (double)r * hu * hu;
                }
            }
        }
    }
}

// mean = m / S and variance = v / S - mean^2 (FP64, one pass), 0 for an
// empty row or zero rating sum
__device__ __forceinline__ void write_features(float* f, uint32_t k, uint32_t t, bool tok, uint32_t d, double S,
                                               double m, double v) {
    if (!tok) return;
    double mean = 0.0, var = 0.0;
    if (d && S != 0.0) {
        mean = m / S;
        var = v / S - mean * mean;
        if (var < 0.0) var = 0.0;
    }
    f[t] = (float)mean;
    f[k + t] = (float)var;
}

// F [rows][2k + 2] of the long rows (more than FOLD_SHORT ratings), one
// 1024-thread block each: lanes take ranks t0 + lane, the row's elements are
// dealt to the 16 waves and the per-wave sums added in wave order.
__global__ __launch_bounds__(LBLOCK) void fold_features_long_kernel(FoldArgs a, const uint32_t* __restrict__ long_rows,
                                                                    float* __restrict__ F) {
    __shared__ double part[3][LWAVES][WAVE];
    const int lane = threadIdx.x & (WAVE - 1), wv = threadIdx.x / WAVE;
    const uint32_t k = a.k;
    const uint32_t row = long_rows[blockIdx.x];
    const uint32_t s = a.ptr[row], e = a.ptr[row + 1], d = e - s;
    float* f = F + (size_t)row * (2 * k + 2);
    double Sr = 0.0;
    for (uint32_t t0 = 0; t0 < k; t0 += WAVE) {
        const uint32_t t = t0 + lane;
        const bool tok = t < k;
        double S = 0.0, m = 0.0, v = 0.0;
        feature_sums(a, s, e, (uint32_t)wv, LWAVES, t, tok, S, m, v);  // wave wv: chunks wv, wv + 16, ...
        part[0][wv][lane] = S;
        part[1][wv][lane] = m;
        part[2][wv][lane] = v;
        __syncthreads();
        if (wv == 0) {
            double St = 0.0, mt = 0.0, vt = 0.0;
            for (int w = 0; w < LWAVES; ++w) {
                St += part[0][w][lane];
                mt += part[1][w][lane];
                vt += part[2][w][lane];
            }
            write_features(f, k, t, tok, d, St, mt, vt);
            Sr = St;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) {
        f[2 * k] = (float)log1p((double)d);
        f[2 * k + 1] = d ? (float)(Sr / d) : 0.0f;
    }
}

// F of the other rows, one single-wave block per row (so a wave that
// finishes a short row frees its slot at once, whatever the lengths of
// its neighbours): lanes take ranks t0 + lane and walk the row's elements
// in order, FEAT_U loads in flight (feature_sums).
__global__ __launch_bounds__(WAVE) void fold_features_short_kernel(FoldArgs a, float* __restrict__ F) {
    const int lane = threadIdx.x;
    const uint32_t k = a.k;
    const uint32_t row = blockIdx.x;
    const uint32_t s = a.ptr[row], e = a.ptr[row + 1], d = e - s;
    if (d > FOLD_SHORT) return;
    float* f = F + (size_t)row * (2 * k + 2);
    double Sr = 0.0;
    for (uint32_t t0 = 0; t0 < k; t0 += WAVE) {
        const uint32_t t = t0 + lane;
        const bool tok = t < k;
        double S = 0.0, m = 0.0, v = 0.0;
        feature_sums(a, s, e, 0, 1, t, tok, S, m, v);
        write_features(f, k, t, tok, d, S, m, v);
        Sr = S;
    }
    if (lane == 0) {
        f[2 * k] = (float)log1p((double)d);
        f[2 * k + 1] = d ? (float)(Sr / d) : 0.0f;
    }
}

// ------------------------------------------------------------ sweeps ---
// The sweeps work on a row's normal equations G = H_O^T H_O (k x k) and
// b = H_O^T r: in exact arithmetic the update of rank t,
//   w_t = (b_t - sum_{s != t} G_ts w_s) / (lambda |O| + G_tt),
// is the one over the row's residual, but a sweep costs k^2 operations on
// one wave instead of |O| k gathers.  Everything is FP64 from the products
// on, so the result is closer to the exact sweeps than an FP32 residual
// carried through them (2.5e-8, the final
// rounding, against 6e-7 relative on the shapes below).
//
// G comes from the FP64 matrix cores, v_mfma_f64_16x16x4_f64: four ratings a
// step, NT = ceil(k / 16) loads of 16 consecutive entries of an item's HT
// row per rating, each of them both operands of its tile pairs (upper
// triangle only).  Operand layout: lane l supplies A[l % 16][l / 16] and
// B[l / 16][l % 16] and receives D[4 q + l / 16][l % 16], q = 0..3.
// NT (NT + 1) / 2 pairs of 64 cycles per four ratings bound this part.
//
// The sweep keeps e_s = (numerator_s) / (denominator_s) - w_s on lane s: rank
// t's change D is e_t, and e_s -= (G_st / denominator_s) D for every s.  One
// step is one cross-lane read of e_t and one FMA (the scaled matrix comes
// from LDS, a column per lane, ahead of time), and the k steps of a sweep
// are a serial chain: its latency (about 60 cycles a step) bounds one row,
// its issue slots (about 27) a batch of short ones.
//
// One row of 206 ratings, k = 40, 20 sweeps: 679 -> 29 us; 48,019 rows with
// 9.9M ratings: 23.6 -> 1.4 ms (7 sweeps 9.1 -> 1.1 ms), against the same
// sweeps over the FP32 residual in registers.
using f64x4 = __attribute__((__vector_size__(4 * sizeof(double)))) double;
constexpr int GSTEP = 4;          // steps of four ratings whose loads are in flight together
constexpr int GRAM_PAIRS = 12;    // tile pairs a wave accumulates at once (96 registers)

constexpr int pair_count(int nt) { return nt * (nt + 1) / 2; }
// tile pair p of the upper triangle, row by row
constexpr int pair_row(int nt, int p) {
    int r = 0;
    while (p >= nt - r) p -= nt - r++;
    return r;
}
constexpr int pair_col(int nt, int p) {
    int r = 0;
    while (p >= nt - r) p -= nt - r++;
    return r + p;
}

// entries of G in LDS: rows of 16 NT, whole groups of the chain
constexpr int CHAIN = 8;
__host__ __device__ constexpr uint32_t fold_matrix(int nt, uint32_t k) { return 16u * nt * ((k + CHAIN - 1) / CHAIN * CHAIN); }

template <int NT, int P0, int P, int I = 0>
__device__ __forceinline__ void gram_mfma(const double (&h)[NT], f64x4 (&acc)[P]) {
    if constexpr (I < P) {
        constexpr int ti = pair_row(NT, P0 + I), tj = pair_col(NT, P0 + I);
        acc[I] = __builtin_amdgcn_mfma_f64_16x16x4f64(h[ti], h[tj], acc[I], 0, 0, 0);
        gram_mfma<NT, P0, P, I + 1>(h, acc);
    }
}

template <int NT, int P0, int P, int I = 0>
__device__ __forceinline__ void gram_store(const f64x4 (&acc)[P], double* G, uint32_t k, int lane, bool first) {
    if constexpr (I < P) {
        constexpr int LD = 16 * NT;
        constexpr int ti = pair_row(NT, P0 + I), tj = pair_col(NT, P0 + I);
        const uint32_t c = 16 * tj + lane % 16;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t r = 16 * ti + 4 * q + lane / 16;
            if (r < k && c < k) {
                const double v = first ? acc[I][q] : G[r * LD + c] + acc[I][q];
                G[r * LD + c] = v;
                if (ti != tj) G[c * LD + r] = v;
            }
        }
        gram_store<NT, P0, P, I + 1>(acc, G, k, lane, first);
    }
}

// G (k x k, rows of 16 NT) and b (k) in LDS of the ratings s .. s + d - 1, by the NW waves of
// the block: wave wv takes chunks wv, wv + NW, ... of 64 ratings, and the
// waves' sums are added in wave order.  Ends with every wave's part stored
// (the caller synchronises).  P0, P1: the tile pairs to form (b comes with
// pair 0).
template <int NT, int NW, int P0 = 0, int P1 = pair_count(NT)>
__device__ __forceinline__ void gram(const FoldArgs& a, uint32_t s, uint32_t d, double* G, double* b) {
    constexpr int P = P1 - P0 < GRAM_PAIRS ? P1 - P0 : GRAM_PAIRS;
    const int lane = threadIdx.x & (WAVE - 1);
    const uint32_t wv = NW == 1 ? 0u : (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const uint32_t k = a.k, sub = lane / 16, col = lane % 16;
    f64x4 acc[P];
    double bacc[NT];
#pragma unroll
    for (int i = 0; i < P; ++i) acc[i] = f64x4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int t = 0; t < NT; ++t) bacc[t] = 0.0;
    for (uint32_t c0 = wv * WAVE; c0 < d; c0 += NW * WAVE) {
        const uint32_t p = c0 + lane;
        const uint32_t cv = p < d ? __builtin_nontemporal_load(a.idx + s + p) : a.n;  // row n of HT is zero
        const float rv = p < d ? __builtin_nontemporal_load(a.val + s + p) : 0.0f;
        const uint32_t n = d - c0 < (uint32_t)WAVE ? d - c0 : (uint32_t)WAVE;
        for (uint32_t j = 0; 4 * j < n; j += GSTEP) {
            float h[GSTEP][NT];
#pragma unroll
            for (int u = 0; u < GSTEP; ++u) {
                const uint32_t c = (uint32_t)__shfl((int)cv, (int)(4 * (j + u) + sub));
                const float* hr = a.HT + (size_t)c * a.ld + col;
#pragma unroll
                for (int t = 0; t < NT; ++t) h[u][t] = hr[16 * t];
            }
#pragma unroll
            for (int u = 0; u < GSTEP; ++u) {
                double hd[NT];
#pragma unroll
                for (int t = 0; t < NT; ++t) hd[t] = (double)h[u][t];
                if constexpr (P0 == 0) {
                    const double r = (double)__shfl(rv, (int)(4 * (j + u) + sub));
#pragma unroll
                    for (int t = 0; t < NT; ++t) bacc[t] = __builtin_fma(r, hd[t], bacc[t]);
                }
                gram_mfma<NT, P0, P>(hd, acc);
            }
        }
    }
    const uint32_t parts = NW == 1 ? 1u : min((uint32_t)NW, (d + WAVE - 1) / WAVE);
    if constexpr (P0 == 0) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            bacc[t] += __shfl_xor(bacc[t], 16);
            bacc[t] += __shfl_xor(bacc[t], 32);
        }
    }
    for (uint32_t w = 0; w < parts; ++w) {
        if (w == wv) {
            gram_store<NT, P0, P>(acc, G, k, lane, w == 0);
            if constexpr (P0 == 0) {
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    const uint32_t i = 16 * t + col;
                    if (sub == 0 && i < k) b[i] = w == 0 ? bacc[t] : b[i] + bacc[t];
                }
            }
        }
        if (NW > 1) __syncthreads();
    }
    if constexpr (P0 + P < P1) gram<NT, NW, P0 + P, P1>(a, s, d, G, b);
}

// The same by SW waves that share the tile pairs, each over all ratings (the
// sums are those of one wave).
template <int NT, int SW, int W = 0>
__device__ __forceinline__ void gram_by_pairs(const FoldArgs& a, uint32_t s, uint32_t d, double* G, double* b,
                                              uint32_t wv) {
    constexpr int PALL = pair_count(NT), PER = (PALL + SW - 1) / SW;
    if (wv == (uint32_t)W) gram<NT, 1, PER * W, (PER * W + PER < PALL ? PER * W + PER : PALL)>(a, s, d, G, b);
    else if constexpr (W + 1 < SW) gram_by_pairs<NT, SW, W + 1>(a, s, d, G, b, wv);
}

__device__ __forceinline__ double lane_value(double v, int lane) {
    const long long x = __double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, lane);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)((unsigned long long)x >> 32), lane);
    return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}

// old with lane LANE replaced by the uniform x
template <int LANE>
__device__ __forceinline__ double with_lane(double old, double x) {
    const unsigned long long a = (unsigned long long)__double_as_longlong(old);
    const unsigned long long b = (unsigned long long)__double_as_longlong(x);
    const uint32_t lo = (uint32_t)write_lane((int)(uint32_t)b, LANE, (int)(uint32_t)a);
    const uint32_t hi = (uint32_t)write_lane((int)(uint32_t)(b >> 32), LANE, (int)(uint32_t)(a >> 32));
    return __longlong_as_double((long long)((unsigned long long)hi << 32 | lo));
}

template <int NS, int J, int L0, int U = 0>
__device__ __forceinline__ void fold_steps(const double (&g)[NS][CHAIN], double (&e)[NS], double& cap) {
    if constexpr (U < CHAIN) {
        const double D = lane_value(e[J], L0 + U);
        cap = with_lane<L0 + U>(cap, D);
#pragma unroll
        for (int j = 0; j < NS; ++j) e[j] = __builtin_fma(-g[j][U], D, e[j]);
        fold_steps<NS, J, L0, U + 1>(g, e, cap);
    }
}

// The chain over ranks 64 J + 8 Q .. of the matrix at m (row 64 J, this
// lane's column of slot 0), group by group; LD: row length in LDS.  Lane and
// row offsets are constants, so a step is two reads and two writes of a lane
// and one FMA per slot.
template <int NS, int J, int LD, int Q = 0>
__device__ __forceinline__ void fold_chain(const double* m, uint32_t groups, const double (&g)[NS][CHAIN],
                                           double (&e)[NS], double& cap) {
    if ((uint32_t)Q >= groups) return;
    // the next group's entries, read ahead of this group's chain
    double gn[NS][CHAIN];
    constexpr int QN = Q + 1 < WAVE / CHAIN ? Q + 1 : 0;
    const double* mn = m + ((uint32_t)QN < groups ? QN * CHAIN * LD : 0);
#pragma unroll
    for (int j = 0; j < NS; ++j)
#pragma unroll
        for (int u = 0; u < CHAIN; ++u) gn[j][u] = mn[u * LD + WAVE * j];
    fold_steps<NS, J, Q * CHAIN>(g, e, cap);
    if constexpr (Q + 1 < WAVE / CHAIN) fold_chain<NS, J, LD, Q + 1>(m, groups, gn, e, cap);
}

// The sweeps of one row from its G and b in LDS, by the first of the SW waves
// that call (the others help to scale G): lane l holds ranks l and, for k >
// 64 (NS = 2), l + 64.  Column s of G is only touched by
// rank s's lane, which scales it in place.  The chain runs in whole groups:
// columns k .. of G, which the products leave unwritten, and rows k .. up to
// a multiple of CHAIN are cleared, so the ranks there stay zero.
template <int NS, int LD, int SW = 1>
__device__ __forceinline__ void fold_solve(const FoldArgs& a, uint32_t row, uint32_t d, double* G, const double* b,
                                           const float* __restrict__ W0, float* __restrict__ W) {
    const uint32_t lane = threadIdx.x & (WAVE - 1), k = a.k;
    const uint32_t wv = SW == 1 ? 0u : (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const double lamd = (double)(a.lambda * (float)d);
    double e[NS], w[NS], scale[NS];
    bool lost = false;
    // Lanes past the matrix hold no rank: their e is never read by a step nor
    // stored, so what the chain gathers for them does not matter, only that
    // it lies in the block's LDS.  With one slot they read column 0; a second
    // slot of lanes from LD - 64 on reads past its row, in the last row up to
    // 128 - LD entries into b.
    static_assert(NS == 1 || WAVE * NS - LD <= LD - 15, "b has more than LD - 16 entries");
    const double* base = G + (lane < (uint32_t)LD ? lane : 0u);
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        const uint32_t s = lane + WAVE * j;
        e[j] = 0.0;
        w[j] = 0.0;
        scale[j] = 0.0;
        if (s < k) {
            double* col = G + s;
            const double sq = col[s * LD];
            lost = lost || !(sq - sq == 0.0);
            scale[j] = 1.0 / (lamd + sq);
            if (wv == 0) {
                w[j] = W0 ? (double)W0[(size_t)row * k + s] : 0.0;
                double p = b[s];
                if (W0) {  // the numerator leaves the rank's own term out
                    for (uint32_t u = 0; u < k; ++u) {
                        const double wu = (double)W0[(size_t)row * k + u];
                        if (u != s) p = __builtin_fma(-col[u * LD], wu, p);
                    }
                }
                e[j] = __builtin_fma(p, scale[j], -w[j]);
            }
        }
    }
    // A rated item with a factor that is not finite (its square stands on the
    // diagonal): from zero the row's residual starts as r - 0 h, no number, and
    // every rank sums over it, the ones before that factor's too.
    if (!W0 && __any(lost)) {
#pragma unroll
        for (int j = 0; j < NS; ++j) e[j] = __builtin_nan("");
    }
    if (SW > 1) __syncthreads();  // the diagonal and the numerators are read
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        const uint32_t s = lane + WAVE * j;
        if (s < (uint32_t)LD) {
#pragma unroll 4
            for (uint32_t u = wv; u < k; u += SW) {
                const double v = G[u * LD + s] * scale[j];
                G[u * LD + s] = s >= k ? 0.0 : u == s ? 1.0 : v;
            }
            if (wv == 0)
                for (uint32_t u = k; u % CHAIN; ++u) G[u * LD + s] = 0.0;
        }
    }
    if (SW > 1) {
        __syncthreads();
        if (wv) return;
    }
    // one wave: its LDS writes above come before its reads below
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (int sw = 0; sw < a.sweeps; ++sw) {
        double g[NS][CHAIN], cap = 0.0;
        auto first = [&](const double* m) {
#pragma unroll
            for (int j = 0; j < NS; ++j)
#pragma unroll
                for (int u = 0; u < CHAIN; ++u) g[j][u] = m[u * LD + WAVE * j];
        };
        first(base);
        fold_chain<NS, 0, LD>(base, (min(k, (uint32_t)WAVE) + CHAIN - 1) / CHAIN, g, e, cap);
        w[0] += cap;
        if constexpr (NS == 2) {
            const double* m = base + WAVE * LD;
            cap = 0.0;
            first(m);
            fold_chain<NS, 1, LD>(m, (k - WAVE + CHAIN - 1) / CHAIN, g, e, cap);
            w[1] += cap;
        }
    }
#pragma unroll
    for (int j = 0; j < NS; ++j) {
        const uint32_t s = lane + WAVE * j;
        if (s < k) W[(size_t)row * k + s] = (float)w[j];
    }
}

// Rows of more than FOLD_WAVE ratings: one block each, in the order of the
// host's list (longest first, so the last blocks to run are short).  The
// waves share the products; the first one then runs the sweeps while the
// others' slots go to the next block.
constexpr int FOLD_LWAVES = 8;
template <int NT>
__global__ __launch_bounds__(FOLD_LWAVES* WAVE) void fold_sweep_long_kernel(FoldArgs a,
                                                                           const uint32_t* __restrict__ long_rows,
                                                                           const float* __restrict__ W0,
                                                                           float* __restrict__ W) {
    extern __shared__ __align__(16) double fold_lds[];  // G, then b
    double* b = fold_lds + fold_matrix(NT, a.k);
    const uint32_t row = long_rows[blockIdx.x];
    const uint32_t s = a.ptr[row], d = a.ptr[row + 1] - s;
    gram<NT, FOLD_LWAVES>(a, s, d, fold_lds, b);
    if (threadIdx.x >= WAVE) return;
    fold_solve<(NT > 4 ? 2 : 1), 16 * NT>(a, row, d, fold_lds, b, W0, W);
}

// The other rows, one block each: a single wave up to k = 64.  Past that the
// matrix (46 to 131 KB) leaves a CU room for three rows down to one, so four
// waves, or from k = 97 one for each 16 ranks, share a row's products and
// scaling.  With one wave a sweep or two over short rows took longer than
// over the row's residual: 48,019 rows of 5 ratings, k = 128, one sweep 4.8
// ms (residual 2.5, now 2.0); of 100 ratings, k = 100, 8.6 (3.0, 2.9), k =
// 65, 2.05 (1.97, 1.23).
constexpr int short_waves(int nt) { return nt > 6 ? nt : nt > 4 ? 4 : 1; }
template <int NT>
__global__ __launch_bounds__(short_waves(NT)* WAVE) void fold_sweep_short_kernel(FoldArgs a,
                                                                                const float* __restrict__ W0,
                                                                                float* __restrict__ W) {
    constexpr int SW = short_waves(NT);
    extern __shared__ __align__(16) double fold_lds[];
    double* b = fold_lds + fold_matrix(NT, a.k);
    const uint32_t row = blockIdx.y * gridDim.x + blockIdx.x;
    if (row >= a.rows) return;
    const uint32_t s = a.ptr[row], d = a.ptr[row + 1] - s;
    if (d > FOLD_WAVE) return;
    if (d == 0 || a.sweeps == 0) {  // nothing to solve: 0 after a sweep, the start before one
        for (uint32_t t = threadIdx.x; t < a.k; t += SW * WAVE)
            W[(size_t)row * a.k + t] = a.sweeps == 0 && W0 ? W0[(size_t)row * a.k + t] : 0.0f;
        return;
    }
    const uint32_t wv = SW == 1 ? 0u : (uint32_t)__builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    gram_by_pairs<NT, SW>(a, s, d, fold_lds, b, wv);
    __syncthreads();
    fold_solve<(NT > 4 ? 2 : 1), 16 * NT, SW>(a, row, d, fold_lds, b, W0, W);
}

template <int NT>
hipError_t launch_sweeps_nt(const FoldArgs& a, const uint32_t* long_rows, uint32_t nlong, const float* W0, float* W,
                            hipStream_t s) {
    const size_t lds = sizeof(double) * (fold_matrix(NT, a.k) + a.k);
    if (nlong)
        hipLaunchKernelGGL(fold_sweep_long_kernel<NT>, dim3(nlong), dim3(FOLD_LWAVES * WAVE), lds, s, a, long_rows, W0,
                           W);
    if (nlong < a.rows) {
        const uint32_t x = std::min(a.rows, 1u << 20);  // a launch takes less than 2^32 threads along x
        hipLaunchKernelGGL(fold_sweep_short_kernel<NT>, dim3(x, (a.rows + x - 1) / x), dim3(short_waves(NT) * WAVE), lds,
                           s, a, W0, W);
    }
    return hipGetLastError();
}

__global__ __launch_bounds__(BLOCK) void transpose_kernel(const float* __restrict__ src, float* __restrict__ dst,
                                                          uint32_t rows, uint32_t cols, uint32_t ld) {
    const uint64_t total = (uint64_t)rows * cols;
    for (uint64_t q = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; q < total; q += (uint64_t)gridDim.x * BLOCK) {
        const uint64_t r = q / cols, c = q % cols;
        dst[c * ld + r] = src[q];
    }
}

}  // namespace

hipError_t launch_fold_features(const FoldArgs& a, const uint32_t* long_rows, uint32_t nlong, float* F,
                                hipStream_t s) {
    if (a.rows == 0) return hipSuccess;
    if (a.k > (uint32_t)FOLD_KMAX) return hipErrorInvalidValue;
    if (nlong) hipLaunchKernelGGL(fold_features_long_kernel, dim3(nlong), dim3(LBLOCK), 0, s, a, long_rows, F);
    hipLaunchKernelGGL(fold_features_short_kernel, dim3(a.rows), dim3(WAVE), 0, s, a, F);
    return hipGetLastError();
}

hipError_t launch_fold_sweeps(const FoldArgs& a, const uint32_t* long_rows, uint32_t nlong, const float* W0, float* W,
                              hipStream_t s) {
    if (a.rows == 0) return hipSuccess;
    switch ((a.k + 15) / 16) {
        case 1: return launch_sweeps_nt<1>(a, long_rows, nlong, W0, W, s);
        case 2: return launch_sweeps_nt<2>(a, long_rows, nlong, W0, W, s);
        case 3: return launch_sweeps_nt<3>(a, long_rows, nlong, W0, W, s);
        case 4: return launch_sweeps_nt<4>(a, long_rows, nlong, W0, W, s);
        case 5: return launch_sweeps_nt<5>(a, long_rows, nlong, W0, W, s);
        case 6: return launch_sweeps_nt<6>(a, long_rows, nlong, W0, W, s);
        case 7: return launch_sweeps_nt<7>(a, long_rows, nlong, W0, W, s);
        case 8: return launch_sweeps_nt<8>(a, long_rows, nlong, W0, W, s);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_transpose(const float* src, float* dst, uint32_t rows, uint32_t cols, uint32_t ld, hipStream_t s) {
    const uint64_t total = (uint64_t)rows * cols;
    if (total == 0) return hipSuccess;
    uint64_t g = (total + BLOCK - 1) / BLOCK;
    if (g > 8192) g = 8192;
    hipLaunchKernelGGL(transpose_kernel, dim3((uint32_t)g), dim3(BLOCK), 0, s, src, dst, rows, cols, ld);
    return hipGetLastError();
}

}  // namespace ccd
