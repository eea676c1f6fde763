// Set-up kernels of a solver context: the caller's numbering to the internal
// one and back.  Factors, residual and index arrays cross the ABI in the
// caller's order; the permutations, the renumbering of both compressed
// copies and the sort inside each row run here, so that a set-up call costs
// its copies over PCIe and little else.
#include "layout.h"

#include "ccd_kernels.h"

#include <algorithm>

namespace ccd {
namespace {

constexpr int WAVE = 64;
constexpr int BLOCK = 256;
constexpr uint32_t RANKS_PER_BLOCK = 8;  // ranks a block of permute_ranks_kernel walks

// Rank-major [k][rows] factors between the caller's numbering and the
// internal one (perm: internal -> caller's).  Bound by the random side, 4 B
// an entry out of one rank's row (at most a few MB, so L2 serves it); the
// other side and perm are coalesced, and perm is read once for
// RANKS_PER_BLOCK ranks.
template <bool TO_INTERNAL>
__global__ __launch_bounds__(BLOCK) void permute_ranks_kernel(const float* __restrict__ src, float* __restrict__ dst,
                                                              const uint32_t* __restrict__ perm, uint32_t k,
                                                              uint64_t rows) {
    const uint64_t i = (uint64_t)blockIdx.x * BLOCK + threadIdx.x;
    if (i >= rows) return;
    const uint64_t r = perm[i];
    for (uint32_t t0 = blockIdx.y * RANKS_PER_BLOCK; t0 < k; t0 += gridDim.y * RANKS_PER_BLOCK) {
        const uint32_t t1 = min(k, t0 + RANKS_PER_BLOCK);
#pragma unroll 8
        for (uint32_t t = t0; t < t1; ++t) {
            if (TO_INTERNAL) dst[t * rows + i] = src[t * rows + r];
            else dst[t * rows + r] = src[t * rows + i];
        }
    }
}

// dst[map[e]] = src[e]
__global__ __launch_bounds__(BLOCK) void scatter_kernel(const float* __restrict__ src,
                                                        const uint32_t* __restrict__ map, float* __restrict__ dst,
                                                        uint64_t count) {
    const uint64_t stride = (uint64_t)gridDim.x * BLOCK;
    for (uint64_t e = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; e < count; e += stride) dst[map[e]] = src[e];
}

__global__ __launch_bounds__(BLOCK) void index_check_kernel(const uint32_t* __restrict__ idx, uint64_t count,
                                                            uint32_t dim, uint32_t* __restrict__ bad) {
    const uint64_t stride = (uint64_t)gridDim.x * BLOCK;
    bool b = false;
    for (uint64_t e = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; e < count; e += stride) b |= idx[e] >= dim;
    if (b) atomicOr(bad, 1u);
}

template <typename IdxT>
__device__ __forceinline__ void put(const RenumArgs& a, uint32_t o, uint32_t key, uint32_t e) {
    static_cast<IdxT*>(a.oidx)[o] = (IdxT)key;
    a.oval[o] = a.val[e];
    a.osrc[o] = e;
}

// Rows of at most RENUM_SHORT elements, a wave at a time (waves stride over
// the rows): an element's place is the number of elements before it in
// (index, caller's position) order, counted against every lane's key in turn.
template <typename IdxT>
__global__ __launch_bounds__(BLOCK) void renum_short_kernel(RenumArgs a, uint32_t row0, uint32_t rows) {
    const uint32_t lane = threadIdx.x & (WAVE - 1);
    uint32_t w = blockIdx.x * (BLOCK / WAVE) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (; w < rows; w += gridDim.x * (BLOCK / WAVE)) {
        const uint32_t row = row0 + w;
        const uint32_t o = a.optr[row], len = a.optr[row + 1] - o, e = a.ptr[a.perm[row]] + lane;
        const bool ok = lane < len;
        const uint32_t key = ok ? a.ipos[a.idx[e]] : 0xffffffffu;
        uint32_t rank = 0;
        for (uint32_t j = 0; j < len; ++j) {
            const uint32_t kj = (uint32_t)__builtin_amdgcn_readlane((int)key, (int)j);
            rank += kj < key + (j < lane ? 1u : 0u) ? 1u : 0u;
        }
        if (ok) put<IdxT>(a, o + rank, key, e);
    }
}

// Rows of RENUM_SHORT + 1 .. MID_MAX elements, a block at a time, the same
// count against the row's keys in LDS (four a read, the same four for every
// lane).  len^2 / 64 compares a wave: past the bound of renum_long_len the
// bitmap below is cheaper.
constexpr uint32_t MID_MAX = 1024;
template <typename IdxT, int NQ>
__device__ __forceinline__ void renum_mid_row(const RenumArgs& a, uint32_t* keys, uint32_t o, uint32_t len,
                                              uint32_t e0) {
    uint32_t key[NQ], rank[NQ];
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const uint32_t p = threadIdx.x + BLOCK * q;
        key[q] = p < len ? a.ipos[a.idx[e0 + p]] : 0xffffffffu;
        rank[q] = 0;
        keys[p] = key[q];  // past the row: larger than any key
    }
    __syncthreads();
    for (uint32_t j = 0; j < len; j += 4) {
        const uint4 k4 = *reinterpret_cast<const uint4*>(keys + j);
        const uint32_t kj[4] = {k4.x, k4.y, k4.z, k4.w};
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int q = 0; q < NQ; ++q)
                rank[q] += kj[u] < key[q] + (j + u < threadIdx.x + BLOCK * q ? 1u : 0u) ? 1u : 0u;
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        const uint32_t p = threadIdx.x + BLOCK * q;
        if (p < len) put<IdxT>(a, o + rank[q], key[q], e0 + p);
    }
}

template <typename IdxT>
__global__ __launch_bounds__(BLOCK) void renum_mid_kernel(RenumArgs a, uint32_t row0, uint32_t rows) {
    __shared__ __align__(16) uint32_t keys[MID_MAX];
    for (uint32_t b = blockIdx.x; b < rows; b += gridDim.x) {
        const uint32_t row = row0 + b;
        const uint32_t o = a.optr[row], len = a.optr[row + 1] - o, e0 = a.ptr[a.perm[row]];
        if (b != blockIdx.x) __syncthreads();  // every wave is done with the last row's keys
        if (len <= BLOCK) renum_mid_row<IdxT, 1>(a, keys, o, len, e0);
        else if (len <= 2 * BLOCK) renum_mid_row<IdxT, 2>(a, keys, o, len, e0);
        else renum_mid_row<IdxT, 4>(a, keys, o, len, e0);
    }
}

// Longer rows, one block each: the row's indices are set in a bitmap of the
// gathered dimension in LDS (in windows of WIN_WORDS words), and an
// element's place is the number of bits set before its own (a prefix sum
// per group of 8 words, then popcounts).  Linear in the row's length plus
// gdim / 32.  An index that occurs twice in a row sets dup[row] and
// dup[nlong]; renum_dup_kernel then sorts that row.
constexpr uint32_t WIN_WORDS = 32768;  // 2^20 indices, 144 KB with the prefix sums
constexpr uint32_t GROUP = 8;
template <typename IdxT, int BS>
__global__ __launch_bounds__(BS) void renum_long_kernel(RenumArgs a, uint32_t* __restrict__ dup, uint32_t words) {
    extern __shared__ __align__(16) uint32_t bits[];  // words, then words / GROUP prefix sums
    __shared__ uint32_t wsum[BS / WAVE];
    uint32_t* pre = bits + words;
    const uint32_t row = blockIdx.x, lane = threadIdx.x & (WAVE - 1), wv = threadIdx.x >> 6;
    const uint32_t o = a.optr[row], len = a.optr[row + 1] - o, e0 = a.ptr[a.perm[row]];
    const uint32_t ng = words / GROUP, per = (ng + BS - 1) / BS;
    uint32_t below = 0;
    int twice = 0;
    for (uint64_t w0 = 0; w0 < a.gdim; w0 += (uint64_t)words * 32) {
        const uint32_t lo = (uint32_t)w0;
        for (uint32_t q = threadIdx.x; q < words; q += BS) bits[q] = 0u;
        __syncthreads();
        for (uint64_t p = threadIdx.x; p < len; p += BS) {  // 64 bits: len + BS may pass 2^32
            const uint32_t k = a.ipos[a.idx[e0 + p]] - lo;  // wraps past the window for smaller indices
            if (k < words * 32) {
                const uint32_t bit = 1u << (k & 31u);
                if (atomicOr(&bits[k >> 5], bit) & bit) twice = 1;
            }
        }
        __syncthreads();
        // exclusive prefix sums of the groups' bit counts
        uint32_t mine = 0;
        for (uint32_t g = threadIdx.x * per; g < min(ng, (threadIdx.x + 1) * per); ++g) {
            pre[g] = mine;
#pragma unroll
            for (uint32_t u = 0; u < GROUP; ++u) mine += (uint32_t)__popc(bits[g * GROUP + u]);
        }
        uint32_t incl = mine;
#pragma unroll
        for (int d = 1; d < WAVE; d <<= 1) {
            const uint32_t t = __shfl_up(incl, d);
            if (lane >= (uint32_t)d) incl += t;
        }
        if (lane == WAVE - 1) wsum[wv] = incl;
        __syncthreads();
        uint32_t off = incl - mine, total = 0;
        for (uint32_t q = 0; q < BS / WAVE; ++q) {
            if (q < wv) off += wsum[q];
            total += wsum[q];
        }
        for (uint32_t g = threadIdx.x * per; g < min(ng, (threadIdx.x + 1) * per); ++g) pre[g] += off;
        __syncthreads();
        for (uint64_t p = threadIdx.x; p < len; p += BS) {
            const uint32_t key = a.ipos[a.idx[e0 + p]], k = key - lo;
            if (k >= words * 32) continue;
            const uint32_t w = k >> 5;
            uint32_t rank = below + pre[w / GROUP] + (uint32_t)__popc(bits[w] & ((1u << (k & 31u)) - 1u));
            for (uint32_t u = w / GROUP * GROUP; u < w; ++u) rank += (uint32_t)__popc(bits[u]);
            put<IdxT>(a, o + rank, key, e0 + (uint32_t)p);
        }
        below += total;
        __syncthreads();
    }
    if (twice) {
        dup[row] = 1u;
        dup[gridDim.x] = 1u;
    }
}

// Long rows that hold an index twice, a block at a time: a stable radix sort
// of the caller's positions by internal index, eight bits a pass, between
// the row's place in osrc (the last pass ends there) and in oval.  A wave
// takes 64 consecutive positions a step of its part of the row; lanes of one
// digit are found by ballots and keep their order.  Linear in the row's
// length, where counting every element against the whole row took its
// square: uploads of 50,000 such rows of 300 elements 29.6 -> 10.3 ms, 60 of
// 30,000 26 -> 2.1, two of 400,000 169 -> 9.2 (58 sorted on the host), one of
// 3,000,000 56 ms.  Without such a row the blocks leave at once.
constexpr int DUP_BLOCK = 1024, DUP_WAVES = DUP_BLOCK / WAVE, DIGITS = 256;
constexpr uint32_t DUP_BLOCKS = 512;  // two a CU
template <typename IdxT>
__global__ __launch_bounds__(DUP_BLOCK) void renum_dup_kernel(RenumArgs a, const uint32_t* __restrict__ dup,
                                                              uint32_t nlong, uint32_t passes) {
    __shared__ uint32_t place[DUP_WAVES][DIGITS];  // counts, then the next place of each digit
    __shared__ uint32_t wsum[DIGITS / WAVE];
    if (!dup[nlong]) return;
    const uint32_t lane = threadIdx.x & (WAVE - 1), wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (uint32_t row = blockIdx.x; row < nlong; row += gridDim.x) {
        if (!dup[row]) continue;
        const uint32_t o = a.optr[row], len = a.optr[row + 1] - o, e0 = a.ptr[a.perm[row]];
        uint32_t* const buf[2] = {a.osrc + o, reinterpret_cast<uint32_t*>(a.oval) + o};
        const uint32_t part = (len / DUP_WAVES / WAVE + 1) * WAVE;  // at least len / DUP_WAVES
        const uint32_t p0 = min(len, wv * part), p1 = p0 + min(len - p0, part);
        for (uint32_t pass = 0; pass < passes; ++pass) {
            const uint32_t* const src = buf[(passes - pass) & 1];
            uint32_t* const dst = buf[(passes - 1 - pass) & 1];
            // f(position, its mask of lanes with the same digit, the digit);
            // a wave's steps see each other's places in LDS
            auto walk = [&](auto f) {
                for (uint64_t b = p0; b < p1; b += WAVE) {
                    const uint64_t p = b + lane;
                    const bool ok = p < p1;
                    const uint32_t e = !ok ? 0u : pass ? src[p] : e0 + (uint32_t)p;
                    const uint32_t digit = ok ? (a.ipos[a.idx[e]] >> (8 * pass)) & (DIGITS - 1) : 0u;
                    uint64_t same = __ballot(ok);
#pragma unroll
                    for (int bit = 0; bit < 8; ++bit) {
                        const uint64_t set = __ballot((digit >> bit) & 1u);
                        same &= (digit >> bit) & 1u ? set : ~set;
                    }
                    if (ok) f(e, same, digit);
                    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                }
            };
            for (uint32_t q = threadIdx.x; q < DUP_WAVES * DIGITS; q += DUP_BLOCK) (&place[0][0])[q] = 0u;
            __syncthreads();
            walk([&](uint32_t, uint64_t same, uint32_t digit) {
                if (lane == (uint32_t)__builtin_ctzll(same)) place[wv][digit] += (uint32_t)__popcll(same);
            });
            __syncthreads();
            // digits in order, and each digit's waves in order
            uint32_t mine = 0, incl;
            if (threadIdx.x < DIGITS) {
                for (int w = 0; w < DUP_WAVES; ++w) mine += place[w][threadIdx.x];
                incl = mine;
#pragma unroll
                for (int d = 1; d < WAVE; d <<= 1) {
                    const uint32_t t = __shfl_up(incl, d);
                    if (lane >= (uint32_t)d) incl += t;
                }
                if (lane == WAVE - 1) wsum[wv] = incl;
            }
            __syncthreads();
            if (threadIdx.x < DIGITS) {
                uint32_t at = incl - mine;
                for (uint32_t w = 0; w < wv; ++w) at += wsum[w];
                for (int w = 0; w < DUP_WAVES; ++w) {
                    const uint32_t n = place[w][threadIdx.x];
                    place[w][threadIdx.x] = at;
                    at += n;
                }
            }
            __syncthreads();
            walk([&](uint32_t e, uint64_t same, uint32_t digit) {
                const uint32_t at = place[wv][digit];
                // read by all before the first of them moves it on
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __builtin_amdgcn_wave_barrier();
                const uint32_t before = (uint32_t)__popcll(same & ((1ull << lane) - 1ull));
                if (before == 0) place[wv][digit] = at + (uint32_t)__popcll(same);
                dst[at + before] = e;
            });
            __syncthreads();
        }
        for (uint64_t p = threadIdx.x; p < len; p += DUP_BLOCK) {
            const uint32_t e = a.osrc[o + p];
            put<IdxT>(a, o + (uint32_t)p, a.ipos[a.idx[e]], e);
        }
        __syncthreads();
    }
}

// One thread per row: the bit of its first element in its lane's word.
__global__ __launch_bounds__(BLOCK) void tile_flags_kernel(const uint32_t* __restrict__ ptr, uint64_t rows,
                                                           uint32_t sigma, uint32_t* __restrict__ flags) {
    const uint64_t stride = (uint64_t)gridDim.x * BLOCK;
    for (uint64_t r = (uint64_t)blockIdx.x * BLOCK + threadIdx.x; r < rows; r += stride) {
        const uint32_t e = ptr[r];
        if (ptr[r + 1] == e) continue;
        const uint32_t ln = e / sigma, bit = e % sigma;  // a tile is 64 whole lanes
        if (sigma <= 16) atomicOr(flags + ln / 2, 1u << (16 * (ln & 1) + bit));
        else atomicOr(flags + ln, 1u << bit);
    }
}

// One block per virtual row (grid-stride): its elements' positions are consecutive in the
// layout.
__global__ __launch_bounds__(BLOCK) void split_positions_kernel(const uint32_t* __restrict__ vptr,
                                                                const uint32_t* __restrict__ lptr,
                                                                const uint32_t* __restrict__ below,
                                                                const uint32_t* __restrict__ cold_row, uint32_t nreal,
                                                                uint64_t vrows, uint32_t* __restrict__ vpos) {
    for (uint64_t v = blockIdx.x; v < vrows; v += gridDim.x) {
        const uint32_t v0 = vptr[v], len = vptr[v + 1] - v0;
        uint32_t src;
        if (v < nreal) {
            src = lptr[v];
        } else {
            const uint32_t r = cold_row[v - nreal];
            src = lptr[r] + below[r];
        }
        for (uint64_t q = threadIdx.x; q < len; q += BLOCK) vpos[v0 + q] = src + (uint32_t)q;
    }
}

constexpr uint32_t MAX_BLOCKS = 16384;
uint32_t grid_for(uint64_t count) {
    return (uint32_t)std::min<uint64_t>(std::max<uint64_t>((count + BLOCK - 1) / BLOCK, 1), MAX_BLOCKS);
}

}  // namespace

hipError_t launch_permute_ranks(const float* src, float* dst, const uint32_t* perm, uint32_t k, uint64_t rows,
                                bool to_internal, hipStream_t s) {
    if (k == 0 || rows == 0) return hipSuccess;
    const uint32_t y = std::min<uint32_t>((k + RANKS_PER_BLOCK - 1) / RANKS_PER_BLOCK, 65535u);
    const dim3 grid((uint32_t)((rows + BLOCK - 1) / BLOCK), y);
    if (to_internal)
        hipLaunchKernelGGL(permute_ranks_kernel<true>, grid, dim3(BLOCK), 0, s, src, dst, perm, k, rows);
    else
        hipLaunchKernelGGL(permute_ranks_kernel<false>, grid, dim3(BLOCK), 0, s, src, dst, perm, k, rows);
    return hipGetLastError();
}

hipError_t launch_scatter(const float* src, const uint32_t* map, float* dst, uint64_t count, hipStream_t s) {
    if (count == 0) return hipSuccess;
    hipLaunchKernelGGL(scatter_kernel, dim3(grid_for(count)), dim3(BLOCK), 0, s, src, map, dst, count);
    return hipGetLastError();
}

hipError_t launch_index_check(const uint32_t* idx, uint64_t count, uint32_t dim, uint32_t* bad, hipStream_t s) {
    if (count == 0) return hipSuccess;
    hipLaunchKernelGGL(index_check_kernel, dim3(grid_for(count)), dim3(BLOCK), 0, s, idx, count, dim, bad);
    return hipGetLastError();
}

// Where a block's count over 256 keys and the bitmap of a small gathered
// dimension cost about the same; a bitmap past 8 KB takes longer to clear
// and sum than to count four times as many keys.
uint32_t renum_long_len(uint32_t gdim) { return gdim <= 65536u ? 256u : MID_MAX; }

template <typename IdxT>
static hipError_t renumber(const RenumArgs& a, const RenumRows& n, uint32_t* dup, hipStream_t s) {
    if (n.nlong) {
        hipError_t e = launch_fill(reinterpret_cast<float*>(dup), 0.0f, (uint64_t)n.nlong + 1, s);
        if (e != hipSuccess) return e;
        const uint32_t words = std::min<uint32_t>((uint32_t)((((uint64_t)a.gdim + 31) / 32 + GROUP - 1) / GROUP * GROUP),
                                                  WIN_WORDS);
        const size_t lds = sizeof(uint32_t) * (words + words / GROUP);
        if (words <= 2048)
            hipLaunchKernelGGL((renum_long_kernel<IdxT, 256>), dim3(n.nlong), dim3(256), lds, s, a, dup, words);
        else
            hipLaunchKernelGGL((renum_long_kernel<IdxT, 1024>), dim3(n.nlong), dim3(1024), lds, s, a, dup, words);
        if ((e = hipGetLastError()) != hipSuccess) return e;
        const uint32_t passes = a.gdim <= 256u ? 1 : a.gdim <= 65536u ? 2 : a.gdim <= 1u << 24 ? 3 : 4;
        hipLaunchKernelGGL(renum_dup_kernel<IdxT>, dim3(std::min(n.nlong, DUP_BLOCKS)), dim3(DUP_BLOCK), 0, s, a, dup,
                           n.nlong, passes);
        if ((e = hipGetLastError()) != hipSuccess) return e;
    }
    // A launch takes less than 2^32 threads, which is 16.7M rows at a block
    // each and 67M at a wave each: a bounded grid strides over the rows.
    if (n.nmid)
        hipLaunchKernelGGL(renum_mid_kernel<IdxT>, dim3(std::min(n.nmid, MAX_BLOCKS)), dim3(BLOCK), 0, s, a, n.nlong,
                           n.nmid);
    if (n.nshort)
        hipLaunchKernelGGL(renum_short_kernel<IdxT>, dim3(grid_for((uint64_t)n.nshort * WAVE)), dim3(BLOCK), 0, s, a,
                           n.nlong + n.nmid, n.nshort);
    return hipGetLastError();
}

hipError_t launch_renumber(const RenumArgs& a, bool idx16, const RenumRows& n, uint32_t* dup, hipStream_t s) {
    return idx16 ? renumber<uint16_t>(a, n, dup, s) : renumber<uint32_t>(a, n, dup, s);
}

hipError_t launch_tile_flags(const uint32_t* ptr, uint64_t rows, uint64_t ntiles, int sigma, uint32_t* flags,
                             hipStream_t s) {
    if (ntiles == 0) return hipSuccess;
    const hipError_t e = launch_fill(reinterpret_cast<float*>(flags), 0.0f, ntiles * (sigma <= 16 ? 32 : 64), s);
    if (e != hipSuccess || rows == 0) return e;
    hipLaunchKernelGGL(tile_flags_kernel, dim3(grid_for(rows)), dim3(BLOCK), 0, s, ptr, rows, (uint32_t)sigma, flags);
    return hipGetLastError();
}

hipError_t launch_split_positions(const uint32_t* vptr, uint64_t vrows, const uint32_t* lptr, const uint32_t* below,
                                  const uint32_t* cold_row, uint32_t nreal, uint32_t* vpos, hipStream_t s) {
    if (vrows == 0) return hipSuccess;
    hipLaunchKernelGGL(split_positions_kernel, dim3((uint32_t)std::min<uint64_t>(vrows, 1u << 20)), dim3(BLOCK), 0, s,
                       vptr, lptr, below, cold_row, nreal, vrows, vpos);
    return hipGetLastError();
}

}  // namespace ccd
