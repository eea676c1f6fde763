// Set-up kernels between the caller's numbering and the internal one
// (layout_kernels.hip).  perm: internal row -> caller's row.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ccd {

// Rank-major [k][rows]: dst[t][i] = src[t][perm[i]] (to_internal), or
// dst[t][perm[i]] = src[t][i].
hipError_t launch_permute_ranks(const float* src, float* dst, const uint32_t* perm, uint32_t k, uint64_t rows,
                                bool to_internal, hipStream_t s);
// dst[map[e]] = src[e], e < count
hipError_t launch_scatter(const float* src, const uint32_t* map, float* dst, uint64_t count, hipStream_t s);


// One compressed copy on its way into internal numbering: rows in perm
// order (falling length), indices mapped through ipos, the elements of every
// row sorted by internal index, equal ones in the caller's order.  All
// arrays on the device; idx holds checked indices (below gdim).
struct RenumArgs {
    const uint32_t* ptr;   // caller's row pointer
    const uint32_t* idx;   // caller's indices and values
    const float* val;
    const uint32_t* perm;  // internal row -> caller's row
    const uint32_t* ipos;  // caller's index -> internal index
    const uint32_t* optr;  // internal row pointer
    void* oidx;            // out: indices, u16 or u32
    float* oval;           // out: values
    uint32_t* osrc;        // out: caller's position of each element
    uint32_t gdim;         // indices are below this
};

// Row counts by length class, in row order: longer than the bound of
// renum_long_len(gdim), then longer than RENUM_SHORT, then the others with
// elements.
constexpr uint32_t RENUM_SHORT = 64;
uint32_t renum_long_len(uint32_t gdim);
struct RenumRows {
    uint32_t nlong, nmid, nshort;
};
// dup: nlong + 1 words of scratch
hipError_t launch_renumber(const RenumArgs& a, bool idx16, const RenumRows& n, uint32_t* dup, hipStream_t s);
// *bad |= 1 when an index is not below dim (*bad set by the caller)
hipError_t launch_index_check(const uint32_t* idx, uint64_t count, uint32_t dim, uint32_t* bad, hipStream_t s);


// Per-element tables of a tiled layout (tile_layout.h).  ptr: row pointer of
// its (virtual) rows.
// flags: zeroed here; per lane one u16 (sigma <= 16) or u32
hipError_t launch_tile_flags(const uint32_t* ptr, uint64_t rows, uint64_t ntiles, int sigma, uint32_t* flags,
                             hipStream_t s);
// Position map of a split layout: vptr, its virtual row pointer (vrows + 1);
// lptr and below, the layout's row pointer and per-row split counts;
// cold_row, the real rows of virtual rows nreal, nreal + 1, ...
hipError_t launch_split_positions(const uint32_t* vptr, uint64_t vrows, const uint32_t* lptr, const uint32_t* below,
                                  const uint32_t* cold_row, uint32_t nreal, uint32_t* vpos, hipStream_t s);

}  // namespace ccd
