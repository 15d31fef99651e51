// Weights of a streamer, fetched whole 128-byte lines at a time.
//
// The "A" operand of the 16 x 16 matrix instructions wants, in lane 16 q + s, piece q (16 bytes) of row s: an instruction that
// fetches it so takes half of a line of each of 16 rows.  Memory gives 7.1 TB/s to loads that say that nobody will want the line
// again (non-temporal) and 6.1 to others, but only where an instruction takes the line whole (halves: the other half is gone
// when the next instruction asks for it).  So two instructions fetch eight rows of 128 bytes each, lanes s and s + 8 sharing a row in
// both, and trade what belongs to the other: lane s of the lower eight keeps its piece of the first instruction and takes the upper
// piece of its row, which its partner fetched there; the upper eight likewise from the second.  Eight lanes apart within sixteen is a
// rotation by eight, a DPP move: twelve moves for 2 KB, no LDS.  A wavefront reading 16 rows of 8 KB / 28 KB / 2 KB / 7 KB, TB/s: halves
// 5.8 / 5.7 / 6.0 / 5.9, halves non-temporal 6.0 / 5.3 / 6.2 / 5.5, lines 5.9 / 5.7 / 6.1 / 5.9, lines non-temporal 6.6 / 6.5 / 6.7 / 6.8.
#pragma once

#include "moe_internal.hpp"

namespace moe355 {
namespace {

typedef uint32_t line_u32x4 __attribute__((ext_vector_type(4)));

// Whether a call's weights (those of the experts that can be hit) are more than the memory-side cache of 256 MB would hold for the next call.
inline bool stream_cold(const FfnArgs& a, int element_bytes) {
    const int64_t pairs = (int64_t)a.S * a.k, experts = pairs < a.E ? pairs : a.E;
    return experts * a.H * a.I * (a.act == MOE_ACT_SWIGLU ? 3 : 2) * element_bytes > ((int64_t)256 << 20);
}

template <bool NONTEMPORAL>
__device__ __forceinline__ line_u32x4 load_piece(const void* p) {
    if constexpr (NONTEMPORAL) return __builtin_nontemporal_load(reinterpret_cast<const line_u32x4*>(p));
    else return *reinterpret_cast<const line_u32x4*>(p);
}
// Bytes from the first of 16 rows to what this lane fetches of 128 bytes of theirs: the first instruction, and how much further the
// second is.
__device__ __forceinline__ int64_t line_first(int lane, int64_t row_bytes) { return (lane & 7) * row_bytes + ((lane >> 4) + ((lane & 8) >> 1)) * 16; }
__device__ __forceinline__ int64_t line_second(int lane, int64_t row_bytes) { return 8 * row_bytes + ((lane & 8) ? -64 : 64); }
// What the two instructions brought -> this lane's piece of the lower and of the upper 64 bytes of row (lane & 15).
__device__ __forceinline__ void line_pieces(const line_u32x4& first, const line_u32x4& second, line_u32x4& lower, line_u32x4& upper) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int a = (int)first[i], b = (int)second[i];
        lower[i] = (uint32_t)__builtin_amdgcn_update_dpp(a, b, 0xE4, 0xF, 0xC, false);                  // lanes 8..15 of sixteen: the second
        const int other = __builtin_amdgcn_update_dpp(0, a, 0x128, 0xF, 0x3, false);                    // row_ror:8, lanes 0..7: the partner's first
        upper[i] = (uint32_t)__builtin_amdgcn_update_dpp(other, b, 0x128, 0xF, 0xC, false);             // lanes 8..15: the partner's second
    }
}

}  // namespace
}  // namespace moe355
