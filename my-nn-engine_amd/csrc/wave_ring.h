// What the rings of a wave's own loads have in common (rowblock.hip, qrows.hip): both operands go global -> LDS by the load unit into stages that
// no other wave touches, and nothing is waited for but the wave's own loads, by count.
//
// The walk over the stages is written out in both kernels, and a change to one belongs in the other: as a function of its parts (closures that ask, read and
// multiply, by value or by reference) it left generic addresses in qrows.hip and other instructions in every kernel of both; what is here leaves them as they were.
#pragma once
#include "mfma.h"

namespace mynn {

// until no more than LEFT loads are in flight, and all LDS reads are through
template <int LEFT> __device__ __forceinline__ void wait_for_loads() {
    static_assert(LEFT < 64, "a counter of six bits");
    __builtin_amdgcn_s_waitcnt((LEFT & 15) | (LEFT >> 4) << 14 | 0x70);
    asm volatile("" ::: "memory");
}

// Row 8 * i + lane / 8 of an int8 operand (`last`: its last one), and of the row's 8 chunks of 16 bytes the one that makes the fragment reads
// meet different banks: as load_group_to_lds takes them, the i-th loads in groups of four, from 4096 bytes in front of a step
__device__ __forceinline__ uint32_t ring_chunk(int lane, int i, int last, int K) {
    return (uint32_t)(min(8 * i + (lane >> 3), last) * K + (((lane & 7) ^ (lane >> 3)) << 4) + 4096 - 1024 * (i % 4));
}

}  // namespace mynn
