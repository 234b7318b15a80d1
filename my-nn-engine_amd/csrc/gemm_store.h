// The store of a matrix-core product: a workgroup's accumulator tiles -> row-major 16-bit output, with the residual add
// or SwiGLU of the operator that follows.
#pragma once
#include "kernels.h"
#include "mfma.h"

namespace mynn {

// ---- store of a workgroup tile.  The MFMAs take the weight fragment as their first operand, so an
// accumulator tile is the transpose of the output tile: lane l holds output row l % 32 and, in elements
// 4q..4q+3, the four neighbouring output columns 8q + 4*(l/32) + 0..3 -- one 8-byte piece of a row.  Each
// wave turns one 32-row strip of its tile at a time into row-major 16-bit values in its own LDS patch (the
// operand buffers are free by now) and writes it out, and reads the residual, 16 bytes per lane, rows
// contiguous.
// GEMM_SWIGLU: gate and up columns alternate in groups of 32 (two column tiles of a wave); GEMM_SWIGLU_PAIRS: they
// alternate one by one (column 2i gate_i, 2i+1 up_i: two neighbours in a lane); _EXP: the same with expf and a division.
// at(i, j, e): element e of the accumulator of MFMA tile (i, j), as f32 ready to be rounded.
template <typename T, typename G, int EPI, typename AccAt>
__device__ __forceinline__ void gemm_store(AccAt at, uint16_t *lds, T *C, const T *R, int M, int N, int m0,
                                           int n0, int wrow, int wcol, int lane, int wave) {
    constexpr int TI = G::TI, TJ = G::TJ;
    constexpr int EST = G::EST;
    constexpr bool GROUPS = EPI == GEMM_SWIGLU || EPI == GEMM_SWIGLU_EXP;
    static_assert(!GROUPS || TJ % 2 == 0, "the SwiGLU store pairs neighbouring column tiles");
    constexpr bool PAIRS = EPI == GEMM_SWIGLU_PAIRS || EPI == GEMM_SWIGLU_PAIRS_EXP;
    constexpr bool HALF = GROUPS || PAIRS;  // two accumulator columns per output column
    constexpr int OC = HALF ? TJ * 16 : TJ * 32;  // output columns of the wave tile
    constexpr int CPR = OC / 8;                   // 16-byte chunks per strip row
    const int ldc = HALF ? N >> 1 : N;
    const int c0 = HALF ? (n0 + wcol) >> 1 : n0 + wcol;
    T *patch = (T *)lds + (size_t)wave * 32 * EST;
    const bool vec_ok = (ldc & 7) == 0 && ((uintptr_t)C & 15) == 0 && (EPI != GEMM_RESIDUAL || ((uintptr_t)R & 15) == 0);  // (uniform)
#pragma unroll
    for (int i = 0; i < TI; i++) {
        T *prow = patch + (lane & 31) * EST + (lane >> 5) * (PAIRS ? 2 : 4);
        // hardware 2^x and reciprocal (about 1 ulp of f32 each, far below the 16-bit rounding that follows); the exact
        // expf and division cost ~35 instructions per element here (a layer of 300 x 5632 outputs 1.7 us).  _EXP has them:
        // for executors whose SwiGLU would otherwise be mynn_swiglu's
        auto swiglu = [](float gate, float up) {
            const float g = Elem<T>::rnd(gate), u = Elem<T>::rnd(up);
            if constexpr (EPI == GEMM_SWIGLU_PAIRS_EXP || EPI == GEMM_SWIGLU_EXP) return (g * (1.0f / (1.0f + expf(-g)))) * u;
            else return (g * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(g * -1.4426950408889634f))) * u;
        };
#pragma unroll
        for (int q = 0; q < 4; q++) {
            if constexpr (GROUPS) {
#pragma unroll
                for (int j = 0; j < TJ; j += 2) {
                    float o[4];
#pragma unroll
                    for (int x = 0; x < 4; x++) o[x] = swiglu(at(i, j, 4 * q + x), at(i, j + 1, 4 * q + x));
                    *(uint2 *)(prow + j * 16 + 8 * q) = uint2{pack2<T>(o[0], o[1]), pack2<T>(o[2], o[3])};
                }
            } else if constexpr (PAIRS) {
#pragma unroll
                for (int j = 0; j < TJ; j++)
                    *(uint32_t *)(prow + j * 16 + 4 * q) = pack2<T>(swiglu(at(i, j, 4 * q), at(i, j, 4 * q + 1)), swiglu(at(i, j, 4 * q + 2), at(i, j, 4 * q + 3)));
            } else {
#pragma unroll
                for (int j = 0; j < TJ; j++)
                    *(uint2 *)(prow + j * 32 + 8 * q) = uint2{pack2<T>(at(i, j, 4 * q), at(i, j, 4 * q + 1)),
                                                              pack2<T>(at(i, j, 4 * q + 2), at(i, j, 4 * q + 3))};
            }
        }
        __builtin_amdgcn_wave_barrier();
        const int row0 = m0 + wrow + i * 32;
#pragma unroll
        for (int q = 0; q < 32 * CPR / 64; q++) {
            const int ch = q * 64 + lane, r = ch / CPR, cc = (ch % CPR) * 8;
            const int row = row0 + r, col = c0 + cc;
            if (row >= M || col >= ldc) continue;
            U4 v = *(const U4 *)&patch[r * EST + cc];
            const size_t at = (size_t)row * ldc + col;
            if (vec_ok) {  // (col, like ldc, is a multiple of 8: all eight lie within the row)
                if (EPI == GEMM_RESIDUAL) {
                    float fv[8], fr8[8];
                    widen8<T>(v, fv);
                    widen8<T>(*(const U4 *)(R + at), fr8);
                    v = U4{pack2<T>(fr8[0] + fv[0], fr8[1] + fv[1]), pack2<T>(fr8[2] + fv[2], fr8[3] + fv[3]),
                           pack2<T>(fr8[4] + fv[4], fr8[5] + fv[5]), pack2<T>(fr8[6] + fv[6], fr8[7] + fv[7])};
                }
                *(U4 *)(C + at) = v;
            } else {
                for (int x = 0; x < 8 && col + x < ldc; x++) {
                    const float f = Elem<T>::ld(patch, r * EST + cc + x);
                    if (EPI == GEMM_RESIDUAL) Elem<T>::st(C, at + x, Elem<T>::ld(R, at + x) + f);
                    else C[at + x] = patch[r * EST + cc + x];
                }
            }
        }
        __builtin_amdgcn_wave_barrier();
    }
}

}  // namespace mynn
