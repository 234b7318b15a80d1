// Thin wrappers over the gfx950 matrix-core builtins used by the GEMM and attention kernels.
// v_mfma_f32_32x32x16_{f16,bf16}: A is 32 x 16 (lane l holds row l%32, k = 8*(l/32) .. +7),
// B is 16 x 32 (lane l holds column l%32, k = 8*(l/32) .. +7), D is 32 x 32 f32 (lane l holds
// column l%32 and the 16 rows 8*(e/4) + 4*(l/32) + e%4, e = 0..15).
#pragma once
#include <type_traits>

#include "mynn_common.h"

namespace mynn {

typedef _Float16 h8_t __attribute__((ext_vector_type(8)));
typedef __bf16 b8_t __attribute__((ext_vector_type(8)));
typedef float f16x_t __attribute__((ext_vector_type(16)));

template <typename T> struct Mfma;
template <> struct Mfma<f16_t> {
    __device__ static f16x_t run(const U4 &a, const U4 &b, f16x_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8_t, a), __builtin_bit_cast(h8_t, b), c, 0, 0, 0);
    }
};
template <> struct Mfma<bf16_t> {
    __device__ static f16x_t run(const U4 &a, const U4 &b, f16x_t c) {
        return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(b8_t, a), __builtin_bit_cast(b8_t, b), c, 0, 0, 0);
    }
};

// ds_read_b64_tr_b16: of each 16 lanes, lane i names the 8 bytes at row i / 4, columns 4 * (i % 4) .. +3 of a 4 x 16 block of 16-bit
// values (anywhere in LDS, 8-byte aligned), and receives the block's column i, rows 0 .. 3
typedef short s4_t __attribute__((ext_vector_type(4)));
__device__ inline uint2 lds_read_tr16(const char *p) {
    return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s4_t *)p));
}

// 16 bytes per lane to LDS byte lds + 16 * lane (wave-uniform), from base + off (base wave-uniform) or from p.  As instructions of
// their own and not through the builtin: behind the builtin the compiler puts a wait for EVERY load in flight before the next
// ds_read that it cannot tell apart from what is being written, the stages further ahead among them.  The caller waits (vmcnt,
// then a barrier) before it reads what was loaded.
__device__ inline uint32_t lds_offset(const void *p) { return (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char *)p; }
__device__ inline const char *scalar_pointer(const char *p) {  // (nothing where it is in scalar registers already)
    const uint64_t u = (uint64_t)(uintptr_t)p;
    return (const char *)(((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(u >> 32)) << 32) | (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)u));
}
// (m0 is a register that the compiler keeps for itself and sets in front of whatever uses it: named as overwritten, which it warns of)
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ inline void load_to_lds(const char *base, uint32_t off, uint32_t lds) {
    lds = __builtin_amdgcn_readfirstlane(lds);
    base = scalar_pointer(base);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(off), "s"(base) : "memory", "m0");
}
__device__ inline void load_to_lds(const char *p, uint32_t lds) {
    lds = __builtin_amdgcn_readfirstlane(lds);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds), "v"(p) : "memory", "m0");
}

// N <= 4 of them to consecutive kilobytes of LDS from one setting of m0: load i adds 1024 * i to both of its addresses, so off[i] is
// 1024 * i short of the distance from base.  NT: with the non-temporal hint, for what is read once.
template <int N, bool NT = false> __device__ inline void load_group_to_lds(const char *base, const uint32_t *off, uint32_t lds) {
    static_assert(N >= 1 && N <= 4, "the offset has 12 bits");
    lds = __builtin_amdgcn_readfirstlane(lds);
    base = scalar_pointer(base);
#define MYNN_LOAD(i, o, nt) "\n\tglobal_load_lds_dwordx4 %" #i ", %1 offset:" #o nt
#define MYNN_GROUP(nt)                                                                                                                                          \
    if constexpr (N == 1) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" MYNN_LOAD(2, 0, nt) ::"s"(lds), "s"(base), "v"(off[0]) : "memory", "m0");                  \
    else if constexpr (N == 2)                                                                                                                                  \
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" MYNN_LOAD(2, 0, nt) MYNN_LOAD(3, 1024, nt) ::"s"(lds), "s"(base), "v"(off[0]), "v"(off[1]) : "memory", "m0"); \
    else if constexpr (N == 3)                                                                                                                                  \
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" MYNN_LOAD(2, 0, nt) MYNN_LOAD(3, 1024, nt) MYNN_LOAD(4, 2048, nt) ::"s"(lds), "s"(base), "v"(off[0]),       \
                     "v"(off[1]), "v"(off[2])                                                                                                                   \
                     : "memory", "m0");                                                                                                                         \
    else                                                                                                                                                        \
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0" MYNN_LOAD(2, 0, nt) MYNN_LOAD(3, 1024, nt) MYNN_LOAD(4, 2048, nt) MYNN_LOAD(5, 3072, nt) ::"s"(lds),        \
                     "s"(base), "v"(off[0]), "v"(off[1]), "v"(off[2]), "v"(off[3])                                                                              \
                     : "memory", "m0");
    if constexpr (NT) {
        MYNN_GROUP(" nt")
    } else {
        MYNN_GROUP("")
    }
#undef MYNN_GROUP
#undef MYNN_LOAD
}
#pragma clang diagnostic pop

// two f32 -> one dword of two storage-type values (low half first), round to nearest even: one packed
// convert instruction.  The inputs are values ALREADY rounded to f32 (the empty asm keeps the compiler from
// fusing the producing multiply into a mixed-precision op that would round the exact product once).
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 h2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf2_t __attribute__((ext_vector_type(2)));
template <typename T> __device__ inline uint32_t cvt2(float lo, float hi) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){lo, hi}, std::conditional_t<std::is_same<T, f16_t>::value, h2_t, bf2_t>));
}
template <typename T> __device__ inline uint32_t pack2(float lo, float hi);
template <> __device__ inline uint32_t pack2<f16_t>(float lo, float hi) {
    asm volatile("" : "+v"(lo), "+v"(hi));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){lo, hi}, h2_t));
}
template <> __device__ inline uint32_t pack2<bf16_t>(float lo, float hi) {
    asm volatile("" : "+v"(lo), "+v"(hi));
    return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2_t){lo, hi}, bf2_t));
}

// A weight held in f32 as kParts<T> values of T whose sum it is: for operands that must not lose bits.  take_part packs the
// next part of two weights (low half first) and takes it off them.  fp16: rounded, two parts hold 22 bits; bf16: the upper
// half of the f32 number as it is, three parts are all 24 bits exactly (and the conversion is one v_perm).
template <typename T> constexpr int kParts = std::is_same<T, f16_t>::value ? 2 : 3;
template <typename T> __device__ inline uint32_t take_part(float &a, float &b) {
    if constexpr (std::is_same<T, f16_t>::value) {
        const uint32_t w = pack2<T>(a, b);
        const h2_t h = __builtin_bit_cast(h2_t, w);
        a -= (float)h[0];
        b -= (float)h[1];
        return w;
    } else {
        const uint32_t ua = __builtin_bit_cast(uint32_t, a), ub = __builtin_bit_cast(uint32_t, b);
        a -= __builtin_bit_cast(float, ua & 0xFFFF0000u);
        b -= __builtin_bit_cast(float, ub & 0xFFFF0000u);
        return __builtin_amdgcn_perm(ub, ua, 0x07060302u);
    }
}

// 8 int8 (two dwords) -> 8 values of T packed in a U4; exact
template <typename T> __device__ inline U4 i8x8_to_operand(uint32_t w0, uint32_t w1) {
    if constexpr (std::is_same<T, f16_t>::value) {
        // byte b + 128 under an 0x64 high byte is the fp16 number 1024 + (b + 128); subtract 1152
        const h2_t bias = {(_Float16)1152.f, (_Float16)1152.f};
        const uint32_t x0 = w0 ^ 0x80808080u, x1 = w1 ^ 0x80808080u;
        auto two = [&](uint32_t x, uint32_t sel) {
            const h2_t h = __builtin_bit_cast(h2_t, __builtin_amdgcn_perm(0x64646464u, x, sel)) - bias;
            return __builtin_bit_cast(uint32_t, h);
        };
        return U4{two(x0, 0x04010400u), two(x0, 0x04030402u), two(x1, 0x04010400u), two(x1, 0x04030402u)};
    } else {
        // |b| <= 128 has at most 8 significant bits: the upper half of its f32 form is the bf16 value
        auto two = [&](uint32_t w, int sh) {
            const float a = (float)(int8_t)((w >> sh) & 0xFF), b = (float)(int8_t)((w >> (sh + 8)) & 0xFF);
            return __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, b), __builtin_bit_cast(uint32_t, a), 0x07060302u);
        };
        return U4{two(w0, 0), two(w0, 16), two(w1, 0), two(w1, 16)};
    }
}

}  // namespace mynn
