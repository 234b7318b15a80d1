// Matrix products of ordinary size: too many activation rows for the kernels that stream the weights past a few rows
// (gemv.hip, skinny.hip), too few tiles for one round of the 256-row kernel of gemm.hip.
//
//   TG_W8   out = act . T(wq * scale)^T   16-bit activations, int8 weights dequantised WITH the scale (one rounding, as the
//                                         reference's matrix-core path: dequant_matmul_wmma.cuh:65-76)
//   TG_W8S  out = T((act . wq^T) * scale) the same operands, scale after the f32 sum (fewer than 16 rows: dequant_gemv.cuh:12-59)
//   TG_I8   out = T((acc * a_scale) * b_scale), acc = int8 x int8 in exact int32 (QuantizedMatMul)
//
// The weights are read once per row tile, as the int8 they are stored as: no dequantised copy is written or read (a pass of
// 3 bytes per weight that cost more than the product itself below a few hundred rows).  Operand tiles go global -> LDS with
// global_load_lds_dwordx4, NS stages deep.  A K step is 128 bytes of an activation row (64 values of 16 bits, 128 int8).  16-byte
// chunks are placed so that the 128-bit fragment reads of 16 neighbouring rows fall into different LDS banks: row r's chunk c at
// 8r + (c ^ (r/2 & 7)) for 128-byte rows, 4r + (c ^ (r/4 & 3)) for the 64-byte rows of int8 weights against 16-bit activations.
//
// What bounds it: few rows, the latency of the weight stream, which the stages in flight hide (the loads are instructions of
// their own, mfma.h: through the builtin the compiler waited for all of them in every step; bf16, 6 x 4096 x 14336 24.4 -> 18.9 us
// a call, 16 x 4096 x 14336 26.3 -> 20.9); many rows, the issue slots of a SIMD.  An MFMA of 32 clocks leaves room for some five
// vector operations; the conversion of a weight fragment is 14 (fp16) or 20 (bf16) of them, and every further one costs 4 - 6
// clocks more (one or two waves a SIMD, MFMA + 4 operations 33 clocks, + 8 operations 47 - 57).  So a wave of a large tile has 3 - 5
// fragments of activations for each of weights (96 .. 160 rows x 32 or 64 columns: 160 x 256 per workgroup of four waves), the
// conversions, the LDS reads and the loads' requests are pinned between the MFMAs, and a step's bookkeeping is kept short: one
// setting of m0 and one scalar base per operand, fragment addresses that need one addition per MFMA step.  fp16, us a call before /
// now: 300 x 28672 x 4096 115 / 75, 700 x 11264 x 2048 47.5 / 38.5, 500 x 4096 x 14336 81 / 72, 1000 x 28672 x 4096 264 / 236; bf16
// 500 x 28672 x 4096 156 / 118, 700 x 4096 x 14336 133 / 99.
// PIN: not in 64 x 64 with one fragment of each operand a wave, where the order the compiler finds is the better one, together with KM = 2
// (fp16, 300 x 2048 x 2048: pinned 12.8 us a call, KM = 2 12.7, not pinned 12.8, both 11.8; bf16 13.8 / 13.3 / 13.8 / 13.1).
// KM: the waves meet at a barrier every KM steps; 2 helps where a step is short against the meeting (the eight waves of the int8
// 64 x 128 tile, 500 x 4096 x 14336: 55.5 -> 50.6 us together with six stages against three).
//
// When the tiles do not fill the device the K range is split over workgroups.  Each leaves its partial sums in scratch
// memory (agent-scope stores, which go past the XCD's L2) and counts itself in; the last to arrive adds them up in the
// order of the ranges -- the result does not depend on who was last -- and stores the output.  Nobody waits for anybody.
// SEQ: one workgroup takes all ranges of its tile one after the other and adds them up in registers: the same bits without
// scratch memory, for calls that are being captured (a graph may be replayed on any stream and outlive any block).
// It costs the parallelism (us, bf16, captured / not): 6 rows x 4096 x 14352 61 / 18, 6 x 2048 x 2064 13.6 / 8.1, 16 x 4096 x 14336 80 / 21, 100 x
// 4096 x 4096 25 / 16, 300 x 2048 x 5632 32 / 23 (with the steps' loop called in two places, not inlined and its registers in
// memory: 1045, 185, 1961, 588, 770).
#pragma once
#include <type_traits>

#include "gemm_store.h"
#include "kernels.h"
#include "mfma.h"

namespace mynn {

typedef int i4x_t __attribute__((ext_vector_type(4)));
typedef int i16x_t __attribute__((ext_vector_type(16)));

template <int KIND_, int BM_, int BN_, int WM_, int WN_, int NS_, int WPE_, int KM_, bool PIN_ = true>
struct TgTile {
    static constexpr bool PIN = PIN_;
    static constexpr int KIND = KIND_, BM = BM_, BN = BN_, WM = WM_, WN = WN_, NS = NS_, WPE = WPE_, KM = KM_;
    static constexpr int THREADS = WM * WN * 64;
    static constexpr int TI = BM / WM / 32, TJ = BN / WN / 32;
    static constexpr bool WIDE = TI >= 3 || TJ >= 3;
    static constexpr int BROW = KIND == TG_I8 ? 128 : 64;  // bytes of a weight row per K step
    static constexpr int STAGE = BM * 128 + BN * BROW;
    static constexpr int CHA = BM * 8 / THREADS, CHB = BN * (BROW / 16) / THREADS;  // 16-byte chunks per thread
    static constexpr int EST = BN / WN + 8;                                         // store staging row stride
    static constexpr int STORE = WM * WN * 32 * EST * 2;
    static constexpr int LDS = NS * STAGE > STORE + BN * 4 ? NS * STAGE : STORE + BN * 4;  // (column scales above the staging)
    static_assert(BM * 8 % THREADS == 0 && BN * (BROW / 16) % THREADS == 0, "whole load instructions per wave");
};

static __device__ U4 g_tg_zero;  // what the chunks past the end of a row are read from

template <typename T> __device__ inline U4 scale_operand(const U4 &v, float sc);
template <> __device__ inline U4 scale_operand<f16_t>(const U4 &v, float sc) {
    // |w| <= 128 times a 16-bit scale is exact in f32, so this product's one rounding is the rounding of T(w * scale)
    const h2_t s2 = {(_Float16)sc, (_Float16)sc};
    auto m = [&](uint32_t x) { return __builtin_bit_cast(uint32_t, __builtin_bit_cast(h2_t, x) * s2); };
    return U4{m(v.x), m(v.y), m(v.z), m(v.w)};
}
template <> __device__ inline U4 scale_operand<bf16_t>(const U4 &v, float sc) { return v; }  // (see weight_operand)

// 8 int8 weights -> an MFMA operand, scaled or not
template <typename T, bool SCALED> __device__ inline U4 weight_operand(uint32_t w0, uint32_t w1, float sc) {
    if constexpr (!SCALED) return i8x8_to_operand<T>(w0, w1);
    else if constexpr (std::is_same<T, f16_t>::value) return scale_operand<T>(i8x8_to_operand<T>(w0, w1), sc);
    else {
        auto two = [&](uint32_t w, int sh) {
            return pack2<T>((float)(int8_t)((w >> sh) & 0xFF) * sc, (float)(int8_t)((w >> (sh + 8)) & 0xFF) * sc);
        };
        return U4{two(w0, 0), two(w0, 16), two(w1, 0), two(w1, 16)};
    }
}

// TAIL: the rows are not whole K steps, the last one reads zeros past their end
template <typename T, typename G, int EPI, bool TAIL, bool SEQ>
__global__ __launch_bounds__(G::THREADS, G::WPE) void tile_gemm_kernel(const void *A_, const int8_t *B, int M, int N, int K, int ks, T *C,
                                                                      const T *R, const T *a_scale, const T *b_scale,
                                                                      uint64_t *part, int *counter, int32_t *acc_out) {
    constexpr int KIND = G::KIND, BM = G::BM, BN = G::BN, TI = G::TI, TJ = G::TJ, NS = G::NS, BROW = G::BROW;
    constexpr bool I8 = KIND == TG_I8;
    constexpr int EA = I8 ? 1 : 2;
    constexpr int CHA = G::CHA, CHB = G::CHB;
    extern __shared__ __align__(16) char lds[];
    const char *A = (const char *)A_;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / G::WN, wn = wave % G::WN;
    const int wrow = wm * TI * 32, wcol = wn * TJ * 32;

    // Workgroup -> (row tile, K range, column tile).  Consecutive ids go round-robin over the 8 XCDs, so an id is first
    // turned into an index that is contiguous inside an XCD; there the row tiles of a band share the weight tile they
    // multiply by, then come the K ranges, then the columns.
    const int tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
    int tm, tn, kz;
    {
        constexpr int XCD = 8, BAND = 8;
        const int nb = gridDim.x, x = blockIdx.x % XCD, per = nb / XCD, rem = nb % XCD;
        const int l = x * per + min(x, rem) + blockIdx.x / XCD;
        const int side = SEQ ? 1 : ks;  // K ranges side by side
        const int band = l / (BAND * tiles_n * side), in_band = l - band * BAND * tiles_n * side;
        const int rows_here = min(BAND, tiles_m - band * BAND);
        tm = band * BAND + in_band % rows_here;
        const int rest = in_band / rows_here;
        kz = rest % side;
        tn = rest / side;
    }
    const int m0 = __builtin_amdgcn_readfirstlane(tm * BM), n0 = __builtin_amdgcn_readfirstlane(tn * BN);
    const int a_bytes = K * EA;                    // bytes of an activation row; a weight row is K bytes
    const int iters = (a_bytes + 127) / 128;
    int it0, n_it;
    auto range = [&](int z) {  // (gemm_nt_mfma_kernel cuts K in the same places)
        it0 = __builtin_amdgcn_readfirstlane((int)((long)iters * z / ks));  // (the division is done in vector registers)
        n_it = __builtin_amdgcn_readfirstlane((int)((long)iters * (z + 1) / ks)) - it0;
    };
    range(kz);

    // this lane's chunks of each operand tile: LDS position P = (CH * wave + i) * 64 + lane.  Offsets are from 4096 bytes in front of
    // the tile's first row less what load_group_to_lds adds, so that a step's address is a scalar base plus a 32-bit lane offset.
    uint32_t aoff[CHA], boff[CHB];
#pragma unroll
    for (int i = 0; i < CHA; i++) {
        const int P = (CHA * wave + i) * 64 + lane, r = P >> 3;
        aoff[i] = (uint32_t)(min(r, M - 1 - m0) * a_bytes + ((P & 7) ^ ((r >> 1) & 7)) * 16 + 4096 - 1024 * (i % 4));
    }
#pragma unroll
    for (int i = 0; i < CHB; i++) {
        const int P = (CHB * wave + i) * 64 + lane;
        const int r = BROW == 128 ? P >> 3 : P >> 2;
        boff[i] = (uint32_t)(min(r, N - 1 - n0) * K + (BROW == 128 ? (P & 7) ^ ((r >> 1) & 7) : (P & 3) ^ ((r >> 2) & 3)) * 16 + 4096 - 1024 * (i % 4));
    }
    const uint32_t lds0 = lds_offset(lds);
    const char *anext, *bnext;  // the bases of the next step to be requested
    int wanted;                 // its number within the range
    int whole_steps;            // steps below this one lie within the rows
    uint32_t fill;              // the stage it goes to, in bytes
    auto first_request = [&]() {
        whole_steps = it0 + n_it == iters ? n_it - 1 : 1 << 30;
        anext = A + (size_t)m0 * a_bytes + (size_t)it0 * 128 - 4096;
        bnext = (const char *)B + (size_t)n0 * K + (size_t)it0 * BROW - 4096;
        wanted = 0;
        fill = 0;
    };
    // A step's loads in two halves, the activations' and the weights'; past the range the last step once more, never read: it
    // keeps the counts.  at_end: the step may reach past the rows' end.  A lane then picks its address by itself, a dozen instructions a
    // load, so only the steps from whole_steps on are asked for in that way, by a loop of their own (us a call, all steps in that way / those
    // alone: int8, 64 x 4330 x 4000 11.6 / 10.3, 33 x 6496 x 6592 15.6 / 12.8; int8 weights, 300 x 5476 x 7456, fp16 59 / 49, bf16 67 / 49).
    auto request_a = [&](auto at_end) {
        const uint32_t to = lds0 + fill + CHA * wave * 1024;
        if constexpr (decltype(at_end)::value) {
#pragma unroll
            for (int i = 0; i < CHA; i++) {
                const int P = (CHA * wave + i) * 64 + lane;
                load_to_lds((it0 + wanted) * 128 + ((P & 7) ^ ((P >> 4) & 7)) * 16 >= a_bytes ? (const char *)&g_tg_zero : anext + aoff[i] + 1024 * (i % 4), to + i * 1024);
            }
        } else {
            load_group_to_lds<(CHA < 4 ? CHA : 4)>(anext, aoff, to);
            if constexpr (CHA > 4) load_group_to_lds<CHA - 4>(anext, aoff + 4, to + 4096);
        }
    };
    auto request_b = [&](auto at_end) {
        const uint32_t to = lds0 + fill + BM * 128 + CHB * wave * 1024;
        if constexpr (decltype(at_end)::value) {
#pragma unroll
            for (int i = 0; i < CHB; i++) {
                const int P = (CHB * wave + i) * 64 + lane, c = BROW == 128 ? (P & 7) ^ ((P >> 4) & 7) : (P & 3) ^ ((P >> 4) & 3);
                load_to_lds((it0 + wanted) * BROW + c * 16 >= K ? (const char *)&g_tg_zero : bnext + boff[i] + 1024 * (i % 4), to + i * 1024);
            }
        } else {
            load_group_to_lds<(CHB < 4 ? CHB : 4)>(bnext, boff, to);
            if constexpr (CHB > 4) load_group_to_lds<CHB - 4>(bnext, boff + 4, to + 4096);
        }
        const bool more = wanted + 1 < n_it;
        anext += more ? 128 : 0;
        bnext += more ? BROW : 0;
        wanted += more ? 1 : 0;
        fill = fill + G::STAGE == NS * G::STAGE ? 0 : fill + G::STAGE;
    };
    constexpr std::integral_constant<bool, TAIL> end_too;  // steps of any kind
    constexpr std::false_type whole_only;
    auto request = [&]() {
        if (TAIL && wanted >= whole_steps) {
            request_a(end_too);
            request_b(end_too);
        } else {
            request_a(whole_only);
            request_b(whole_only);
        }
    };

    using acc_t = std::conditional_t<I8, i16x_t, f16x_t>;
    using sum_t = std::conditional_t<I8, int32_t, float>;
    acc_t acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; i++)
#pragma unroll
        for (int j = 0; j < TJ; j++)
#pragma unroll
            for (int e = 0; e < 16; e++) acc[i][j][e] = 0;

    // fragment reads: lane l takes row l % 32 of a 32-row tile, and its half g = l / 32 one of two 16-byte chunks (which one
    // depends on the row within the 32 alone)
    const int fr = lane & 31, g = lane >> 5;
    uint32_t abase[4], bbase[4];
    float wsc[TJ];
#pragma unroll
    for (int s = 0; s < 4; s++) {
        abase[s] = 128 * (wrow + fr) + (((2 * s + g) ^ ((fr >> 1) & 7)) << 4);
        bbase[s] = BM * 128 + BROW * (wcol + fr) + (I8 ? ((2 * s + g) ^ ((fr >> 1) & 7)) << 4 : ((s ^ ((fr >> 2) & 3)) << 4) + 8 * g);
    }
#pragma unroll
    for (int j = 0; j < TJ; j++) wsc[j] = KIND == TG_W8 ? Elem<T>::ld(b_scale, min(n0 + wcol + j * 32 + fr, N - 1)) : 0.f;
    // The fragments of one K step: MFMA step s takes chunk 2s + g of the activation row and, of 16-bit kinds, the 8 weights
    // at the same k, half of chunk s -- the order of the 256-row kernel of gemm.hip, so that with one K range a row's sums
    // are the same bits whichever of the two kernels its number of neighbours selects.
    using w_t = std::conditional_t<I8, U4, uint2>;
    struct Frags {
        w_t w[4][TJ];
        U4 a[4][TI];
    };
    auto read = [&](const char *st, Frags &f, int s) {
#pragma unroll
        for (int j = 0; j < TJ; j++)
            f.w[s][j] = *(const w_t *)(st + bbase[s] + j * (32 * BROW));
#pragma unroll
        for (int i = 0; i < TI; i++) f.a[s][i] = *(const U4 *)(st + abase[s] + i * 4096);
    };
    auto convert = [&](const w_t &w, int j) -> U4 {
        if constexpr (I8) return w;
        else return weight_operand<T, KIND == TG_W8>(w.x, w.y, wsc[j]);
    };
    auto multiply = [&](const U4 *fb, const U4 *fa) {
#pragma unroll
        for (int j = 0; j < TJ; j++)
#pragma unroll
            for (int i = 0; i < TI; i++) {
                if constexpr (I8)
                    acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i4x_t, fb[j]), __builtin_bit_cast(i4x_t, fa[i]), acc[i][j], 0, 0, 0);
                else acc[i][j] = Mfma<T>::run(fb[j], fa[i], acc[i][j]);
            }
    };

    // One barrier per KM K steps: behind it the tiles of these steps are whole (every wave has waited for its own share of
    // the loads) and the stages of the KM steps before are free.  While MFMA step s of a K step multiplies, the weights of the
    // MFMA step after it are converted, the fragments of the next K step's s are read and a quarter of a later step's loads is
    // requested: the order is pinned, or the scheduler bunches the reads and the conversions up in front of the MFMAs.
    constexpr int KM = G::KM, AHEAD = NS - KM;  // steps whose loads are in flight ahead of the one that is read
    static_assert(NS % KM == 0 && AHEAD >= KM, "whole groups of stages");
    int it;
    uint32_t cur;  // the stage that is read, in bytes
    U4 fb[2][TJ];
    auto meet = [&]() {
        constexpr int VM = (AHEAD - KM) * (CHA + CHB);  // loads that may stay in flight: those of the later stages
        static_assert(VM < 64, "a counter of six bits");
        __builtin_amdgcn_s_waitcnt((VM & 15) | (VM >> 4) << 14 | 0x70);  // vmcnt(VM) lgkmcnt(0)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto advance = [&]() {
        cur = cur + G::STAGE == NS * G::STAGE ? 0 : cur + G::STAGE;
        ++it;
    };
    // the step in `now` is multiplied, the one in stage cur read into `next`
    auto step = [&](const Frags &now, Frags &next, auto first, auto at_end) {
        if constexpr (decltype(first)::value) meet();
        const char *st = lds + cur;
        auto quarter = [&](auto part) {
            constexpr int s = decltype(part)::value;
            if constexpr (s < 2) {
                read(st, next, 2 * s);
                read(st, next, 2 * s + 1);
            } else if constexpr (s == 2) request_a(at_end);
            else request_b(at_end);
            multiply(fb[s & 1], now.a[s]);
#pragma unroll
            for (int j = 0; j < TJ; j++) fb[(s + 1) & 1][j] = convert(s < 3 ? now.w[(s + 1) & 3][j] : next.w[0][j], j);
            if constexpr (!G::PIN) return;
            constexpr int NM = TI * TJ, RPM = s < 2 ? (2 * (TI + TJ) + NM - 1) / NM : 0, VPM = I8 ? 1 : (std::is_same<T, f16_t>::value ? 16 : 22) / TI;
#pragma unroll
            for (int n = 0; n < NM; n++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                if constexpr (RPM > 0) __builtin_amdgcn_sched_group_barrier(0x100, RPM, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, VPM, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        quarter(std::integral_constant<int, 0>{});
        quarter(std::integral_constant<int, 1>{});
        quarter(std::integral_constant<int, 2>{});
        quarter(std::integral_constant<int, 3>{});
        if constexpr (!G::PIN) __builtin_amdgcn_sched_barrier(0);
        advance();
    };
    auto last = [&](const Frags &now) {
#pragma unroll
        for (int s = 0; s < 4; s++) {
            multiply(fb[s & 1], now.a[s]);
            if (s < 3)
#pragma unroll
                for (int j = 0; j < TJ; j++) fb[(s + 1) & 1][j] = convert(now.w[(s + 1) & 3][j], j);
        }
    };
    constexpr std::true_type whole;
    constexpr std::integral_constant<bool, KM == 1> second;
    auto one_range_step = [&]() {
        first_request();
#pragma unroll
        for (int s = 0; s < AHEAD; s++) request();
        cur = 0;
        it = 0;
        Frags f0, f1;
        meet();
#pragma unroll
        for (int s = 0; s < 4; s++) read(lds, f0, s);
        request();
        advance();
#pragma unroll
        for (int j = 0; j < TJ; j++) fb[0][j] = convert(f0.w[0][j], j);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (TAIL) {
            while (it + 1 < n_it && wanted + 1 < whole_steps) {
                step(f0, f1, second, whole_only);
                step(f1, f0, whole, whole_only);
            }
        }
        while (it + 1 < n_it) {
            step(f0, f1, second, end_too);
            step(f1, f0, whole, end_too);
        }
        if (it < n_it) {
            step(f0, f1, second, end_too);
            last(f1);
        } else last(f0);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the repeats of the last step too, before LDS is reused
        __syncthreads();
    };
    // Tiles of many MFMAs per step read ahead less, one MFMA step of activations and two of weights: a whole K step twice would not
    // fit the registers.  The waves meet in the middle of a step t, behind which step t + 1 is whole and the stage of t - 1 free.
    auto one_range_wide = [&]() {
        constexpr int KEEP = (NS - 3) * (CHA + CHB);  // loads of the steps after t + 1
        static_assert(!G::WIDE || (NS >= 3 && KM == 1 && KEEP < 64), "");
        w_t w[2][TJ];
        U4 a[2][TI];
        auto read_a = [&](const char *st, auto s) {
            constexpr int S = decltype(s)::value & 3;
#pragma unroll
            for (int i = 0; i < TI; i++) a[S & 1][i] = *(const U4 *)(st + abase[S] + i * 4096);
        };
        auto read_w = [&](const char *st, auto s) {
            constexpr int S = decltype(s)::value & 3;
#pragma unroll
            for (int j = 0; j < TJ; j++) w[S & 1][j] = *(const w_t *)(st + bbase[S] + j * (32 * BROW));
        };
        const char *st = lds, *nx = lds;  // the stages of this step and of the next
        auto quarter = [&](auto s, auto half, auto at_end) {
            constexpr int S = decltype(s)::value;
            read_a(S < 3 ? st : nx, std::integral_constant<int, S + 1>{});
            read_w(S < 2 ? st : nx, std::integral_constant<int, S + 2>{});
            if constexpr (decltype(half)::value == 1) request_a(at_end);
            if constexpr (decltype(half)::value == 2) request_b(at_end);
            multiply(fb[S & 1], a[S & 1]);
#pragma unroll
            for (int j = 0; j < TJ; j++) fb[(S + 1) & 1][j] = convert(w[(S + 1) & 1][j], j);
            constexpr int NM = TI * TJ, RPM = (TI + TJ + NM - 1) / NM, VPM = I8 ? 1 : ((std::is_same<T, f16_t>::value ? 14 : 20) + TI - 1) / TI;
#pragma unroll
            for (int n = 0; n < NM; n++) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, RPM, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, VPM, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        constexpr std::integral_constant<int, 0> q0;
        constexpr std::integral_constant<int, 1> q1;
        constexpr std::integral_constant<int, 2> q2;
        constexpr std::integral_constant<int, 3> q3;
        auto meet_wide = [&](auto keep) {
            constexpr int VM = decltype(keep)::value < 0 ? 0 : decltype(keep)::value;
            __builtin_amdgcn_s_waitcnt((VM & 15) | (VM >> 4) << 14 | 0xF70);  // vmcnt(VM); the reads of t - 1 have been multiplied
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        first_request();
#pragma unroll
        for (int s = 0; s < NS - 1; s++) request();
        cur = 0;
        it = 0;
        meet_wide(std::integral_constant<int, (NS - 2) * (CHA + CHB)>{});
        read_a(st, q0);
        read_w(st, q0);
        read_w(st, q1);
#pragma unroll
        for (int j = 0; j < TJ; j++) fb[0][j] = convert(w[0][j], j);
        __builtin_amdgcn_sched_barrier(0);
        quarter(q0, q0, whole_only);
        quarter(q1, q0, whole_only);
        auto round = [&](auto at_end) {
            meet_wide(std::integral_constant<int, KEEP>{});
            cur = cur + G::STAGE == NS * G::STAGE ? 0 : cur + G::STAGE;
            nx = lds + cur;
            quarter(q2, q1, at_end);
            quarter(q3, q2, at_end);
            st = nx;
            quarter(q0, q0, at_end);
            quarter(q1, q0, at_end);
        };
        if constexpr (TAIL) {
            for (; it + 1 < n_it && wanted < whole_steps; ++it) round(whole_only);
        }
        for (; it + 1 < n_it; ++it) round(end_too);
        nx = st;  // (reads past the last step stay within it and are not used)
        quarter(q2, q0, whole_only);
        quarter(q3, q0, whole_only);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    };
    auto one_range = [&]() {
        if constexpr (G::WIDE) one_range_wide();
        else one_range_step();
    };
    if constexpr (SEQ) {
        // (one_range is called in one place, or it is no longer inlined and its registers are memory)
        acc_t sum[TI][TJ];
        for (int z = 0; z < ks; z++) {
            if (z) {
                range(z);
#pragma unroll
                for (int i = 0; i < TI; i++)
#pragma unroll
                    for (int j = 0; j < TJ; j++)
#pragma unroll
                        for (int e = 0; e < 16; e++) acc[i][j][e] = 0;
            }
            one_range();
#pragma unroll
            for (int i = 0; i < TI; i++)
#pragma unroll
                for (int j = 0; j < TJ; j++)
#pragma unroll
                    for (int e = 0; e < 16; e++) sum[i][j][e] = z ? sum[i][j][e] + acc[i][j][e] : acc[i][j][e];
        }
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int j = 0; j < TJ; j++) acc[i][j] = sum[i][j];
    } else one_range();

    if (!SEQ && ks > 1) {
        // partial sums, two per word, [range][(i, j), pair][thread]
        const size_t tile = (size_t)tn * tiles_m + tm;
        constexpr int WORDS = TI * TJ * 8;
        uint64_t *p0 = part + tile * ks * (WORDS * G::THREADS) + tid;
        uint64_t *mine = p0 + (size_t)kz * (WORDS * G::THREADS);
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int j = 0; j < TJ; j++)
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    const sum_t lo = acc[i][j][2 * e], hi = acc[i][j][2 * e + 1];
                    const uint64_t v = (uint64_t)__builtin_bit_cast(uint32_t, lo) | ((uint64_t)__builtin_bit_cast(uint32_t, hi) << 32);
                    __hip_atomic_store(mine + ((i * TJ + j) * 8 + e) * G::THREADS, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // written through before this workgroup counts itself in
        __syncthreads();
        int *flag = (int *)lds;
        if (tid == 0) {
            const int before = __hip_atomic_fetch_add(counter + tile, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (before == ks - 1) __hip_atomic_store(counter + tile, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // ready for the next launch
            *flag = before;
        }
        __syncthreads();
        const bool last = *flag == ks - 1;
        __syncthreads();
        if (!last) return;
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int j = 0; j < TJ; j++) {
                uint64_t v[8];
                auto fetch = [&](int s) {
#pragma unroll
                    for (int e = 0; e < 8; e++)
                        v[e] = __hip_atomic_load(p0 + (size_t)s * (WORDS * G::THREADS) + ((i * TJ + j) * 8 + e) * G::THREADS, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                };
                fetch(0);
#pragma unroll
                for (int e = 0; e < 8; e++) {
                    acc[i][j][2 * e] = __builtin_bit_cast(sum_t, (uint32_t)v[e]);
                    acc[i][j][2 * e + 1] = __builtin_bit_cast(sum_t, (uint32_t)(v[e] >> 32));
                }
                for (int s = 1; s < ks; s++) {
                    fetch(s);
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        acc[i][j][2 * e] += __builtin_bit_cast(sum_t, (uint32_t)v[e]);
                        acc[i][j][2 * e + 1] += __builtin_bit_cast(sum_t, (uint32_t)(v[e] >> 32));
                    }
                }
            }
    }

    if constexpr (I8) {
        constexpr bool F32 = sizeof(T) == 4;  // (f32 scales and output: stored as they lie, like the integer sums)
        if (acc_out || F32) {
#pragma unroll
            for (int i = 0; i < TI; i++)
#pragma unroll
                for (int j = 0; j < TJ; j++)
#pragma unroll
                    for (int e = 0; e < 16; e++) {
                        const int row = m0 + wrow + i * 32 + fr, col = n0 + wcol + j * 32 + 8 * (e >> 2) + 4 * g + (e & 3);
                        if (row >= M || col >= N) continue;
                        if (acc_out) acc_out[(size_t)row * N + col] = acc[i][j][e];
                        if (F32 && C) Elem<T>::st(C, (size_t)row * N + col, ((float)acc[i][j][e] * Elem<T>::ld(a_scale, row)) * Elem<T>::ld(b_scale, col));
                    }
        }
        if (F32 || !C) return;
    }
    if constexpr (sizeof(T) == 4) {
    } else if constexpr (KIND == TG_W8) {
        gemm_store<T, G, EPI>([&](int i, int j, int e) { return acc[i][j][e]; }, (uint16_t *)lds, C, R, M, N, m0, n0, wrow, wcol, lane, wave);
    } else {
        // the column scales of the tile as f32 in LDS above the store's patches, the row scales in registers
        float *bs = (float *)(lds + G::STORE);
        for (int c = tid; c < BN; c += G::THREADS) bs[c] = n0 + c < N ? Elem<T>::ld(b_scale, n0 + c) : 0.f;
        float asc[TI];
#pragma unroll
        for (int i = 0; i < TI; i++) asc[i] = I8 ? Elem<T>::ld(a_scale, min(m0 + wrow + i * 32 + fr, M - 1)) : 1.f;
        __syncthreads();
        const float *bw = bs + wcol + 4 * g;
        gemm_store<T, G, EPI>(
            [&](int i, int j, int e) {
                const float b = bw[j * 32 + 8 * (e >> 2) + (e & 3)];
                if constexpr (I8) return ((float)acc[i][j][e] * asc[i]) * b;
                else return acc[i][j][e] * b;
            },
            (uint16_t *)lds, C, R, M, N, m0, n0, wrow, wcol, lane, wave);
    }
}

struct TgArgs {
    void *out;
    int32_t *acc_out;
    const void *act;
    const int8_t *wq;
    const void *a_scale, *w_scale, *res;
    int M, N, K, ks;
    bool seq;
    uint64_t *part;
    int *counters;
    hipStream_t s;
};

template <typename T, typename G, int EPI, bool TAIL, bool SEQ = false> static int tg_go(const TgArgs &p) {
    static bool lds_set = false;
    if (!lds_set && G::LDS > 64 * 1024) {
        MYNN_HIP(hipFuncSetAttribute((const void *)tile_gemm_kernel<T, G, EPI, TAIL, SEQ>, hipFuncAttributeMaxDynamicSharedMemorySize, G::LDS));
        lds_set = true;
    }
    const int tiles = ((p.M + G::BM - 1) / G::BM) * ((p.N + G::BN - 1) / G::BN);
    MYNN_LAUNCH((tile_gemm_kernel<T, G, EPI, TAIL, SEQ>), dim3(SEQ ? tiles : tiles * p.ks), dim3(G::THREADS), G::LDS, p.s, p.act, p.wq, p.M, p.N, p.K, p.ks, (T *)p.out,
                (const T *)p.res, (const T *)p.a_scale, (const T *)p.w_scale, p.part, p.counters, p.acc_out);
    return launch_status("tile_gemm_kernel");
}
template <typename T, typename G> static int tg_epi(const TgArgs &p, int epi) {
    const bool tail = (size_t)p.K * (G::KIND == TG_I8 ? 1 : 2) % 128 != 0;
    if constexpr (G::KIND != TG_I8 && G::TI * G::TJ <= 4) {  // (two sets of sums fit the registers: tg_choose)
        if (p.seq) return tail ? tg_go<T, G, GEMM_PLAIN, true, true>(p) : tg_go<T, G, GEMM_PLAIN, false, true>(p);
    } else MYNN_REQUIRE(!p.seq, MYNN_ERR_UNSUPPORTED, "tile_gemm: a tile of %d x %d has no form that takes its ranges one after the other", G::BM, G::BN);
    if constexpr (G::KIND == TG_W8S || sizeof(T) == 4)
        return tail ? tg_go<T, G, GEMM_PLAIN, true>(p) : tg_go<T, G, GEMM_PLAIN, false>(p);
    else {
        if (epi == GEMM_RESIDUAL) return tail ? tg_go<T, G, GEMM_RESIDUAL, true>(p) : tg_go<T, G, GEMM_RESIDUAL, false>(p);
        if (epi == GEMM_SWIGLU_PAIRS_EXP) return tail ? tg_go<T, G, GEMM_SWIGLU_PAIRS_EXP, true>(p) : tg_go<T, G, GEMM_SWIGLU_PAIRS_EXP, false>(p);
        if constexpr (G::KIND == TG_W8) {
            if (epi == GEMM_SWIGLU_PAIRS) return tail ? tg_go<T, G, GEMM_SWIGLU_PAIRS, true>(p) : tg_go<T, G, GEMM_SWIGLU_PAIRS, false>(p);
        }
        return tail ? tg_go<T, G, GEMM_PLAIN, true>(p) : tg_go<T, G, GEMM_PLAIN, false>(p);
    }
}
// by kind and type, a translation unit each (tile_gemm_f16.hip, tile_gemm_bf16.hip, tile_gemm_i8.hip)
template <typename T> int tg_launch_w8(int kind, int tile, const TgArgs &p, int epi);
template <typename T> int tg_launch_i8(int tile, const TgArgs &p, int epi);

}  // namespace mynn
