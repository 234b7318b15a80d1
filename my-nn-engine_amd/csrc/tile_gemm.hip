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
// global_load_lds_dwordx4, NS stages deep: with this few workgroups per CU what bounds the product is the latency of the
// weight stream, and the stages in flight are what hides it.  A K step is 128 bytes of an activation row (64 values of 16
// bits, 128 int8); the waves meet at a barrier every KM steps.  KM = 2 where a step is long enough that the meeting, not
// the load, is what it waits for: 64 x 128 (500 x 11264 x 2048 30.5 -> 29.9 us fp16, 300 rows bf16 26.4 -> 24.3) and the
// eight waves of 128 x 128 (1000 rows 44.5 -> 43.4); smaller tiles do not change, 128 x 128 of int8 does not either.
// int8 takes eight waves and six stages where a CU gets one workgroup (64 x 128, 500 x 4096 x 14336: 55.5 -> 50.6 us against
// three stages; 128 x 128 in two K ranges 46.2 -> 43.8 against four waves), four waves and two workgroups otherwise.  16-byte chunks are placed so that the 128-bit fragment reads of 16 neighbouring rows fall into
// different LDS banks: row r's chunk c at 8r + (c ^ (r/2 & 7)) for 128-byte rows, 4r + (c ^ (r/4 & 3)) for the 64-byte
// rows of int8 weights against 16-bit activations.
//
// When the tiles do not fill the device the K range is split over workgroups.  Each leaves its partial sums in scratch
// memory (agent-scope stores, which go past the XCD's L2) and counts itself in; the last to arrive adds them up in the
// order of the ranges -- the result does not depend on who was last -- and stores the output.  Nobody waits for anybody.
// SEQ: one workgroup takes all ranges of its tile one after the other and adds them up in registers: the same bits without
// scratch memory, for calls that are being captured (a graph may be replayed on any stream and outlive any block).
// It costs the parallelism: bf16, 6 rows x 4096 x 14336 109 us against 25, 6 x 2048 x 2048 14.3 against 8.2, 100 x 4096 x 4096
// 29 against 17.
#include <algorithm>
#include <type_traits>

#include "gemm_store.h"
#include "kernels.h"
#include "mfma.h"

namespace mynn {

typedef int i4x_t __attribute__((ext_vector_type(4)));
typedef int i16x_t __attribute__((ext_vector_type(16)));

template <int KIND_, int BM_, int BN_, int WM_, int WN_, int NS_, int WPE_, int KM_>
struct TgTile {
    static constexpr int KIND = KIND_, BM = BM_, BN = BN_, WM = WM_, WN = WN_, NS = NS_, WPE = WPE_, KM = KM_;
    static constexpr int THREADS = WM * WN * 64;
    static constexpr int TI = BM / WM / 32, TJ = BN / WN / 32;
    static constexpr int BROW = KIND == TG_I8 ? 128 : 64;  // bytes of a weight row per K step
    static constexpr int STAGE = BM * 128 + BN * BROW;
    static constexpr int CHA = BM * 8 / THREADS, CHB = BN * (BROW / 16) / THREADS;  // 16-byte chunks per thread
    static constexpr int EST = BN / WN + 8;                                         // store staging row stride
    static constexpr int STORE = WM * WN * 32 * EST * 2;
    static constexpr int LDS = NS * STAGE > STORE + BN * 4 ? NS * STAGE : STORE + BN * 4;  // (column scales above the staging)
    static_assert(BM * 8 % THREADS == 0 && BN * (BROW / 16) % THREADS == 0, "whole load instructions per wave");
};

__device__ U4 g_tg_zero;  // what the chunks past the end of a row are read from

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
    // (pinned by hand for int8, 10 - 15 % at 128 x 256, and for the eight-wave fp tile, 4 - 7 %; the others lose by it)
    constexpr bool MIX = I8 || (TI == 2 && TJ == 1 && G::THREADS == 512);
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
    const int m0 = tm * BM, n0 = tn * BN;
    const int a_bytes = K * EA;                    // bytes of an activation row; a weight row is K bytes
    const int iters = (a_bytes + 127) / 128;
    int it0, n_it;
    auto range = [&](int z) {  // (gemm_nt_mfma_kernel cuts K in the same places)
        it0 = (int)((long)iters * z / ks);
        n_it = (int)((long)iters * (z + 1) / ks) - it0;
    };
    range(kz);

    // this lane's chunks of each operand tile: LDS position P = (CH * wave + i) * 64 + lane.  Offsets are from the tile's
    // first row, so that a step's address is a scalar base plus a 32-bit lane offset.
    uint32_t aoff[CHA], boff[CHB];
#pragma unroll
    for (int i = 0; i < CHA; i++) {
        const int P = (CHA * wave + i) * 64 + lane, r = P >> 3;
        aoff[i] = (uint32_t)(min(r, M - 1 - m0) * a_bytes + ((P & 7) ^ ((r >> 1) & 7)) * 16);
    }
#pragma unroll
    for (int i = 0; i < CHB; i++) {
        const int P = (CHB * wave + i) * 64 + lane;
        const int r = BROW == 128 ? P >> 3 : P >> 2;
        boff[i] = (uint32_t)(min(r, N - 1 - n0) * K + (BROW == 128 ? (P & 7) ^ ((r >> 1) & 7) : (P & 3) ^ ((r >> 2) & 3)) * 16);
    }
    const char *a_tile = A + (size_t)m0 * a_bytes, *b_tile = (const char *)B + (size_t)n0 * K;
    auto dma = [&](const char *src, char *dst) {  // (dst is wave-uniform; the lane's 16 bytes are implicit)
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)src, (__attribute__((address_space(3))) void *)dst, 16, 0, 0);
    };
    auto issue = [&](int it, char *st) {
        it = it0 + min(it, n_it - 1);  // (past the range: a repeat of the last step, never read; it keeps the counts)
        const char *ab = a_tile + (size_t)it * 128, *bb = b_tile + (size_t)it * BROW;
        char *ad = st + CHA * wave * 1024, *bd = st + BM * 128 + CHB * wave * 1024;
        const char *zero = (const char *)&g_tg_zero;
#pragma unroll
        for (int i = 0; i < CHA; i++) {
            const char *p = ab + aoff[i];
            const int P = (CHA * wave + i) * 64 + lane;
            if (TAIL && it * 128 + ((P & 7) ^ ((P >> 4) & 7)) * 16 >= a_bytes) p = zero;
            dma(p, ad + i * 1024);
        }
#pragma unroll
        for (int i = 0; i < CHB; i++) {
            const char *p = bb + boff[i];
            const int P = (CHB * wave + i) * 64 + lane, c = BROW == 128 ? (P & 7) ^ ((P >> 4) & 7) : (P & 3) ^ ((P >> 4) & 3);
            if (TAIL && it * BROW + c * 16 >= K) p = zero;
            dma(p, bd + i * 1024);
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

    // fragment reads: lane l takes row l % 32 of a 32-row tile, and its half g = l / 32 one of two 16-byte chunks
    const int fr = lane & 31, g = lane >> 5;
    int abase[TI], aswz[TI], bbase[TJ], bswz[TJ];
    float wsc[TJ];
#pragma unroll
    for (int i = 0; i < TI; i++) {
        const int r = wrow + i * 32 + fr;
        abase[i] = 128 * r;
        aswz[i] = (r >> 1) & 7;
    }
#pragma unroll
    for (int j = 0; j < TJ; j++) {
        const int r = wcol + j * 32 + fr;
        bbase[j] = BM * 128 + BROW * r;
        bswz[j] = BROW == 128 ? (r >> 1) & 7 : (r >> 2) & 3;
        wsc[j] = KIND == TG_W8 ? Elem<T>::ld(b_scale, min(n0 + r, N - 1)) : 0.f;
    }
    // The fragments of one K step: MFMA step s takes chunk 2s + g of the activation row and, of 16-bit kinds, the 8 weights
    // at the same k, half of chunk s -- the order of the 256-row kernel of gemm.hip, so that with one K range a row's sums
    // are the same bits whichever of the two kernels its number of neighbours selects.
    using w_t = std::conditional_t<I8, U4, uint2>;
    struct Frags {
        w_t w[4][TJ];
        U4 a[4][TI];
    };
    auto read = [&](const char *st, Frags &f) {
#pragma unroll
        for (int s = 0; s < 4; s++) {
#pragma unroll
            for (int j = 0; j < TJ; j++)
                f.w[s][j] = *(const w_t *)(st + bbase[j] + (((I8 ? 2 * s + g : s) ^ bswz[j]) << 4) + (I8 ? 0 : 8 * g));
#pragma unroll
            for (int i = 0; i < TI; i++) f.a[s][i] = *(const U4 *)(st + abase[i] + (((2 * s + g) ^ aswz[i]) << 4));
        }
    };
    auto multiply = [&](const Frags &f) {
#pragma unroll
        for (int s = 0; s < 4; s++)
#pragma unroll
            for (int j = 0; j < TJ; j++) {
                U4 fb;
                if constexpr (I8) fb = f.w[s][j];
                else fb = weight_operand<T, KIND == TG_W8>(f.w[s][j].x, f.w[s][j].y, wsc[j]);
#pragma unroll
                for (int i = 0; i < TI; i++) {
                    if constexpr (I8)
                        acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i4x_t, fb), __builtin_bit_cast(i4x_t, f.a[s][i]), acc[i][j], 0, 0, 0);
                    else acc[i][j] = Mfma<T>::run(fb, f.a[s][i], acc[i][j]);
                }
            }
    };

    // One barrier per KM K steps: behind it the tiles of these steps are whole (every wave has waited for its own share of
    // the loads) and the stages of the KM steps before are free.  The fragments of a step are read while the step before
    // multiplies, so that neither the barrier nor the LDS latency is in front of the MFMAs.
    constexpr int KM = G::KM, AHEAD = NS - KM;  // steps whose loads are in flight ahead of the one that is read
    static_assert(NS % KM == 0 && AHEAD >= KM, "whole groups of stages");
    int cur, fill, it;
    auto fetch = [&](Frags &f, auto first) {
        if constexpr (decltype(first)::value) {
            constexpr int VM = (AHEAD - KM) * (CHA + CHB);  // loads that may stay in flight: those of the later stages
            static_assert(VM < 64, "a counter of six bits");
            __builtin_amdgcn_s_waitcnt((VM & 15) | (VM >> 4) << 14 | 0x70);  // vmcnt(VM) lgkmcnt(0)
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        }
        read(lds + cur * G::STAGE, f);
        issue(it + AHEAD, lds + fill * G::STAGE);
        cur = cur + 1 == NS ? 0 : cur + 1;
        fill = fill + 1 == NS ? 0 : fill + 1;
        ++it;
        if constexpr (!MIX) __builtin_amdgcn_sched_barrier(0);
    };
    // the order inside a step where it is pinned: reads, copies and conversions between the MFMAs
    auto end_of_step = [&]() {
        if constexpr (MIX) {
            constexpr int NM = 4 * TI * TJ, RPM = (4 * (TI + TJ) + NM - 1) / NM, DPM = (CHA + CHB + NM - 1) / NM;
#pragma unroll
            for (int n = 0; n < NM; n++) {
                __builtin_amdgcn_sched_group_barrier(0x100, RPM, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, I8 ? 1 : 4, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x010, DPM, 0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr std::true_type whole;
    constexpr std::integral_constant<bool, KM == 1> second;
    auto one_range = [&]() {
#pragma unroll
        for (int s = 0; s < AHEAD; s++) issue(s, lds + s * G::STAGE);
        cur = 0;
        fill = AHEAD;
        it = 0;
        Frags f0, f1;
        fetch(f0, whole);
        __builtin_amdgcn_sched_barrier(0);
        while (it + 1 < n_it) {
            fetch(f1, second);
            multiply(f0);
            end_of_step();
            fetch(f0, whole);
            multiply(f1);
            end_of_step();
        }
        if (it < n_it) {
            fetch(f1, second);
            multiply(f0);
            multiply(f1);
        } else multiply(f0);
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the repeats of the last step too, before LDS is reused
        __syncthreads();
    };
    one_range();
    if constexpr (SEQ) {
        acc_t sum[TI][TJ];
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int j = 0; j < TJ; j++) sum[i][j] = acc[i][j];
        for (int z = 1; z < ks; z++) {
#pragma unroll
            for (int i = 0; i < TI; i++)
#pragma unroll
                for (int j = 0; j < TJ; j++)
#pragma unroll
                    for (int e = 0; e < 16; e++) acc[i][j][e] = 0;
            range(z);
            one_range();
#pragma unroll
            for (int i = 0; i < TI; i++)
#pragma unroll
                for (int j = 0; j < TJ; j++)
#pragma unroll
                    for (int e = 0; e < 16; e++) sum[i][j][e] += acc[i][j][e];
        }
#pragma unroll
        for (int i = 0; i < TI; i++)
#pragma unroll
            for (int j = 0; j < TJ; j++) acc[i][j] = sum[i][j];
    }

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

// ---- which tile, and over how many K ranges.
// The time of a launch, in microseconds, fitted per tile to measured times of the linear layers of the benchmark's models
// and others (every tile at 1 .. 12 ranges):
//
//   t = launch + steps per range * (a * rounds + b * workgroups on the fullest CU) + g * further workgroups + e * ranges
//       + partial sums at 4 TB/s
//
// a: what a step costs a CU however few workgroups it holds (latency); b: what each resident workgroup adds (LDS, MFMA and
// dequantisation work); rounds: how often a CU takes a new set of workgroups; g: what every workgroup on the fullest CU but
// the first adds outside its steps (ramp and store).  Never less than the weights' bytes at 4.6 TB/s or the tiles'
// operations at the rate the tile keeps up in long launches (padding included).  From 256 rows on the constants are those
// that, over some 250 shapes per type, choose best (not those that predict best: some tiles have a `g` that only says that they
// are never taken for more than one workgroup per CU); launches of fewer rows, one or two workgroups per CU and bound by
// latency, keep a fit of their own.  Choosing by it, and by the models of gemm.hip against the 256-row kernels, is 1 % above
// the best measured choice on average (1050 shapes, 2 <= M <= 8192; 33 of them by more than 10 %, 24 % at worst,
// profiles/tile_gemm_plans.csv has them); without ranges 16-bit products of fewer than 256 rows would take 1.6 times as long
// (4.4 at worst) and int8 ones 1.07 times.  (Two columns where the conversion of the weights costs differ: it is 14 vector
// operations per 8 fp16 weights, 20 per 8 bf16 weights.)
struct TgCost {
    int bm, bn, per_cu;  // rows and columns of the tile, workgroups a CU holds
    float launch[2], a[2], b[2], e[2], g[2], rate[2];  // [0] fp16, [1] bf16; rate: 10^9 operations per microsecond
};
// (the order of the tiles in tg_launch)
constexpr TgCost kTgW8Few[] = {
    {32, 64, 3, {2.85f, 3.26f}, {0.308f, 0.311f}, {0.070f, 0.076f}, {0.53f, 0.47f}, {0.0f, 0.0f}, {0.93f, 0.88f}},
    {32, 128, 3, {2.95f, 3.26f}, {0.241f, 0.254f}, {0.150f, 0.145f}, {0.67f, 0.66f}, {0.0f, 0.0f}, {0.93f, 0.88f}},
    {64, 64, 2, {3.24f, 3.67f}, {0.237f, 0.236f}, {0.131f, 0.141f}, {0.62f, 0.60f}, {0.0f, 0.0f}, {0.93f, 0.88f}},
    {64, 128, 2, {2.87f, 3.61f}, {0.296f, 0.313f}, {0.165f, 0.147f}, {1.07f, 1.06f}, {0.0f, 0.0f}, {0.93f, 0.88f}},
    {128, 128, 1, {4.17f, 5.17f}, {0.281f, 0.312f}, {0.234f, 0.267f}, {0.95f, 0.90f}, {0.0f, 0.0f}, {0.93f, 0.88f}},
    {128, 128, 2, {4.51f, 5.83f}, {0.231f, 0.319f}, {0.323f, 0.316f}, {1.65f, 1.65f}, {0.0f, 0.0f}, {0.93f, 0.88f}},
};
constexpr TgCost kTgW8[] = {
    {32, 64, 3, {2.84f, 3.17f}, {0.308f, 0.300f}, {0.062f, 0.066f}, {0.41f, 0.42f}, {0.0f, 0.0f}, {0.77f, 0.37f}},
    {32, 128, 3, {2.07f, 2.89f}, {0.322f, 0.254f}, {0.105f, 0.148f}, {0.62f, 0.62f}, {0.0f, 0.0f}, {0.63f, 0.94f}},
    {64, 64, 2, {2.96f, 3.84f}, {0.254f, 0.239f}, {0.110f, 0.122f}, {0.79f, 0.72f}, {0.5f, 0.0f}, {0.94f, 1.41f}},
    {64, 128, 2, {2.81f, 3.22f}, {0.342f, 0.327f}, {0.153f, 0.169f}, {0.69f, 0.76f}, {0.0f, 0.0f}, {0.71f, 0.72f}},
    {128, 128, 1, {3.70f, 5.54f}, {0.309f, 0.317f}, {0.240f, 0.282f}, {0.29f, 2.88f}, {32.0f, 35.0f}, {0.88f, 0.64f}},
    {128, 128, 2, {4.53f, 5.49f}, {0.234f, 0.426f}, {0.306f, 0.324f}, {3.14f, 1.06f}, {2.5f, 0.5f}, {0.88f, 0.80f}},
};
constexpr TgCost kTgW8S[] = {
    {32, 32, 3, {2.42f, 2.26f}, {0.300f, 0.350f}, {0.049f, 0.024f}, {0.65f, 0.71f}, {0.0f, 0.0f}, {0.93f, 0.88f}},
    {32, 64, 3, {2.26f, 2.02f}, {0.266f, 0.320f}, {0.101f, 0.067f}, {0.68f, 0.73f}, {0.0f, 0.0f}, {0.93f, 0.88f}},
    {32, 128, 3, {1.92f, 1.71f}, {0.229f, 0.245f}, {0.177f, 0.166f}, {1.00f, 1.05f}, {0.0f, 0.0f}, {0.93f, 0.88f}},
};
constexpr TgCost kTgI8Few[] = {
    {32, 64, 2, {3.61f, 3.61f}, {0.001f, 0.001f}, {0.179f, 0.179f}, {0.63f, 0.63f}, {0.0f, 0.0f}, {1.85f, 1.85f}},
    {64, 64, 1, {3.28f, 3.28f}, {0.146f, 0.146f}, {0.096f, 0.096f}, {0.93f, 0.93f}, {0.0f, 0.0f}, {1.85f, 1.85f}},
    {64, 128, 1, {3.54f, 3.54f}, {0.190f, 0.190f}, {0.141f, 0.141f}, {0.80f, 0.80f}, {0.0f, 0.0f}, {1.85f, 1.85f}},
    {64, 128, 2, {3.47f, 3.47f}, {0.101f, 0.101f}, {0.271f, 0.271f}, {1.12f, 1.12f}, {0.0f, 0.0f}, {1.85f, 1.85f}},
    {128, 128, 1, {4.44f, 4.44f}, {0.244f, 0.244f}, {0.197f, 0.197f}, {0.92f, 0.92f}, {0.0f, 0.0f}, {1.85f, 1.85f}},
    {128, 256, 1, {6.13f, 6.13f}, {0.377f, 0.377f}, {0.334f, 0.334f}, {1.76f, 1.76f}, {0.0f, 0.0f}, {1.85f, 1.85f}},
};
constexpr TgCost kTgI8[] = {
    {32, 64, 2, {3.40f, 3.40f}, {0.002f, 0.002f}, {0.177f, 0.177f}, {0.55f, 0.55f}, {9.0f, 9.0f}, {0.65f, 0.65f}},
    {64, 64, 1, {2.98f, 2.98f}, {0.146f, 0.146f}, {0.094f, 0.094f}, {0.47f, 0.47f}, {53.0f, 53.0f}, {1.02f, 1.02f}},
    {64, 128, 1, {3.70f, 3.70f}, {0.141f, 0.141f}, {0.130f, 0.130f}, {1.63f, 1.63f}, {19.0f, 19.0f}, {1.52f, 1.52f}},
    {64, 128, 2, {3.55f, 3.55f}, {0.049f, 0.049f}, {0.262f, 0.262f}, {1.37f, 1.37f}, {2.0f, 2.0f}, {1.14f, 1.14f}},
    {128, 128, 1, {4.20f, 4.20f}, {0.270f, 0.270f}, {0.218f, 0.218f}, {1.38f, 1.38f}, {5.5f, 5.5f}, {1.83f, 1.83f}},
    {128, 256, 1, {6.54f, 6.54f}, {0.509f, 0.509f}, {0.321f, 0.321f}, {0.44f, 0.44f}, {9.0f, 9.0f}, {2.03f, 2.03f}},
};

bool tile_gemm_supported(int kind, int M, int N, int K) {
    return M >= 1 && N >= 1 && K >= 16 && K % (kind == TG_I8 ? 32 : 16) == 0 && (long)K * 256 * 2 < (1l << 31);
}

static TgPlan tg_choose(int kind, int dtype, int M, int N, int K, size_t scratch_bytes) {
    const bool few = M < 256;
    const TgCost *tab = kind == TG_W8S ? kTgW8S : kind == TG_W8 ? (few ? kTgW8Few : kTgW8) : few ? kTgI8Few : kTgI8;
    const int n_tiles = kind == TG_W8S ? 3 : 6, d = dtype == MYNN_BF16 ? 1 : 0;
    const int iters = (K * (kind == TG_I8 ? 1 : 2) + 127) / 128;
    const double weights_us = (double)N * K / 4.6e6;
    TgPlan best;
    best.us = 1e30;
    for (int t = 0; t < n_tiles; t++) {
        const TgCost &c = tab[t];
        const long tiles = (long)((M + c.bm - 1) / c.bm) * ((N + c.bn - 1) / c.bn);
        for (int ks = 1; ks <= 16; ks += ks < 4 ? 1 : ks < 8 ? 2 : 4) {
            const size_t part = ks > 1 ? (size_t)tiles * ks * c.bm * c.bn * 4 : 0;
            // (a range is at least three steps, from 256 rows on 2048 values: shorter ranges did not win there, and so a
            // block of rows has the same sums whatever it is multiplied with when K < 4096; a launch that already has four workgroups per CU gains nothing by ranges)
            if (ks > 1 && (ks * (M >= 256 && kind != TG_I8 ? 32 : 3) > iters || tiles * ks > 1024 || tiles > kTgCounters || part > scratch_bytes)) continue;
            const long wgs = (tiles * ks + 255) / 256, rounds = (wgs + c.per_cu - 1) / c.per_cu;
            double us = (double)((iters + ks - 1) / ks) * (c.a[d] * rounds + c.b[d] * wgs) + c.g[d] * (wgs - 1);
            if (ks > 1) us += c.e[d] * ks + part * 2e-6 / 4.0;
            us = std::max(us, std::max(weights_us, 2.0 * tiles * c.bm * c.bn * K / (c.rate[d] * 1e9))) + c.launch[d];
            if (us < best.us) best = TgPlan{t, ks, us, part};
        }
    }
    return best;
}

// (the search is some 50 evaluations, half a microsecond of an operator call: a thread remembers its last few)
TgPlan tile_gemm_plan(int kind, int dtype, int M, int N, int K, size_t scratch_bytes) {
    struct Entry {
        int kind = -1, dtype, M, N, K;
        size_t scratch;
        TgPlan plan;
    };
    thread_local Entry table[32];
    Entry &e = table[((unsigned)M * 31u + (unsigned)N * 17u + (unsigned)K * 7u + (unsigned)kind * 5u + (unsigned)dtype) % 32u];
    if (e.kind != kind || e.dtype != dtype || e.M != M || e.N != N || e.K != K || e.scratch != scratch_bytes)
        e = Entry{kind, dtype, M, N, K, scratch_bytes, tg_choose(kind, dtype, M, N, K, scratch_bytes)};
    return e.plan;
}

TgPlan tile_gemm_plan_seq(int kind, int dtype, int M, int N, int K, int ks) {
    TgPlan plan = tile_gemm_plan(kind, dtype, M, N, K, 0);
    plan.ks = kind == TG_I8 ? 1 : ks;  // (int32 sums are the same in any order)
    plan.seq = plan.ks > 1;
    return plan;
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
    if constexpr (G::KIND != TG_I8) {
        if (p.seq) return tail ? tg_go<T, G, GEMM_PLAIN, true, true>(p) : tg_go<T, G, GEMM_PLAIN, false, true>(p);
    }
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
template <typename T> static int tg_launch(int kind, int tile, const TgArgs &p, int epi) {
    if constexpr (sizeof(T) == 2) {
        if (kind == TG_W8) {
            if (tile == 0) return tg_epi<T, TgTile<TG_W8, 32, 64, 1, 2, 6, 2, 1>>(p, epi);
            if (tile == 1) return tg_epi<T, TgTile<TG_W8, 32, 128, 1, 4, 4, 2, 1>>(p, epi);
            if (tile == 2) return tg_epi<T, TgTile<TG_W8, 64, 64, 2, 2, 6, 2, 1>>(p, epi);
            if (tile == 3) return tg_epi<T, TgTile<TG_W8, 64, 128, 1, 4, 4, 2, 2>>(p, epi);
            if (tile == 4) return tg_epi<T, TgTile<TG_W8, 128, 128, 2, 4, 6, 2, 2>>(p, epi);
            // fp16: every weight is converted by one wave only (128 x 32 per wave); bf16: that form spills, 64 x 64 per wave
            if constexpr (std::is_same<T, f16_t>::value) return tg_epi<T, TgTile<TG_W8, 128, 128, 1, 4, 3, 2, 1>>(p, epi);
            else return tg_epi<T, TgTile<TG_W8, 128, 128, 2, 2, 3, 2, 1>>(p, epi);
        }
        if (kind == TG_W8S) {
            if (tile == 0) return tg_epi<T, TgTile<TG_W8S, 32, 32, 1, 1, 8, 1, 1>>(p, epi);
            if (tile == 1) return tg_epi<T, TgTile<TG_W8S, 32, 64, 1, 2, 6, 2, 1>>(p, epi);
            return tg_epi<T, TgTile<TG_W8S, 32, 128, 1, 4, 4, 2, 1>>(p, epi);
        }
    }
    if (tile == 0) return tg_epi<T, TgTile<TG_I8, 32, 64, 1, 2, 6, 1, 1>>(p, epi);
    if (tile == 1) return tg_epi<T, TgTile<TG_I8, 64, 64, 2, 2, 6, 2, 1>>(p, epi);
    if (tile == 2) return tg_epi<T, TgTile<TG_I8, 64, 128, 2, 4, 6, 2, 2>>(p, epi);
    if (tile == 3) return tg_epi<T, TgTile<TG_I8, 64, 128, 2, 2, 3, 2, 1>>(p, epi);
    if (tile == 4) return tg_epi<T, TgTile<TG_I8, 128, 128, 2, 4, 4, 2, 1>>(p, epi);
    return tg_epi<T, TgTile<TG_I8, 128, 256, 2, 4, 3, 2, 1>>(p, epi);
}

int tile_gemm(int kind, const TgPlan &plan, void *out, int32_t *acc_out, const void *act, const int8_t *wq, const void *a_scale, const void *w_scale,
              const void *res, int M, int N, int K, int dtype, int epi, void *part, int *counters, hipStream_t s) {
    MYNN_REQUIRE((out || acc_out) && act && wq && (w_scale || !out) && (kind != TG_I8 || a_scale || !out), MYNN_ERR_INVALID, "tile_gemm: null operand");
    MYNN_REQUIRE(tile_gemm_supported(kind, M, N, K), MYNN_ERR_UNSUPPORTED, "tile_gemm: M=%d N=%d K=%d", M, N, K);
    MYNN_REQUIRE(aligned16(act) && aligned16(wq), MYNN_ERR_INVALID, "tile_gemm: operands must be 16-byte aligned");
    MYNN_REQUIRE(epi != GEMM_RESIDUAL || res, MYNN_ERR_INVALID, "tile_gemm: residual store without a residual");
    MYNN_REQUIRE((epi != GEMM_SWIGLU_PAIRS && epi != GEMM_SWIGLU_PAIRS_EXP) || (N % 2 == 0 && !acc_out), MYNN_ERR_INVALID, "tile_gemm: SwiGLU store needs row pairs, N=%d", N);
    MYNN_REQUIRE(epi != GEMM_SWIGLU && (kind != TG_W8S || epi == GEMM_PLAIN) && (kind != TG_I8 || epi != GEMM_SWIGLU_PAIRS), MYNN_ERR_INVALID, "tile_gemm: store %d", epi);
    MYNN_REQUIRE(plan.ks >= 1 && (plan.ks == 1 || plan.seq || (part && counters && aligned16(part))), MYNN_ERR_INVALID, "tile_gemm: K ranges without scratch memory");
    MYNN_REQUIRE(!plan.seq || (kind != TG_I8 && epi == GEMM_PLAIN), MYNN_ERR_UNSUPPORTED, "tile_gemm: ranges one after the other: kind %d, store %d", kind, epi);
    const TgArgs p{out, acc_out, act, wq, a_scale, w_scale, res, M, N, K, plan.ks, plan.seq, (uint64_t *)part, counters, s};
    MYNN_REQUIRE(dtype != MYNN_F32 || (kind == TG_I8 && epi == GEMM_PLAIN), MYNN_ERR_UNSUPPORTED, "tile_gemm: f32 output of int8 products only");
    return dispatch_dtype(dtype, [&](auto *t) {
        using T = std::remove_pointer_t<decltype(t)>;
        return tg_launch<T>(kind, plan.tile, p, epi);
    });
}

}  // namespace mynn
