// DequantMatMul for a handful of activation rows (2 <= M <= 64: decode batches), one launch per linear.
//
// At this size a linear is a few microseconds, of which skinny.hip's form -- K ranges over workgroups, partial sums through
// memory, a second launch that adds them up -- spends more on the second launch than on the weights.  Here one workgroup
// owns 16 .. 96 weight rows (NB blocks of 16) over the WHOLE K range, its waves share K, and the partial sums meet in LDS, so the
// workgroup stores finished output: scale, residual or SwiGLU, and in front the RMSNorm of the activation rows (NORM, up to 16 rows).
//
//   out[m,n] = T(scale[n] * sum_k act[m,k] * wq[n,k])   (scale after the f32 sum, as skinny.hip)
//
// A wave's share of K is its own alone, weights and activations: both go global -> LDS by the load unit into rings that no other
// wave touches, so up to the final sum nothing is waited for but the wave's own loads, by count.  A step is 64 k: a kilobyte of
// weights per row block (skinny.hip's tiled copy: 16 rows x 4 pieces of 16 bytes) and a kilobyte of activations per 8 rows (whole 128-byte
// lines; through registers, as the matrix cores want them, a load would touch half lines of 16 rows, and half the rate came of it).
// The waves of a workgroup take steps in turn, so that they sweep the copy together.  PACKED false: weights as they are stored, row by row
// (operator calls), two steps at a time.
//
// What bounds it: few rows, the weights (4096 x 14336, 8 rows: 12.2 us of which a flat read is 9); many, what a CU gets of the
// activations, which every workgroup reads in full: some 80 KB a microsecond from the XCD's L2 (that keeps large K with many rows out
// of this kernel: rowblock_supported).  Against panels of activations for all waves, two in turn behind a barrier each, with the
// weights in registers, fp16, us: 8 rows, 2048 x 2048 4.3 -> 3.7, 2048 x 5632 6.2 -> 5.6, 4096 x 4096 7.0 -> 5.2, 6144 x 4096 8.7 -> 6.5,
// 4096 x 14336 14.7 -> 12.2, 11264 x 2048 7.4 -> 6.1; 32 rows, 2048 x 2048 5.4 -> 4.0, 11264 x 2048 9.7 -> 8.4.
//
// NORM: a wave squares what it loaded, the waves add up the rows' sums over one barrier, and each normalises its share in place; all of
// it is in LDS and all weights are in flight in registers meanwhile.  8 rows, 2560 x 2048 5.8 -> 5.0 us, 11264 x 2048 8.2 -> 7.5, 6144 x
// 4096 10.2 -> 9.7 (with whole rows a wave each, normalised by every workgroup before its first product).
#include <type_traits>

#include "kernels.h"
#include "mfma.h"
#include "wave_ring.h"

namespace mynn {

constexpr int kRbMaxRows = 64;
// NB row blocks of 16 per workgroup, A8 groups of 8 activation rows, ND stages of weights, NA stages of activations, WAVES waves
// (NORM: NA >= the steps of a wave; its weights are in registers, ND = 0)
template <int NB_, int A8_, int ND_, int NA_, int WAVES_, bool PACKED_ = true> struct RbShape {
    static constexpr bool PACKED = PACKED_;
    static constexpr int H = PACKED ? 1 : 2;  // steps of 64 k that are asked for together
    static constexpr int NB = NB_, A8 = A8_, ND = ND_, NA = NA_, WAVES = WAVES_, MT = (A8 + 1) / 2;
    static constexpr int WAVE_BYTES = (ND * NB + NA * A8) * H * 1024;
    static constexpr int RED = 16 + 4;  // floats per row of partial sums
    static constexpr int SQUARES = ND ? 0 : WAVES * A8 * 8 * 4;
    static size_t lds(int M) {
        const size_t st = (size_t)WAVES * WAVE_BYTES + SQUARES, red = (size_t)WAVES * NB * M * RED * sizeof(float);
        return st > red ? st : red;
    }
};

typedef float f4x_t __attribute__((ext_vector_type(4)));
// D[16 x 16] += A[16 x 32] . B[32 x 16]: lane l holds row (column) l % 16, k = 8 * (l / 16) .. +7, of D column l % 16, rows 4 * (l / 16) .. +3
template <typename T> __device__ inline f4x_t rb_mfma(const U4 &a, const U4 &b, f4x_t c) {
    if constexpr (std::is_same<T, f16_t>::value) return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, a), __builtin_bit_cast(h8_t, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8_t, a), __builtin_bit_cast(b8_t, b), c, 0, 0, 0);
}

// EPI: the store, GEMM_*, or kRbParts: out is f32 sums [K range][M][N] that another launch adds up and finishes
constexpr int kRbParts = -1;
template <typename T, typename S, int EPI, bool NORM>
__global__ __launch_bounds__(S::WAVES * 64) void rowblock_gemm_kernel(const T *act, const U4 *pk, int M, int N, int K, const T *scale, const T *res,
                                                                      const T *norm_w, T *out, float eps) {
    constexpr int NB = S::NB, A8 = S::A8, ND = S::ND, NA = S::NA, MT = S::MT, WAVES = S::WAVES, RS = S::RED, H = S::H;
    constexpr bool PACKED = S::PACKED;
    static_assert(PACKED || !NORM, "");
    extern __shared__ __align__(16) char lds[];
    const int tid = threadIdx.x, lane = tid & 63, kw = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, h = lane >> 4;
    const int row_blocks = (N + 31) / 32, b0 = (int)blockIdx.x * NB;
    // steps up to the end of this workgroup's K range (PARTS: one of gridDim.y), the range's first, and how many are this wave's
    constexpr bool PARTS = EPI == kRbParts;
    const int total = K / (64 * H), halves = PARTS ? total * ((int)blockIdx.y + 1) / (int)gridDim.y : total, first_half = PARTS ? total * (int)blockIdx.y / (int)gridDim.y : 0;
    const int n = __builtin_amdgcn_readfirstlane(max(halves - first_half - kw + WAVES - 1, 0) / WAVES);
    char *ring_w = lds + kw * S::WAVE_BYTES, *ring_a = ring_w + ND * NB * H * 1024;
    // Addresses of this lane's 16 bytes, as load_group_to_lds takes them, from 4096 bytes in front of a step.  Activations: row 8 * i +
    // lane / 8, and of its 8 chunks the one that makes the fragment reads below meet different banks.  Weights: row r of the block, piece h
    // of the step's half of 128 k (the copy's piece of k 64 * a + 16 * j, row i of 32, is number 64 * j + 32 * a + i).
    uint32_t aoff[A8], woff[NB * H];
#pragma unroll
    for (int i = 0; i < A8; i++) {
        const int row = 8 * i + (lane >> 3);
        aoff[i] = (uint32_t)(min(row, M - 1) * K * 2 + (((lane & 7) ^ (lane >> 3)) << 4) + 4096 - 1024 * (i % 4));
    }
    if constexpr (!PACKED) {
#pragma unroll
        for (int j = 0; j < NB * H; j++) woff[j] = ring_chunk(lane, j, N - 1 - b0 * 16, K);
    } else
#pragma unroll
    for (int b = 0; b < NB; b++) {
        const int block = min(b0 + b, row_blocks * 2 - 1);
        woff[b] = (uint32_t)((block >> 1) * 4096 + (64 * h + (block & 1) * 16 + r) * 16 + 4096 - 1024 * (b % 4));
    }
    // the i-th step of this wave (within the matrix whatever i: a wave without steps of its own asks for the last one's where NORM counts on it)
    auto half_of = [&](int i) { return min(first_half + i * WAVES + kw, halves - 1); };
    auto step_w = [&](int i) {
        const int hs = half_of(i);
        if constexpr (!PACKED) return (const char *)pk + (size_t)b0 * 16 * K + (size_t)hs * 128 - 4096;
        else return (const char *)pk + (size_t)(hs >> 1) * row_blocks * 4096 + (hs & 1) * 512 - 4096;
    };
    auto request_w = [&](int i, int slot) {
        constexpr int L = NB * H;
        const uint32_t to = lds_offset(ring_w) + slot * L * 1024;
        const char *src = step_w(i);
        load_group_to_lds<(L < 4 ? L : 4), true>(src, woff, to);
        if constexpr (L > 4) load_group_to_lds<(L < 8 ? L - 4 : 4), true>(src, woff + 4, to + 4096);
        if constexpr (L > 8) load_group_to_lds<L - 8, true>(src, woff + 8, to + 8192);
    };
    auto request_a = [&](int i, int slot) {
#pragma unroll
        for (int x = 0; x < H; x++) {
            const char *src = (const char *)act + (size_t)(half_of(i) * H + x) * 128 - 4096;
            const uint32_t to = lds_offset(ring_a) + (slot * H + x) * A8 * 1024;
            load_group_to_lds<(A8 < 4 ? A8 : 4)>(src, aoff, to);
            if constexpr (A8 > 4) load_group_to_lds<A8 - 4>(src, aoff + 4, to + 4096);
        }
    };
    // what the store of this thread's first output needs (mostly its only one), fetched in front of everything else
    constexpr int PR = EPI == GEMM_SWIGLU ? 8 : 16;  // outputs per row block and activation row
    T sc0, sc1, rs0;
    if constexpr (!PARTS) {
        const int o = min(tid, NB * M * PR - 1), c = o % PR, m = (o / PR) % M, c0 = min((b0 + o / (PR * M)) * 16 + (EPI == GEMM_SWIGLU ? 2 * c : c), N - 1);
        sc0 = scale[c0];
        if constexpr (EPI == GEMM_SWIGLU) sc1 = scale[min(c0 + 1, N - 1)];
        if constexpr (EPI == GEMM_RESIDUAL) rs0 = res[(size_t)m * N + c0];
    }
    f4x_t acc[NB][MT];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int t = 0; t < MT; t++) acc[b][t] = f4x_t{0.f, 0.f, 0.f, 0.f};
    const int fr = A8 == 1 ? r & 7 : r;  // (rows past the loaded ones: columns that are not stored)
    const int frag = fr * 128, f0 = frag + (((2 * h) ^ (fr & 7)) << 4), f1 = frag + (((2 * h + 1) ^ (fr & 7)) << 4);
    U4 w[NB], a[MT][2];
    auto read_a = [&](int slot) {
        const char *st = ring_a + slot * A8 * 1024;
#pragma unroll
        for (int t = 0; t < MT; t++) {
            a[t][0] = *(const U4 *)(st + f0 + t * 2048);
            a[t][1] = *(const U4 *)(st + f1 + t * 2048);
        }
    };
    auto multiply = [&]() {
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const U4 lo = i8x8_to_operand<T>(w[b].x, w[b].y), hi = i8x8_to_operand<T>(w[b].z, w[b].w);
#pragma unroll
            for (int t = 0; t < MT; t++) {
                acc[b][t] = rb_mfma<T>(lo, a[t][0], acc[b][t]);
                acc[b][t] = rb_mfma<T>(hi, a[t][1], acc[b][t]);
            }
        }
    };
    asm volatile("" ::: "memory");  // (the counts below rely on the order of the requests)
    if constexpr (NORM) {
        // (steps past the wave's share are the matrix's last one and not used: they keep the counts)
        U4 nw[NA], wr[NA][NB];
#pragma unroll
        for (int i = 0; i < NA; i++) nw[i] = *(const U4 *)(norm_w + half_of(i) * 64 + (((lane & 7) ^ (lane >> 3)) << 3));
        asm volatile("" ::: "memory");
#pragma unroll
        for (int i = 0; i < NA; i++) request_a(i, i);
#pragma unroll
        for (int i = 0; i < NA; i++)
#pragma unroll
            for (int b = 0; b < NB; b++) wr[i][b] = __builtin_nontemporal_load((const U4 *)(step_w(i) + woff[b] + 1024 * (b % 4)));
        wait_for_loads<(NA * NB < 63 ? NA * NB : 63)>();
        float ss[A8];
#pragma unroll
        for (int g = 0; g < A8; g++) ss[g] = 0.f;
        auto mine = [&](int i, int g) { return (U4 *)(ring_a + (i * A8 + g) * 1024 + lane * 16); };  // what this lane loaded
#pragma unroll
        for (int i = 0; i < NA; i++)
#pragma unroll
            for (int g = 0; g < A8; g++) {
                float f[8], t = 0.f;
                widen8<T>(*mine(i, g), f);
#pragma unroll
                for (int x = 0; x < 8; x++) t += f[x] * f[x];
                ss[g] += i < n ? t : 0.f;
            }
        float *squares = (float *)(lds + WAVES * S::WAVE_BYTES);  // [wave][row]
#pragma unroll
        for (int g = 0; g < A8; g++) {
            ss[g] = group_sum<8>(ss[g]);
            if ((lane & 7) == 0) squares[kw * 8 * A8 + 8 * g + (lane >> 3)] = ss[g];
        }
        __syncthreads();
#pragma unroll
        for (int g = 0; g < A8; g++) {
            float t = 0.f;
#pragma unroll
            for (int k = 0; k < WAVES; k++) t += squares[k * 8 * A8 + 8 * g + (lane >> 3)];
            const float inv = 1.0f / sqrtf(t / (float)K + eps);
#pragma unroll
            for (int i = 0; i < NA; i++) {
                float f[8], q[8];
                widen8<T>(*mine(i, g), f);
                widen8<T>(nw[i], q);
                *mine(i, g) = U4{pack2<T>((f[0] * inv) * q[0], (f[1] * inv) * q[1]), pack2<T>((f[2] * inv) * q[2], (f[3] * inv) * q[3]),
                                 pack2<T>((f[4] * inv) * q[4], (f[5] * inv) * q[5]), pack2<T>((f[6] * inv) * q[6], (f[7] * inv) * q[7])};
            }
        }
#pragma unroll
        for (int i = 0; i < NA; i++) {
            if (i >= n) break;
            read_a(i);
#pragma unroll
            for (int b = 0; b < NB; b++) {
                w[b] = wr[i][b];
                pin(w[b]);  // (converted here, not when they were loaded)
            }
            multiply();
        }
    } else {
        constexpr int C = (A8 + NB) * H;  // loads of a step
        static_assert(NORM || NA == ND, "one count for both rings");
        auto request = [&](int i, int slot) {
            request_w(i, slot);
            request_a(i, slot);
        };
        int i = 0, slot = 0;
        const int wrow = r * 128;  // !PACKED: row r's chunks of 16 bytes, placed as those of the activations
        auto use = [&](int x) {
#pragma unroll
            for (int b = 0; b < NB; b++)
                w[b] = *(const U4 *)(ring_w + (slot * NB + b) * H * 1024 + (PACKED ? lane * 16 : wrow + (((4 * x + h) ^ (r & 7)) << 4)));
            read_a(slot * H + x);
        };
#pragma unroll
        for (int d = 0; d < ND - 1; d++)
            if (d < n) request(d, d);
        for (; i + ND - 1 < n; i++) {
            wait_for_loads<(ND - 2) * C>();
            use(0);
            request(i + ND - 1, slot == 0 ? ND - 1 : slot - 1);  // (the stage that the step before was read from)
            multiply();
            if constexpr (H > 1) {
                use(1);
                multiply();
            }
            slot = slot + 1 == ND ? 0 : slot + 1;
        }
        // the last ND - 1 steps, with nothing left to ask for
        auto rest = [&](auto left) {
            constexpr int L = decltype(left)::value;
            if constexpr (L < ND) {
                if (n - i != L) return;
                wait_for_loads<(L - 1) * C>();
                use(0);
                multiply();
                if constexpr (H > 1) {
                    use(1);
                    multiply();
                }
                slot = slot + 1 == ND ? 0 : slot + 1;
                i++;
            }
        };
        static_assert(NORM || (ND >= 2 && ND <= 8), "");
        rest(std::integral_constant<int, 7>{});
        rest(std::integral_constant<int, 6>{});
        rest(std::integral_constant<int, 5>{});
        rest(std::integral_constant<int, 4>{});
        rest(std::integral_constant<int, 3>{});
        rest(std::integral_constant<int, 2>{});
        rest(std::integral_constant<int, 1>{});
    }
    __syncthreads();  // the rings are done with: their memory takes the partial sums
    float *red = (float *)lds;
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int t = 0; t < MT; t++) {
            const int m = t * 16 + r;
            if (m < M) *(float4 *)(red + ((size_t)(kw * NB + b) * M + m) * RS + 4 * h) = float4{acc[b][t][0], acc[b][t][1], acc[b][t][2], acc[b][t][3]};
        }
    __syncthreads();
    if constexpr (PARTS) {  // (N % 16 == 0)
        float *part = (float *)out + (size_t)blockIdx.y * M * N;
        for (int o = tid; o < NB * M * 4; o += WAVES * 64) {
            const int c = o % 4 * 4, b = (o / 4) % NB, m = o / (4 * NB), col = (b0 + b) * 16 + c;
            float4 t = float4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int k = 0; k < WAVES; k++) {
                const float4 v = *(const float4 *)(red + ((size_t)(k * NB + b) * M + m) * RS + c);
                t.x += v.x, t.y += v.y, t.z += v.z, t.w += v.w;
            }
            if (col < N) *(float4 *)(part + (size_t)m * N + col) = t;
        }
        return;
    }
    for (int o = tid; o < NB * M * PR; o += WAVES * 64) {
        const int c = o % PR, m = (o / PR) % M, b = o / (PR * M);
        const int c0 = (b0 + b) * 16;
        const bool first = o == tid;
        auto sum = [&](int col) {
            float t = 0.f;
#pragma unroll
            for (int k = 0; k < WAVES; k++) t += red[((size_t)(k * NB + b) * M + m) * RS + col];
            return t;
        };
        if constexpr (EPI == GEMM_SWIGLU) {  // rows 2i / 2i+1 of the weight are gate_i / up_i
            const int col = c0 + 2 * c;
            if (col + 1 < N) {
                const T sg = first ? sc0 : scale[col], su = first ? sc1 : scale[col + 1];
                const float g = Elem<T>::rnd(sum(2 * c) * Elem<T>::ld(&sg, 0)), u = Elem<T>::rnd(sum(2 * c + 1) * Elem<T>::ld(&su, 0));
                const float sig = 1.0f / (1.0f + expf(-g));
                Elem<T>::st(out, (size_t)m * (N >> 1) + (col >> 1), (g * sig) * u);
            }
        } else {
            const int col = c0 + c;
            if (col < N) {
                const T sn = first ? sc0 : scale[col];
                float y = sum(c) * Elem<T>::ld(&sn, 0);
                if constexpr (EPI == GEMM_RESIDUAL) {
                    const T rn = first ? rs0 : res[(size_t)m * N + col];
                    y = Elem<T>::rnd(y) + Elem<T>::ld(&rn, 0);
                }
                Elem<T>::st(out, (size_t)m * N + col, y);
            }
        }
    }
}

// ---- which form: as many row blocks per workgroup as leave one workgroup per CU (its rings take most of the LDS), stages as the
// 160 KB allow.
template <bool NORM, typename F> static auto rb_shape(int M, int N, int K, F &&f) {
    auto rows = [&](auto b) {
        constexpr int NB = decltype(b)::value;
        if constexpr (NORM) {
            if (K <= 2048) return M <= 8 ? f(RbShape<NB, 1, 0, 4, 8>{}) : f(RbShape<NB, 2, 0, 4, 8>{});
            if constexpr (NB <= 3) return M <= 8 ? f(RbShape<NB, 1, 0, 8, 8>{}) : f(RbShape<NB, 2, 0, 8, 8>{});
            return f(RbShape<NB, 2, 0, 4, 8>{});  // (refused by rowblock_supported)
        } else {
            constexpr int D1 = 20 / (NB + 1) < 8 ? 20 / (NB + 1) : 8, D2 = 20 / (NB + 2), D4 = 20 / (NB + 4);
            if (M <= 8) return f(RbShape<NB, 1, D1, D1, 8>{});
            if (M <= 16) return f(RbShape<NB, 2, D2, D2, 8>{});
            if (M <= 32) return f(RbShape<NB, 4, D4, D4, 8>{});
            if constexpr (NB <= 2) return f(RbShape<NB, 8, 2, 2, 8>{});
            else return f(RbShape<NB, 8, 40 / (NB + 8), 40 / (NB + 8), 4>{});  // (a stage of eight waves would be the only one)
        }
    };
    if (N <= 256 * 16) return rows(std::integral_constant<int, 1>{});
    if (N <= 256 * 32) return rows(std::integral_constant<int, 2>{});
    if (N <= 256 * 48) return rows(std::integral_constant<int, 3>{});
    if (N <= 256 * 64) return rows(std::integral_constant<int, 4>{});
    return rows(std::integral_constant<int, 6>{});
}
// From 768 row blocks of 32 on skinny.hip's one-launch form streams the weights just as fast (28672 x 4096, 8 rows: 23 us).
// More than 16 rows: the activations' bytes keep large K out unless there are many weight rows to use them for.
// The norm rides along up to 16 rows (it costs 1.0 us for 8 rows x 2048, 2.2 for 16, 2.9 for 8 x 4096, against a launch of 2.5 - 5); over
// 2048 values with more than 12288 weight rows it would cost 6 (the weights that wait in registers meanwhile).
bool rowblock_fits(int M, int N, int K, bool norm) {
    return M >= 1 && M <= kRbMaxRows && K % 128 == 0 && N >= 1 && (N + 31) / 32 < 768 && (long)M * K * 2 < (1l << 31) && (!norm || (M <= 16 && K <= (N <= 256 * 48 ? 4096 : 2048)));
}
bool rowblock_supported(int M, int N, int K, bool norm) {
    return rowblock_fits(M, N, K, norm) && (M <= 16 || (long)N * K <= (12l << 20) || (N + 31) / 32 > 256);
}

template <typename T, typename S, int EPI, bool NORM>
static int rb_go(const void *act, const void *pk, const void *scale, const void *res, const void *norm_w, void *out, int M, int N, int K, float eps,
                 hipStream_t s, int ranges = 1) {
    static size_t lds_set = 64 * 1024;
    const size_t lds = S::lds(M);
    static_assert(S::WAVES * S::WAVE_BYTES + S::SQUARES <= 160 * 1024 && S::WAVES * S::NB * S::A8 * 8 * S::RED * 4 <= 160 * 1024, "");
    if (lds > lds_set) {
        MYNN_HIP(hipFuncSetAttribute((const void *)rowblock_gemm_kernel<T, S, EPI, NORM>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        lds_set = 160 * 1024;
    }
    constexpr int rows = S::NB * 16;
    MYNN_LAUNCH((rowblock_gemm_kernel<T, S, EPI, NORM>), dim3((N + rows - 1) / rows, ranges), dim3(S::WAVES * 64), lds, s, (const T *)act, (const U4 *)pk, M, N, K,
                (const T *)scale, (const T *)res, (const T *)norm_w, (T *)out, eps);
    return launch_status("rowblock_gemm_kernel");
}

int rowblock_gemm(void *out, const void *act, const void *packed, const void *scale, const void *res, const void *norm_w, float eps, int M, int N,
                  int K, int dtype, int epi, hipStream_t s) {
    MYNN_REQUIRE(out && act && packed && scale && (epi != GEMM_RESIDUAL || res), MYNN_ERR_INVALID, "rowblock_gemm: null operand");
    MYNN_REQUIRE(rowblock_fits(M, N, K, norm_w != nullptr) && (epi != GEMM_SWIGLU || N % 2 == 0), MYNN_ERR_UNSUPPORTED, "rowblock_gemm: M=%d N=%d K=%d", M, N, K);
    MYNN_REQUIRE(aligned16(act) && aligned16(packed) && (!norm_w || aligned16(norm_w)), MYNN_ERR_INVALID, "rowblock_gemm: operands must be 16-byte aligned");
    return dispatch_dtype16(dtype, [&](auto *t) {
        using T = std::remove_pointer_t<decltype(t)>;
        auto go = [&](auto norm) {
            constexpr bool NORM = decltype(norm)::value;
            return rb_shape<NORM>(M, N, K, [&](auto shape) {
                using S = decltype(shape);
                if (epi == GEMM_RESIDUAL) return rb_go<T, S, GEMM_RESIDUAL, NORM>(act, packed, scale, res, norm_w, out, M, N, K, eps, s);
                if (epi == GEMM_SWIGLU) return rb_go<T, S, GEMM_SWIGLU, NORM>(act, packed, scale, res, norm_w, out, M, N, K, eps, s);
                return rb_go<T, S, GEMM_PLAIN, NORM>(act, packed, scale, res, norm_w, out, M, N, K, eps, s);
            });
        };
        return norm_w ? go(std::true_type{}) : go(std::false_type{});
    });
}

// ---- sums of two K ranges for a launch that adds them up (and makes the norm of the row): half of K for twice the weight rows halves what
// a workgroup reads of the activations.  Against skinny.hip's product of some 1000 waves' ranges, us a pass: TinyLlama, 17 rows 890 / 850, 32
// rows 943 / 905, 64 rows 1153 / 1102; 8B widths, 8 layers, 64 rows 904 / 886, steps of 48 sequences 991 / 971, of 64 1045 / 1036; but of 32
// 759 / 770 (4096 x 14336: the bytes of a workgroup again), so up to 32 rows for narrow matrices alone.
bool rowblock_parts_supported(int M, int N, int K) {
    return M >= 17 && M <= kRbMaxRows && N <= (M <= 32 ? 256 * 8 : 256 * 16) && N % 16 == 0 && K % 128 == 0 && K >= 4 * 128 && (long)M * K * 2 < (1l << 31);
}
int rowblock_parts(float *part, const void *act, const void *packed, int M, int N, int K, int dtype, hipStream_t s) {
    MYNN_REQUIRE(part && act && packed && rowblock_parts_supported(M, N, K), MYNN_ERR_UNSUPPORTED, "rowblock_parts: M=%d N=%d K=%d", M, N, K);
    MYNN_REQUIRE(aligned16(act) && aligned16(packed) && aligned16(part), MYNN_ERR_INVALID, "rowblock_parts: operands must be 16-byte aligned");
    return dispatch_dtype16(dtype, [&](auto *t) {
        using T = std::remove_pointer_t<decltype(t)>;
        return rb_shape<false>(M, 2 * N, K, [&](auto shape) {  // (two ranges: as many workgroups as twice the rows)
            using S = decltype(shape);
            if constexpr (S::NB <= 2 && S::A8 >= 4) return rb_go<T, S, kRbParts, false>(act, packed, nullptr, nullptr, nullptr, part, M, N, K, 0.f, s, kRbRanges);
            return (int)MYNN_ERR_UNSUPPORTED;
        });
    });
}

// ---- row-major weights, up to 16 rows: stages of 128 k, so that a load touches whole lines of 8 weight rows.  One workgroup per CU up to
// 12288 weight rows, as above; beyond, workgroups of four waves, two per CU, whose ramps and stores overlap (6 rows, bf16, us, eight waves /
// four: 14336 x 4096 12.6 with 64 rows each / 12.8 with 32, 15 rows 18.2 with 48 / 14.1 with 32; 28672 x 4096 25.7 with 32 / 22.9 with 64).
template <typename F> static int rb_rows_shape(int M, int N, F &&f) {
    auto form = [&](auto b, auto waves) {
        constexpr int NB = decltype(b)::value, W = decltype(waves)::value, D1 = 20 / (2 * NB + 2), D2 = 20 / (2 * NB + 4);
        if constexpr (D2 < 2) return f(RbShape<NB, 1, D1, D1, W, false>{});
        else return M <= 8 ? f(RbShape<NB, 1, D1, D1, W, false>{}) : f(RbShape<NB, 2, D2, D2, W, false>{});
    };
    using std::integral_constant;
    if (N <= 256 * 16) return form(integral_constant<int, 1>{}, integral_constant<int, 8>{});
    if (N <= 256 * 32) return form(integral_constant<int, 2>{}, integral_constant<int, 8>{});
    if (N <= 256 * 48) return form(integral_constant<int, 3>{}, integral_constant<int, 8>{});
    if (N <= 512 * 32 || M > 8) return form(integral_constant<int, 2>{}, integral_constant<int, 4>{});
    return form(integral_constant<int, 4>{}, integral_constant<int, 4>{});
}
// (one row streams faster through the GEMV, and more than 15 are summed with the scale inside)
bool rowblock_rows_supported(const void *out, const void *act, const void *wq, const void *scale, int M, int N, int K) {
    return out && act && wq && scale && M >= 2 && M <= 15 && N >= 1 && K >= 128 && K % 128 == 0 && (long)K * 128 < (1l << 31) && aligned16(act) && aligned16(wq);
}
// ... and where it is the one to take (us a call with weights that are not cached, tiles over K ranges / so; profiles/few_row_times.csv has both over
// 1200 shapes):
//   Few weight rows leave most CUs without a workgroup, and a workgroup's own share, 16 weight rows and all of the activations over the whole
//   of K, outlasts K ranges over the device from some 800 KB on (15 rows: 500 x 14336 14.2 / 13.0, 1024 x 32768 19.8 / 25.9, 500 x 65536
//   26.8 / 48.9; 8 rows, 500 x 65536 26.7 / 35.7), with 1536 weight rows from 1100 KB (9 rows, 2048 x 32768 23.0 / 23.6).
//   Rows of whole 8192 bytes begin at the same channels of the memory; workgroups of four waves, two per CU, ask for little of each at a time
//   and meet there: 15 rows, 18432 x 8192 37.3 / 44.4 (x 7168 34.5 / 33.9), 32000 x 8192 61.0 / 64.5 (x 7168 46.3 / 42.0).  (16384 x 8192 with its 32 weight
//   rows each by where the matrices lie: 6 rows 26.4 / 31.4 and 36.6 / 32.0.)
bool rowblock_rows_first(int M, int N, int K) {
    if (N < 3072 && (16 + 2l * M) * K > (N < 1536 ? 790000 : 1100000)) return false;
    return N <= 512 * 32 || M <= 8 || K % 8192 != 0;
}
int rowblock_rows_gemm(void *out, const void *act, const int8_t *wq, const void *scale, int M, int N, int K, int dtype, hipStream_t s) {
    MYNN_REQUIRE(rowblock_rows_supported(out, act, wq, scale, M, N, K), MYNN_ERR_UNSUPPORTED, "rowblock_rows_gemm: M=%d N=%d K=%d", M, N, K);
    return dispatch_dtype16(dtype, [&](auto *t) {
        using T = std::remove_pointer_t<decltype(t)>;
        return rb_rows_shape(M, N, [&](auto shape) {
            return rb_go<T, decltype(shape), GEMM_PLAIN, false>(act, wq, scale, nullptr, nullptr, out, M, N, K, 0.f, s);
        });
    });
}

}  // namespace mynn
