// DequantMatMul for a handful of activation rows (2 <= M <= 64: decode batches), one launch per linear.
//
// At this size a linear is a few microseconds, of which skinny.hip's form -- K ranges over workgroups, partial sums through
// memory, a second launch that adds them up -- spends more on the second launch than on the weights.  Here one workgroup
// owns 16 .. 64 weight rows (RB row blocks of RH) over the WHOLE K range: its waves split K among themselves, every wave has
// its share of the weights in flight before the first product, and the partial sums meet in LDS, so the workgroup stores
// finished output: scale, residual or SwiGLU, and in front the RMSNorm of the activation rows while they are staged (NORM).
//
//   out[m,n] = T(scale[n] * sum_k act[m,k] * wq[n,k])   (scale after the f32 sum, as skinny.hip)
//
// The weights are skinny.hip's tiled copy: a wave's step of 32 rows x 128 k is 4 KB, read by four sequential loads, and
// turned exactly into the A operand of v_mfma_f32_32x32x16 (or half of it into that of 16x16x32); the activation rows are the
// B operand's columns, read from LDS.
#include <type_traits>

#include "kernels.h"
#include "mfma.h"

namespace mynn {

// The waves of a workgroup: row blocks times shares of a slab of WK * 128 k (a step per wave) times groups of activation rows.  DEPTH slabs of
// weights are in flight per wave.  Activations, plain form: panels of SPP slabs, [M] rows, copied global -> LDS by the load
// unit, the next panel while one is multiplied; NORM > 0: whole rows at once, NORM 16-byte pieces per lane.
constexpr int kRbMaxRows = 64, kRbDepth = 4;
// RB row blocks of RH weight rows per workgroup, WK waves that share a slab's K, CG groups of waves with MC tiles of RH
// activation rows each
template <int RB_, int RH_, int WK_, int CG_, int MC_, int SPP_> struct RbShape {
    static constexpr int RB = RB_, RH = RH_, WK = WK_, CG = CG_, MC = MC_, SPP = SPP_, WAVES = RB * WK * CG, ROWS = CG * MC * RH;
    static constexpr int PANEL = WK * 128 * SPP, ROW_BYTES = (PANEL + 511) / 512 * 1024 + 16;
    static constexpr int RED = RH + 4;  // floats per row of partial sums
    static size_t lds(int M, int K, bool norm) {
        const size_t act = norm ? (size_t)M * (K * 2 + 16) : (size_t)(K > PANEL ? 2 : 1) * M * ROW_BYTES, red = (size_t)WK * RB * M * RED * sizeof(float);
        return act > red ? act : red;
    }
};

typedef float f4x_t __attribute__((ext_vector_type(4)));
template <typename T> __device__ inline f16x_t rb_mfma(const U4 &a, const U4 &b, f16x_t c) { return Mfma<T>::run(a, b, c); }
template <typename T> __device__ inline f4x_t rb_mfma(const U4 &a, const U4 &b, f4x_t c) {
    if constexpr (std::is_same<T, f16_t>::value) return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, a), __builtin_bit_cast(h8_t, b), c, 0, 0, 0);
    else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8_t, a), __builtin_bit_cast(b8_t, b), c, 0, 0, 0);
}

template <typename T, typename S, int EPI, int NORM>
__global__ __launch_bounds__(S::WAVES * 64) void rowblock_gemm_kernel(const T *act, const U4 *pk, const T *scale, const T *res, const T *norm_w, T *out,
                                                                      int M, int N, int K, float eps) {
    constexpr int RB = S::RB, RH = S::RH, WK = S::WK, MC = S::MC, SPP = S::SPP, WAVES = S::WAVES, DEPTH = kRbDepth, RS = S::RED;
    extern __shared__ __align__(16) char lds[];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane % RH, h = lane / RH, cg = wave / (RB * WK), rb = wave / WK % RB, kw = wave % WK;
    const int row_blocks = (N + 31) / 32, iters = K / 128, slabs = (iters + WK - 1) / WK;
    const size_t pitch = (size_t)row_blocks * 256;  // 16-byte pieces of one step over all row blocks
    // The copy's 16-byte piece of k 64 * a + 16 * j, row i of a block is number 64 * j + 32 * a + i of its step.  A lane of
    // the 32-row form reads pieces (h, 0 .. 3), of the 16-row form (h % 2, h / 2) and (h % 2, 2 + h / 2).
    const int block = min((int)blockIdx.x * RB + rb, row_blocks * (32 / RH) - 1);
    constexpr int LPW = RH / 8;  // loads of a step
    const U4 *wsrc = pk + (size_t)(block / (32 / RH)) * 256 + (RH == 32 ? lane : (h >> 1) * 64 + (h & 1) * 32 + (block & 1) * 16 + r);
    U4 w[DEPTH][LPW];
    auto load_w = [&](int sl, U4 *dst) {
        const U4 *p = wsrc + (size_t)min(sl * WK + kw, iters - 1) * pitch;
#pragma unroll
        for (int j = 0; j < LPW; j++) dst[j] = __builtin_nontemporal_load(p + j * (RH == 32 ? 64 : 128));
    };
    // what the store of this thread's first output needs (mostly its only one), fetched in front of everything else
    constexpr int PR = EPI == GEMM_SWIGLU ? RH / 2 : RH;  // outputs per row block and activation row
    T sc0, sc1, rs0;
    {
        const int o = min(tid, RB * M * PR - 1), c = o % PR, m = (o / PR) % M, n = min((((int)blockIdx.x * RB + o / (PR * M)) * RH) + (EPI == GEMM_SWIGLU ? 2 * c : c), N - 1);
        sc0 = scale[n];
        if constexpr (EPI == GEMM_SWIGLU) sc1 = scale[min(n + 1, N - 1)];
        if constexpr (EPI == GEMM_RESIDUAL) rs0 = res[(size_t)m * N + n];
    }
    std::conditional_t<RH == 32, f16x_t, f4x_t> acc[MC];
    int arow0[MC];  // this lane's activation row of each tile (rows past M repeat the last one and are not stored)
#pragma unroll
    for (int mc = 0; mc < MC; mc++) {
#pragma unroll
        for (int e = 0; e < RH * RH / 64; e++) acc[mc][e] = 0.f;
        arow0[mc] = min((cg * MC + mc) * RH + r, M - 1);
    }
    auto multiply = [&](const U4 *q, const char *a0, int pitch) {  // a0: the activations at the step's first k
        U4 b[MC][2 * LPW];
#pragma unroll
        for (int mc = 0; mc < MC; mc++)
#pragma unroll
            for (int i = 0; i < 2 * LPW; i++)
                b[mc][i] = *(const U4 *)(a0 + (size_t)arow0[mc] * pitch + (RH == 32 ? 128 * h + 16 * i : 128 * (h & 1) + 32 * (h >> 1) + 64 * (i >> 1) + 16 * (i & 1)));
#pragma unroll
        for (int i = 0; i < LPW; i++) {
            U4 c = q[i];
            pin(c);  // (converted here, not when they were loaded)
            const U4 lo = i8x8_to_operand<T>(c.x, c.y), hi = i8x8_to_operand<T>(c.z, c.w);
#pragma unroll
            for (int mc = 0; mc < MC; mc++) {
                acc[mc] = rb_mfma<T>(lo, b[mc][2 * i], acc[mc]);
                acc[mc] = rb_mfma<T>(hi, b[mc][2 * i + 1], acc[mc]);
            }
        }
    };
    if constexpr (NORM > 0) {
        // whole rows, a wave each: requested before the weights, as loads return in order
        const int AS = K * 2 + 16, pieces = K >> 3;
        for (int m = wave; m < M || m == wave; m += WAVES) {
            U4 v[NORM], nw[NORM];
            const int ml = min(m, M - 1);
#pragma unroll
            for (int q = 0; q < NORM; q++) {
                const int c = min(lane + q * 64, pieces - 1);
                v[q] = *(const U4 *)(act + (size_t)ml * K + c * 8);
                nw[q] = *(const U4 *)(norm_w + c * 8);
            }
            if (m == wave) {
#pragma unroll
                for (int d = 0; d < DEPTH; d++) load_w(d, w[d]);
            }
            if (m >= M) break;
            float ss = 0.f;
#pragma unroll
            for (int q = 0; q < NORM; q++) {
                float f[8];
                widen8<T>(v[q], f);
                if (lane + q * 64 < pieces) {
#pragma unroll
                    for (int i = 0; i < 8; i++) ss += f[i] * f[i];
                }
            }
            const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)K + eps);
#pragma unroll
            for (int q = 0; q < NORM; q++) {
                const int c = lane + q * 64;
                float f[8], g[8];
                widen8<T>(v[q], f);
                widen8<T>(nw[q], g);
                if (c < pieces)
                    *(U4 *)(lds + (size_t)m * AS + c * 16) = U4{pack2<T>((f[0] * inv) * g[0], (f[1] * inv) * g[1]), pack2<T>((f[2] * inv) * g[2], (f[3] * inv) * g[3]),
                                                               pack2<T>((f[4] * inv) * g[4], (f[5] * inv) * g[5]), pack2<T>((f[6] * inv) * g[6], (f[7] * inv) * g[7])};
            }
        }
        __syncthreads();
        for (int s0 = 0; s0 < slabs; s0 += DEPTH) {
#pragma unroll
            for (int d = 0; d < DEPTH; d++) {
                const int sl = s0 + d;
                if (sl * WK + kw < iters) multiply(w[d], lds + (size_t)(sl * WK + kw) * 256, AS);
                if (s0 + DEPTH < slabs) load_w(sl + DEPTH, w[d]);
            }
        }
    } else {
        constexpr int PK = S::PANEL, AS = S::ROW_BYTES, CPR = (PK + 511) / 512;  // 1 KB copies per row
        const int panels = (slabs + SPP - 1) / SPP;
        auto issue_panel = [&](int p) {
            char *dst = lds + (size_t)(p & 1) * M * AS;
            for (int c = wave; c < M * CPR; c += WAVES) {
                const int m = c / CPR, k = p * PK + (c % CPR) * 512 + lane * 8;
                if (k - lane * 8 >= K) continue;
                load_to_lds((const char *)(act + (size_t)m * K + min(k, K - 8)), lds_offset(dst + (size_t)m * AS + (c % CPR) * 1024));
            }
        };
        issue_panel(0);
        asm volatile("" ::: "memory");  // (the counts below rely on the order of the requests)
#pragma unroll
        for (int d = 0; d < DEPTH; d++) load_w(d, w[d]);
        constexpr int AGE = (SPP < DEPTH ? SPP : DEPTH) * LPW;  // weight loads younger than the panel that is waited for, at least
        for (int s0 = 0; s0 < slabs; s0 += DEPTH) {
#pragma unroll
            for (int d = 0; d < DEPTH; d++) {
                const int sl = s0 + d;
                if (sl < slabs) {
                    if (sl % SPP == 0) {
                        // this panel is here, everyone is done with the one before it: its buffer takes the next
                        __builtin_amdgcn_s_waitcnt((AGE & 15) | (AGE >> 4) << 14 | 0x70);
                        asm volatile("" ::: "memory");
                        __builtin_amdgcn_s_barrier();
                        asm volatile("" ::: "memory");
                        if (sl / SPP + 1 < panels) issue_panel(sl / SPP + 1);
                        asm volatile("" ::: "memory");
                    }
                    if (sl * WK + kw < iters) multiply(w[d], lds + (size_t)((sl / SPP) & 1) * M * AS + (size_t)((sl % SPP) * WK + kw) * 256, AS);
                }
                load_w(sl + DEPTH, w[d]);  // (past the end: the last step once more, unused; it keeps the counts)
            }
        }
    }
    __syncthreads();  // the activations are done with: their memory takes the partial sums

    // D[n][m]: lane holds column m = lane % RH and rows n = 4 * (lane / RH) + e % 4, + 8 * (e / 4) in the 32-row form
    float *red = (float *)lds;
#pragma unroll
    for (int mc = 0; mc < MC; mc++) {
        const int m = (cg * MC + mc) * RH + r;
        if (m >= M) continue;
        float *dst = red + ((size_t)(kw * RB + rb) * M + m) * RS + 4 * h;
#pragma unroll
        for (int e4 = 0; e4 < RH * RH / 256; e4++) *(float4 *)(dst + e4 * 8) = float4{acc[mc][e4 * 4], acc[mc][e4 * 4 + 1], acc[mc][e4 * 4 + 2], acc[mc][e4 * 4 + 3]};
    }
    __syncthreads();
    for (int o = tid; o < RB * M * PR; o += WAVES * 64) {
        const int c = o % PR, m = (o / PR) % M, b = o / (PR * M);
        const int n0 = ((int)blockIdx.x * RB + b) * RH;
        const bool first = o == tid;
        auto total = [&](int n) {
            float t = 0.f;
#pragma unroll
            for (int k = 0; k < WK; k++) t += red[((size_t)(k * RB + b) * M + m) * RS + n];
            return t;
        };
        if constexpr (EPI == GEMM_SWIGLU) {  // rows 2i / 2i+1 of the weight are gate_i / up_i
            const int n = n0 + 2 * c;
            if (n + 1 < N) {
                const T sg = first ? sc0 : scale[n], su = first ? sc1 : scale[n + 1];
                const float g = Elem<T>::rnd(total(2 * c) * Elem<T>::ld(&sg, 0)), u = Elem<T>::rnd(total(2 * c + 1) * Elem<T>::ld(&su, 0));
                const float sig = 1.0f / (1.0f + expf(-g));
                Elem<T>::st(out, (size_t)m * (N >> 1) + (n >> 1), (g * sig) * u);
            }
        } else {
            const int n = n0 + c;
            if (n < N) {
                const T sn = first ? sc0 : scale[n];
                float y = total(c) * Elem<T>::ld(&sn, 0);
                if constexpr (EPI == GEMM_RESIDUAL) {
                    const T rn = first ? rs0 : res[(size_t)m * N + n];
                    y = Elem<T>::rnd(y) + Elem<T>::ld(&rn, 0);
                }
                Elem<T>::st(out, (size_t)m * N + n, y);
            }
        }
    }
}

// ---- which form: as many workgroups as there are CUs and no more, each with whole row blocks.
// HALF   up to 256 blocks of 16 rows
// ONE    one block of 32 rows per workgroup while that is at most one per CU (more than 32 activation rows: two of 16)
// THREE  three blocks of 16 rows, twelve waves, up to 256 such workgroups (16 activation rows; with a norm over more than 2048
//        values its rows do not fit the registers of twelve waves)
// TWO    two blocks of 32 rows; from 768 row blocks on skinny.hip's one-launch form streams the weights just as fast
//        (28672 x 4096, 8 rows: 23 us) and this kernel is not taken
// 8 rows, us, 32-row forms / HALF or THREE: 2560 x 2048 with norm 7.2 / 6.1, 2048 x 2048 6.3 / 4.9, 2048 x 5632 9.4 / 7.2, 4096 x
// 14336 18.6 / 14.5, 11264 x 2048 with norm 9.5 / 7.9, 10000 x 4096 12.6 / 11.2; but 6144 x 4096 9.1 / 9.7, 10000 x 4096 with norm
// 14.1 / 15.9.  24 rows, ONE or TWO / HALF with two tiles of activation rows: 2048 x 2048 6.9 / 5.7, 2048 x 5632 11.0 / 9.0.  48 rows,
// here / two launches of skinny.hip: 2560 x 2048 7.4 / 12, 2048 x 2048 7.0 / 12, 11264 x 2048 11.5 / 18, 2048 x 5632 13.1 / 12.6.
// A CU gets some 50 GB/s of weights and 180 GB/s of activations, which every workgroup reads in full: that is what keeps
// large K with many rows out of this kernel (rowblock_supported).
// The norm rides along up to 16 rows (8 rows x 2560 x 2048: 7.2 us with it in the ONE form against 6.0 + a launch of 2.5;
// every workgroup normalises all rows for itself, at 32 rows that costs 3.7 us).
template <typename F> static auto rb_shape(int M, int N, int K, bool norm, F &&f) {
    if (N <= 256 * 16) {
        if (M > 32) return f(RbShape<1, 16, 4, 2, 2, 1>{});
        if (M > 16) return f(RbShape<1, 16, 8, 1, 2, 1>{});
        if (norm || K > 8192) return f(RbShape<1, 16, 8, 1, 1, 1>{});  // (4096 x 14336: 14.5 us against 15.4 with two slabs per panel)
        return f(RbShape<1, 16, 8, 1, 1, 2>{});
    }
    if (N <= 256 * 32) return M > 32 ? f(RbShape<2, 16, 4, 1, 4, 1>{}) : f(RbShape<1, 32, 8, 1, 1, 1>{});
    if (M <= 16 && N <= 256 * 48 && (!norm || K <= 2048)) return f(RbShape<3, 16, 4, 1, 1, 2>{});
    return M > 32 ? f(RbShape<2, 32, 4, 1, 2, 1>{}) : f(RbShape<2, 32, 4, 1, 1, 2>{});
}
bool rowblock_supported(int M, int N, int K, bool norm) {
    return M >= 1 && M <= kRbMaxRows && (M <= 16 || (long)N * K <= (12l << 20) || (N + 31) / 32 > 256) && K % 128 == 0 && N >= 1 && (N + 31) / 32 < 768 && (!norm || (M <= 16 && K <= 4096)) &&
           rb_shape(M, N, K, norm, [&](auto s) { return decltype(s)::lds(M, K, norm); }) <= 160 * 1024;
}

template <typename T, typename S, int EPI, int NORM>
static int rb_go(const void *act, const void *pk, const void *scale, const void *res, const void *norm_w, void *out, int M, int N, int K, float eps,
                 hipStream_t s) {
    static size_t lds_set = 64 * 1024;
    const size_t lds = S::lds(M, K, NORM > 0);
    if (lds > lds_set) {
        MYNN_HIP(hipFuncSetAttribute((const void *)rowblock_gemm_kernel<T, S, EPI, NORM>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        lds_set = 160 * 1024;
    }
    constexpr int rows = S::RB * S::RH;
    MYNN_LAUNCH((rowblock_gemm_kernel<T, S, EPI, NORM>), dim3((N + rows - 1) / rows), dim3(S::WAVES * 64), lds, s, (const T *)act,
                (const U4 *)pk, (const T *)scale, (const T *)res, (const T *)norm_w, (T *)out, M, N, K, eps);
    return launch_status("rowblock_gemm_kernel");
}

int rowblock_gemm(void *out, const void *act, const void *packed, const void *scale, const void *res, const void *norm_w, float eps, int M, int N,
                  int K, int dtype, int epi, hipStream_t s) {
    MYNN_REQUIRE(out && act && packed && scale && (epi != GEMM_RESIDUAL || res), MYNN_ERR_INVALID, "rowblock_gemm: null operand");
    MYNN_REQUIRE(rowblock_supported(M, N, K, norm_w != nullptr) && (epi != GEMM_SWIGLU || N % 2 == 0), MYNN_ERR_UNSUPPORTED, "rowblock_gemm: M=%d N=%d K=%d", M, N, K);
    MYNN_REQUIRE(aligned16(act) && aligned16(packed) && (!norm_w || aligned16(norm_w)), MYNN_ERR_INVALID, "rowblock_gemm: operands must be 16-byte aligned");
    return dispatch_dtype16(dtype, [&](auto *t) {
        using T = std::remove_pointer_t<decltype(t)>;
        return rb_shape(M, N, K, norm_w != nullptr, [&](auto shape) {
            using S = decltype(shape);
            auto go = [&](auto e) {
                constexpr int EPI = decltype(e)::value;
                if constexpr (S::ROWS <= 32 && !(S::ROWS == 32 && S::RH == 16)) {  // (the shapes of up to 16 rows)
                    if (norm_w && K <= 2048) return rb_go<T, S, EPI, 4>(act, packed, scale, res, norm_w, out, M, N, K, eps, s);
                    if constexpr (S::RB != 3)
                        if (norm_w) return rb_go<T, S, EPI, 8>(act, packed, scale, res, norm_w, out, M, N, K, eps, s);
                }
                return rb_go<T, S, EPI, 0>(act, packed, scale, res, norm_w, out, M, N, K, eps, s);
            };
            if (epi == GEMM_RESIDUAL) return go(std::integral_constant<int, GEMM_RESIDUAL>{});
            if (epi == GEMM_SWIGLU) return go(std::integral_constant<int, GEMM_SWIGLU>{});
            return go(std::integral_constant<int, GEMM_PLAIN>{});
        });
    });
}

}  // namespace mynn
