// Int8 weight-dequant GEMV for gfx950 (wave64): out[m,n] = T(scale[n] * sum_k act[m,k] * wq[n,k]).
//
// Replaces the reference's dequant_gemv.cuh:12-59 (one 32-lane warp per row) and
// dequant_matmul.cuh:12-51 (the scale-after-sum fallback for 1 < M < 16).
//
// Shape of the kernel: the weight matrix [N,K] int8 is streamed exactly once with 128-bit
// loads (16 weights per lane per load); the activation row(s) are staged once per workgroup in
// LDS as f32; each wave owns R consecutive rows so R independent 16-byte loads per lane are in
// flight before the first FMA; dequantisation is an in-register int8->f32 convert; the f32
// partial sums are combined with a wave64 xor butterfly; the scale is applied after the sum, as
// the reference does.  Optional fused prologue/epilogues keep the decoder at five launches per
// layer:
//   NORM      RMSNorm of the activation row computed while it is staged (rms_norm.cuh:9-59
//             semantics: y = (x * (1/sqrt(mean(x^2)+eps))) * w, rounded to T like the stored tensor)
//   RESIDUAL  out = T(T(acc*scale) + residual[n])            (the Add that follows o/down proj)
//   SWIGLU    rows interleaved gate,up: out[i] = T(silu(T(g)) * T(u))  (Swish+Mul group)
#include "kernels.h"
#include "gemv_dot.h"

namespace mynn {

enum { EPI_PLAIN = 0, EPI_RESIDUAL = 1, EPI_SWIGLU = 2 };

struct GemvParams {
    void *out;
    const void *act;       // [MB, K]
    const int8_t *wq;      // [N, K]
    const void *scale;     // [N]
    const void *residual;  // [MB, N_out] (EPI_RESIDUAL)
    const void *norm_w;    // [K] (NORM)
    float eps;
    int N, K;
    int act_stride;        // elements between activation rows
    int out_stride;        // elements between output rows
    // ARGMAX (the decode step's lm_head): the greedy token is found by the same launch.  Every GEMV workgroup leaves
    // its best (value, row) in cand[block] (one 8-byte word, row low / value bits high, ~0 = "empty" between launches);
    // one more workgroup waits for them (bounded spin, error word), takes the best, moves the loop state on and empties
    // the words again.
    uint64_t *cand;
    int32_t *next;
    AdvanceState adv;
    int *err;
    int spin_limit;
    uint64_t *fill;        // optional: fill_words words that this launch sets to ~0 (the hand-over vectors of the
    int fill_words;        // fused q|k|v + attention + o launch, emptied between two of its uses)
};

constexpr int kGemvWaves = 4;
constexpr int kGemvThreads = kGemvWaves * kWave;

template <typename TA, typename TO, int R, int MB, int EPI, bool NORM>
__global__ __launch_bounds__(kGemvThreads) void dequant_gemv_kernel(GemvParams p) {
    extern __shared__ float act_lds[];  // [MB][K]
    __shared__ float red[kGemvWaves];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int K = p.K, N = p.N;
    const TA *act = (const TA *)p.act;

    // ---- stage the activation row(s) in LDS as f32 (with the RMSNorm prologue when asked)
    if constexpr (NORM) {
        static_assert(!NORM || MB == 1, "norm prologue is a decode (one row) feature");
        float ss = 0.f;
        for (int k = tid; k < K; k += kGemvThreads) {
            float v = Elem<TA>::ld(act, k);
            act_lds[k] = v;
            ss += v * v;
        }
        ss = wave_sum(ss);
        if (lane == 0) red[wave] = ss;
        __syncthreads();
        float tot = 0.f;
#pragma unroll
        for (int w = 0; w < kGemvWaves; w++) tot += red[w];
        const float inv = 1.0f / sqrtf(tot / (float)K + p.eps);
        const TA *nw = (const TA *)p.norm_w;
        for (int k = tid; k < K; k += kGemvThreads)
            act_lds[k] = Elem<TA>::rnd((act_lds[k] * inv) * Elem<TA>::ld(nw, k));
    } else {
#pragma unroll
        for (int m = 0; m < MB; m++)
            for (int k = tid; k < K; k += kGemvThreads)
                act_lds[m * K + k] = Elem<TA>::ld(act, (size_t)m * p.act_stride + k);
    }
    __syncthreads();

    // ---- each wave: R rows
    const int row0 = (blockIdx.x * kGemvWaves + wave) * R;
    if (row0 >= N) return;
    const U4 *wrow[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        int row = row0 + r < N ? row0 + r : N - 1;
        wrow[r] = (const U4 *)(p.wq + (size_t)row * K);
    }
    float acc[R][MB];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int m = 0; m < MB; m++) acc[r][m] = 0.f;

    const int nchunks = K >> 4;
    for (int c = lane; c < nchunks; c += kWave) {
        U4 w[R];
#pragma unroll
        for (int r = 0; r < R; r++) w[r] = __builtin_nontemporal_load(&wrow[r][c]);
        float a[MB][16];
#pragma unroll
        for (int m = 0; m < MB; m++) {
            const float4 *ap = (const float4 *)(act_lds + m * K + c * 16);
#pragma unroll
            for (int q = 0; q < 4; q++) {
                float4 t = ap[q];
                a[m][4 * q] = t.x; a[m][4 * q + 1] = t.y; a[m][4 * q + 2] = t.z; a[m][4 * q + 3] = t.w;
            }
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            float wf[16];
            widen16_i8(w[r], wf);
#pragma unroll
            for (int m = 0; m < MB; m++)
#pragma unroll
                for (int i = 0; i < 16; i++) acc[r][m] = fmaf(a[m][i], wf[i], acc[r][m]);
        }
    }
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int m = 0; m < MB; m++) acc[r][m] = wave_sum(acc[r][m]);

    // ---- epilogue: lane r finishes row r
    const TO *scale = (const TO *)p.scale;
    TO *out = (TO *)p.out;
    if constexpr (EPI == EPI_SWIGLU) {
        static_assert(EPI != EPI_SWIGLU || (R % 2 == 0), "gate/up rows come in pairs");
#pragma unroll
        for (int r = 0; r < R; r += 2) {
            if (lane == r && row0 + r + 1 < N) {
#pragma unroll
                for (int m = 0; m < MB; m++) {
                    float g = Elem<TO>::rnd(acc[r][m] * Elem<TO>::ld(scale, row0 + r));
                    float u = Elem<TO>::rnd(acc[r + 1][m] * Elem<TO>::ld(scale, row0 + r + 1));
                    float sig = 1.0f / (1.0f + expf(-g));
                    Elem<TO>::st(out, (size_t)m * p.out_stride + ((row0 + r) >> 1), (g * sig) * u);
                }
            }
        }
    } else {
#pragma unroll
        for (int r = 0; r < R; r++) {
            if (lane == r && row0 + r < N) {
#pragma unroll
                for (int m = 0; m < MB; m++) {
                    float y = acc[r][m] * Elem<TO>::ld(scale, row0 + r);
                    size_t o = (size_t)m * p.out_stride + row0 + r;
                    if constexpr (EPI == EPI_RESIDUAL)
                        y = Elem<TO>::rnd(y) + Elem<TO>::ld((const TO *)p.residual, o);
                    Elem<TO>::st(out, o, y);
                }
            }
        }
    }
}

// Decode form (one activation row, 16-bit types).  A workgroup stages the activation row ONCE
// in LDS as f32 (128-bit global loads; with NORM the RMSNorm statistics come from the same
// registers: one butterfly + one cross-wave step), then its waves walk row groups of R rows
// (group g, g + total_waves, ...).  For a group every lane issues all R x NC 16-byte weight loads
// before the first multiply, dequantises in registers (int8 -> f32 convert + FMA) and the partial
// sums meet in a wave64 butterfly; the scale is applied after the sum.  NC = ceil(K / 1024).
// D < NC: only D chunks of each row are in flight, the next is asked for when one is used up: with all of a long row at once the
// device delivers less (fp16, us, all / D as in gemv1_dispatch: 4096 x 14336 13.4 / 10.5, 8192 x 14000 24.8 / 19.2, 2048 x 9600 7.3 /
// 5.3, 8192 x 8192 13.5 / 12.7, 4096 x 6000 6.2 / 5.8; bf16 12.6 / 10.8, 21.0 / 19.4, 6.8 / 5.2, 13.1 / 12.7, 6.4 / 5.6; rows of up to
// 4096 are short enough: 28672 x 4096 19.8 us whatever D).
// What the first loads need (pointers, sizes) are leading scalar arguments: they arrive preloaded in SGPRs with
// the wave (-amdgpu-kernarg-preload-count) instead of through a scalar load from the kernarg segment.
//
// Waves a SIMD whose registers a form is held to (1: left alone).  Left alone the compiler took 154 registers for 14 chunks of fp16
// (4096 x 14336 11.5 us, 5120 x 13824 16.0 against 13.5), and scheduled the short rows no better (batch-1 generation 0.3 %); held to eight
// waves a step of 8B widths takes a fifth longer, to three 2 % of the TinyLlama shape.  With a norm over more than 8192 values a thread's
// activation and norm pieces (56 registers) join its weights (40): that fits three waves (133 .. 136 registers) but not four, where 21
// to 27 of them went through scratch memory (batch-1 steps of two layers, vocabulary 32000, hidden 9216 / 12288 / 14336, us, four waves
// with the values kept in f32 as well / so: fp16 294, 436, 516 / 250, 360, 433; bf16 311, 456, 536 / 256, 368, 439).
// bf16 rows of 4097 to 6144 values are left alone: scheduled for four waves, the staging of the activation waited for the first weights too
// (us, all chunks at once / a ring, held / a ring, left alone: 512 x 4608 3.26 / 3.52 / 3.09, 2048 x 5120 4.06 / 4.32 / 3.64, 2048 x 5632 4.33 / 4.54 /
// 3.88, 4096 x 6144 6.49 / 5.80 / 5.55, 11264 x 6144 13.5 / 12.0 / 11.9).  So are rows of 1025 to 2048 without a norm (fp16, held / left alone: 32000 x
// 1280 8.73 / 7.97, 32000 x 1536 9.48 / 9.09, 4096 x 2048 3.25 / 3.15, 32000 x 2048 11.17 / 11.24; bf16 32000 x 1536 9.84 / 9.22).
template <typename T, int R, int NC, int D, bool NORM> constexpr int gemv1_waves() {
    if (R * D > 10 || (!std::is_same<T, f16_t>::value && NC == 6) || (!NORM && NC == 2)) return 1;
    return NORM && NC > 8 ? 3 : 4;
}
template <typename T, int R, int NC, int EPI, bool NORM, bool ARGMAX = false, int D = NC>
__global__ __launch_bounds__(kGemvThreads, (gemv1_waves<T, R, NC, D, NORM>())) void dequant_gemv1_kernel(const int8_t *wq, const void *act, const void *scale_p, const void *norm_w,
                                                                       const void *residual, int N, int K, int groups,
                                                                       int total_waves, GemvParams p) {
    extern __shared__ float act_lds[];  // [K]
    __shared__ float red[kGemvWaves];
    __shared__ float best_v[kGemvWaves];
    __shared__ int best_i[kGemvWaves];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    float bv = -INFINITY;  // ARGMAX: this thread's best stored value and its row
    int bi = -1;
    auto meet = [&]() {  // best of the workgroup in thread 0
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const float ov = __shfl_xor(bv, off, kWave);
            const int oi = __shfl_xor(bi, off, kWave);
            if (oi >= 0) argmax_take(bv, bi, ov, oi);
        }
        if (lane == 0) { best_v[wave] = bv; best_i[wave] = bi; }
        __syncthreads();
        if (tid == 0)
            for (int w = 1; w < kGemvWaves; w++)
                if (best_i[w] >= 0) argmax_take(bv, bi, best_v[w], best_i[w]);
    };
    if constexpr (ARGMAX) {
        if (blockIdx.x == gridDim.x - 1) {
            // ---- the extra workgroup: every GEMV workgroup's candidate -> the token, the loop state moves on
            const int nb = gridDim.x - 1;
            int st_step = 0, st_past = 0, st_active = 0;
            int64_t st_pos = 0;
            if (p.adv.ids && tid == 0) {
                st_step = *p.adv.step;
                st_pos = p.adv.pos[0];
                st_past = *p.adv.past;
                st_active = *p.adv.active;
            }
            // a thread's candidate words are asked for together every round: one round trip per round, not per word
            constexpr int CW = (kGemvArgmaxWords + kGemvThreads - 1) / kGemvThreads;
            uint64_t w[CW];
            for (int spins = 0;; spins++) {
                bool empty = false;
#pragma unroll
                for (int k = 0; k < CW; k++) {
                    const int i = tid + k * kGemvThreads;
                    w[k] = i < nb ? __hip_atomic_load(p.cand + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : 0ull;
                }
#pragma unroll
                for (int k = 0; k < CW; k++) empty = empty || w[k] == ~0ull;
                if (!empty) break;
                if (spins > p.spin_limit) {
                    __hip_atomic_store(p.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
#pragma unroll
            for (int k = 0; k < CW; k++) {
                const int i = tid + k * kGemvThreads;
                if (i < nb) {
                    const int oi = (int)(uint32_t)w[k];
                    if (w[k] != ~0ull && oi >= 0) argmax_take(bv, bi, __builtin_bit_cast(float, (uint32_t)(w[k] >> 32)), oi);
                    p.cand[i] = ~0ull;  // empty again for the next launch
                }
            }
            meet();
            if (tid == 0) {
                p.next[0] = bi;
                if (p.adv.ids) {
                    if (st_step < p.adv.cap) p.adv.tokens[st_step] = bi;
                    *p.adv.step = st_step + 1;
                    p.adv.ids[0] = bi;
                    p.adv.pos[0] = st_pos + 1;
                    *p.adv.past = st_past + 1;
                    *p.adv.active = st_active + 1;
                }
            }
            return;
        }
    }
    const int nchunks = K >> 4;
    int g = blockIdx.x * kGemvWaves + wave;

    // one row group's operands: R x NC weight chunks per lane, plus, in lane r < R, what the store of row r
    // needs (scale, the next row's scale for SwiGLU, the residual) -- fetched with the weights, not after the sum
    struct Group {
        U4 w[R][D];
        T sc, sc1, res;  // as loaded: widening them here would make the wave wait for every load above
    };
    const T *scale = (const T *)scale_p;
    // (unconditional: the wait for the activation can then be counted exactly; chunks past K are not used)
    auto load_chunk = [&](int gg, Group &G, int r, int j) {
        const int row = gg * R + r < N ? gg * R + r : N - 1;
        G.w[r][j % D] = __builtin_nontemporal_load((const U4 *)(wq + (size_t)row * K) + min(lane + j * kWave, nchunks - 1));
    };
    auto load_group = [&](int gg, Group &G) {
#pragma unroll
        for (int i = 0; i < R * D; i++) load_chunk(gg, G, D == NC ? i / D : i % R, D == NC ? i % D : i / R);
        const int row = min(gg * R + min(lane, R - 1), N - 1);
        G.sc = scale[row];
        if constexpr (EPI == EPI_SWIGLU) G.sc1 = scale[min(row + 1, N - 1)];
        if constexpr (EPI == EPI_RESIDUAL) G.res = ((const T *)residual)[row];
    };
    // the activation pieces (and their norm weights) are requested FIRST: loads return in order, so a wave that asked
    // for its weights before them would sit out the whole weight fetch before it could stage anything
    const int npieces = K >> 3;
    constexpr int PMAX = (NC * 1024 / 8 + kGemvThreads - 1) / kGemvThreads;  // pieces per thread
    U4 apv[PMAX], nwv[NORM ? PMAX : 1];
#pragma unroll
    for (int q = 0; q < PMAX; q++) {
        const int pc = tid + q * kGemvThreads;
        if (pc < npieces) {
            apv[q] = ((const U4 *)act)[pc];
            if constexpr (NORM) nwv[q] = ((const U4 *)norm_w)[pc];
        }
    }
    Group ga;
    load_group(min(g, groups - 1), ga);  // in flight while the activation is staged

    // ---- stage: thread t owns the 8-element pieces t, t + 256, ... of the row
    {
        float f[PMAX][8];
        float ss = 0.f;
#pragma unroll
        for (int q = 0; q < PMAX; q++) {
            const int pc = tid + q * kGemvThreads;
            if (pc < npieces) {
                widen8<T>(apv[q], f[q]);
                if constexpr (NORM) {
#pragma unroll
                    for (int i = 0; i < 8; i++) ss = fmaf(f[q][i], f[q][i], ss);
                }
            }
        }
        float inv = 1.f;
        if constexpr (NORM) {
            ss = wave_sum(ss);
            if (lane == 0) red[wave] = ss;
            __syncthreads();
            float tot = 0.f;
#pragma unroll
            for (int i = 0; i < kGemvWaves; i++) tot += red[i];
            inv = 1.0f / sqrtf(tot / (float)K + p.eps);
        }
#pragma unroll
        for (int q = 0; q < PMAX; q++) {
            const int pc = tid + q * kGemvThreads;
            if (pc < npieces) {
                if constexpr (NORM) {
                    if constexpr (PMAX > 4) {  // (widened again: a long row's values held in f32 over the barrier would be 56 registers more)
                        pin(apv[q]);
                        widen8<T>(apv[q], f[q]);
                    }
                    float nw[8];
                    widen8<T>(nwv[q], nw);
#pragma unroll
                    for (int i = 0; i < 8; i++) f[q][i] = Elem<T>::rnd((f[q][i] * inv) * nw[i]);
                }
                gemv_stage_piece<T>(act_lds, K, pc, f[q]);
            }
        }
    }
    __syncthreads();

    T *out = (T *)p.out;
    auto compute = [&](int gg, Group &G) {
        float acc[R];
        if constexpr (D == NC) gemv_rows_dot<T, R, NC>(act_lds, K, lane, G.w, acc);
        else gemv_rows_dot<T, R, NC, D>(act_lds, K, lane, G.w, acc, [&](int j) {
#pragma unroll
            for (int r = 0; r < R; r++) load_chunk(gg, G, r, j);
        });
#pragma unroll
        for (int r = 0; r < R; r++) acc[r] = wave_sum(acc[r]);
        const int row0 = gg * R;
        // lane r finishes row r (SwiGLU: lane r = 0, 2, .. the pair r, r + 1): one pass for all rows of the group
        float mine = acc[0], next = R > 1 ? acc[1] : 0.f;
#pragma unroll
        for (int r = 1; r < R; r++) {
            if (lane == r) {
                mine = acc[r];
                if (r + 1 < R) next = acc[r + 1];
            }
        }
        if constexpr (EPI == EPI_SWIGLU) {
            if (lane < R && (lane & 1) == 0 && row0 + lane + 1 < N) {
                float gt = Elem<T>::rnd(mine * Elem<T>::ld(&G.sc, 0));
                float up = Elem<T>::rnd(next * Elem<T>::ld(&G.sc1, 0));
                float sig = 1.0f / (1.0f + expf(-gt));
                Elem<T>::st(out, (size_t)((row0 + lane) >> 1), (gt * sig) * up);
            }
        } else {
            if (lane < R && row0 + lane < N) {
                float y = mine * Elem<T>::ld(&G.sc, 0);
                if constexpr (EPI == EPI_RESIDUAL) y = Elem<T>::rnd(y) + Elem<T>::ld(&G.res, 0);
                Elem<T>::st(out, row0 + lane, y);
                if constexpr (ARGMAX) argmax_take(bv, bi, Elem<T>::rnd(y), row0 + lane);  // (the value as stored)
            }
        }
    };
    bool loaded = true;  // (requesting the next group into a second register set before these sums: measured, no gain)
    for (; g < groups; g += total_waves) {
        if (!loaded) load_group(g, ga);
        loaded = false;
        compute(g, ga);
    }
    if (p.fill && blockIdx.x == gridDim.x - 1)
        for (int i = tid; i < p.fill_words; i += kGemvThreads) p.fill[i] = ~0ull;
    if constexpr (ARGMAX) {
        meet();
        if (tid == 0) {
            // (a workgroup without rows leaves index -1: not ~0 as a word, since -inf's bits sit in the high half)
            const uint64_t word = (uint64_t)(uint32_t)bi | ((uint64_t)__builtin_bit_cast(uint32_t, bv) << 32);
            __hip_atomic_store(p.cand + blockIdx.x, word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}
template <typename T, int R, int NC, int EPI, bool NORM, bool ARGMAX = false, int D = NC>
static int launch_gemv1(const GemvParams &p, hipStream_t s) {
    const int groups = (p.N + R - 1) / R;
    const int max_waves = 256 * 16;  // four resident waves per SIMD (measured best of 8/12/16/20/24/32 per CU)
    const int passes = (groups + max_waves - 1) / max_waves;
    int waves = (groups + passes - 1) / passes;
    const int blocks = (waves + kGemvWaves - 1) / kGemvWaves;
    waves = blocks * kGemvWaves;
    MYNN_LAUNCH((dequant_gemv1_kernel<T, R, NC, EPI, NORM, ARGMAX, D>), dim3(blocks + (ARGMAX ? 1 : 0)), dim3(kGemvThreads),
                (size_t)p.K * sizeof(float), s, p.wq, p.act, p.scale, p.norm_w, p.residual, p.N, p.K, groups, waves, p);
    return launch_status("dequant_gemv1_kernel");
}

template <typename TA, typename TO, int R, int MB, int EPI, bool NORM>
static int launch_gemv(const GemvParams &p, hipStream_t s) {
    const int rows_per_block = kGemvWaves * R;
    dim3 grid((p.N + rows_per_block - 1) / rows_per_block);
    size_t lds = (size_t)MB * p.K * sizeof(float);
    MYNN_LAUNCH((dequant_gemv_kernel<TA, TO, R, MB, EPI, NORM>), grid, dim3(kGemvThreads), lds, s, p);
    return launch_status("dequant_gemv_kernel");
}

static int check_gemv(const GemvParams &p, int mb) {
    MYNN_REQUIRE(p.out && p.act && p.wq && p.scale, MYNN_ERR_INVALID, "dequant_gemv: null operand");
    MYNN_REQUIRE(p.N > 0 && p.K > 0, MYNN_ERR_INVALID, "dequant_gemv: N=%d K=%d", p.N, p.K);
    MYNN_REQUIRE(p.K % 16 == 0, MYNN_ERR_UNSUPPORTED, "dequant_gemv: K=%d is not a multiple of 16", p.K);
    MYNN_REQUIRE(aligned16(p.wq), MYNN_ERR_INVALID, "dequant_gemv: wq must be 16-byte aligned");
    MYNN_REQUIRE((size_t)mb * p.K * sizeof(float) <= 64 * 1024, MYNN_ERR_UNSUPPORTED,
                 "dequant_gemv: %d x K=%d activations do not fit the 64 KiB LDS stage", mb, p.K);
    return 0;
}

// Picks rows-per-wave so that small matrices still spread over the chip: 4 rows per wave when
// that leaves at least ~2 workgroups per CU, else 2.
static int pick_r(int N) { return N >= 256 * 2 * kGemvWaves * 4 ? 4 : 2; }

template <typename TA, typename TO, int MB>
static int gemv_plain(const GemvParams &p, hipStream_t s) {
    if (pick_r(p.N) == 4) return launch_gemv<TA, TO, 4, MB, EPI_PLAIN, false>(p, s);
    return launch_gemv<TA, TO, 2, MB, EPI_PLAIN, false>(p, s);
}

// out [M,N]; M in 1..15 handled in row tiles of at most 4 activation rows
template <typename TA, typename TO>
static int gemv_small_m(GemvParams p, int M, hipStream_t s) {
    const TA *act = (const TA *)p.act;
    TO *out = (TO *)p.out;
    int m = 0;
    while (m < M) {
        int mb = M - m >= 4 ? 4 : (M - m >= 2 ? 2 : 1);
        GemvParams q = p;
        q.act = act + (size_t)m * p.act_stride;
        q.out = out + (size_t)m * p.out_stride;
        int rc = check_gemv(q, mb);
        if (rc) return rc;
        rc = mb == 4 ? gemv_plain<TA, TO, 4>(q, s) : mb == 2 ? gemv_plain<TA, TO, 2>(q, s) : gemv_plain<TA, TO, 1>(q, s);
        if (rc) return rc;
        m += mb;
    }
    return 0;
}

// Fallback for shapes the streaming kernel does not take (K not a multiple of 16, unaligned
// weights): one wave per output element, scalar loads -- the reference's dequant_matmul.cuh:12-51.
template <typename TA, typename TO>
__global__ __launch_bounds__(64) void dequant_matmul_naive_kernel(TO *out, const TA *act, const int8_t *wq,
                                                                 const TO *scale, int N, int K) {
    const int n = blockIdx.x, m = blockIdx.y, lane = threadIdx.x;
    float acc = 0.f;
    for (int k = lane; k < K; k += 64) acc = fmaf(Elem<TA>::ld(act, (size_t)m * K + k), (float)wq[(size_t)n * K + k], acc);
    acc = wave_sum(acc);
    if (lane == 0) Elem<TO>::st(out, (size_t)m * N + n, acc * Elem<TO>::ld(scale, n));
}

template <typename T, int EPI, bool NORM>
static int gemv1_dispatch(const GemvParams &p, hipStream_t s);

// scale-after-sum path for any act/out type pair the reference allows (f32 or 16-bit act;
// out type = scale type)
int dequant_gemv_dispatch(void *out, const void *act, const int8_t *wq, const void *scale, int M, int N,
                          int K, int act_dtype, int out_dtype, hipStream_t s) {
    GemvParams p{};
    p.out = out; p.act = act; p.wq = wq; p.scale = scale; p.N = N; p.K = K; p.act_stride = K; p.out_stride = N;
    MYNN_REQUIRE(M >= 1, MYNN_ERR_INVALID, "dequant_gemv: M=%d", M);
    MYNN_REQUIRE(out && act && wq && scale && N > 0 && K > 0, MYNN_ERR_INVALID, "dequant_matmul: bad operand");
    MYNN_REQUIRE(dtype_ok(act_dtype) && dtype_ok(out_dtype), MYNN_ERR_INVALID, "dequant_matmul: dtype");
    const bool streaming = K % 16 == 0 && aligned16(wq) && M < 16 &&
                           (size_t)(M < 4 ? M : 4) * K * sizeof(float) <= 64 * 1024;
    return dispatch_dtype(act_dtype, [&](auto *ta) {
        using TA = std::remove_pointer_t<decltype(ta)>;
        return dispatch_dtype(out_dtype, [&](auto *to) {
            using TO = std::remove_pointer_t<decltype(to)>;
            if constexpr (std::is_same<TA, TO>::value && sizeof(TA) == 2) {
                if (streaming && M == 1) return gemv1_dispatch<TA, EPI_PLAIN, false>(p, s);
            }
            if (streaming) return gemv_small_m<TA, TO>(p, M, s);
            MYNN_REQUIRE(M <= 65535, MYNN_ERR_UNSUPPORTED, "dequant_matmul: M=%d too large for the plain kernel", M);
            MYNN_LAUNCH((dequant_matmul_naive_kernel<TA, TO>), dim3(N, M), dim3(64), 0, s, (TO *)out,
                               (const TA *)act, wq, (const TO *)scale, N, K);
            return launch_status("dequant_matmul_naive_kernel");
        });
    });
}

// ---- fused decode variants used by the decoder executor (one activation row, T in == T out)
template <typename T, int EPI, bool NORM>
static int gemv1_dispatch(const GemvParams &p, hipStream_t s) {
    const int nc = (p.K + 1023) / 1024;
    // four rows per wave: faster for short rows (gate/up at K = 2048: 6.1 against 6.35 us), slower for long ones
    // (down at K = 5632: 6.0 against 4.6 us, the wave holds 24 chunks per lane)
    const bool wide = nc <= 2;
    if (!aligned16(p.act) || (NORM && !aligned16(p.norm_w)) || p.K % 8 != 0 || nc > 14) {
        if (wide) return launch_gemv<T, T, 4, 1, EPI, NORM>(p, s);  // the looping kernel
        return launch_gemv<T, T, 2, 1, EPI, NORM>(p, s);
    }
#define MYNN_GEMV1(NC_)                                                   \
    return wide ? launch_gemv1<T, 4, NC_, EPI, NORM>(p, s) : launch_gemv1<T, 2, NC_, EPI, NORM>(p, s)
    if (nc <= 1) { MYNN_GEMV1(1); }
    if (nc <= 2) { MYNN_GEMV1(2); }
    if (nc <= 4) { MYNN_GEMV1(4); }
    if (nc <= 6) return launch_gemv1<T, 2, 6, EPI, NORM, false, 3>(p, s);
    if (nc <= 8) return launch_gemv1<T, 2, 8, EPI, NORM, false, 4>(p, s);
    if (nc <= 14) return launch_gemv1<T, 2, 14, EPI, NORM, false, 5>(p, s);
#undef MYNN_GEMV1
    // longer rows: the looping kernel
    if (wide) return launch_gemv<T, T, 4, 1, EPI, NORM>(p, s);
    return launch_gemv<T, T, 2, 1, EPI, NORM>(p, s);
}

// ---- measurement aid: the weight stream of dequant_gemv1_kernel and nothing else.  Same grid, same row groups per
// wave, the same non-temporal 16-byte loads per lane and group, R x NC with R x D of them in flight (long rows: D < NC, as gemv1_dispatch), no
// activation, no arithmetic beyond an xor that keeps the loads alive, no store.  Launched like the GEMV (dependent launches on one
// stream, a different matrix each time) it gives the time a launch of this geometry needs just to pull its bytes in: the floor the
// GEMV's duration is judged against.
template <int R, int NC, int D>
__global__ __launch_bounds__(kGemvThreads) void gemv_read_probe_kernel(const int8_t *wq, uint32_t *sink, int N, int K, int groups,
                                                                         int total_waves) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nchunks = K >> 4;
    uint32_t acc = 0;
    for (int g = blockIdx.x * kGemvWaves + wave; g < groups; g += total_waves) {
        U4 w[R][D];
        auto load = [&](int r, int j) {
            const int row = g * R + r < N ? g * R + r : N - 1;
            w[r][j % D] = __builtin_nontemporal_load((const U4 *)(wq + (size_t)row * K) + min(lane + j * kWave, nchunks - 1));
        };
#pragma unroll
        for (int i = 0; i < R * D; i++) load(D == NC ? i / D : i % R, D == NC ? i % D : i / R);
#pragma unroll
        for (int j = 0; j < NC; j++) {
#pragma unroll
            for (int r = 0; r < R; r++) {
                U4 &c = w[r][j % D];
                if constexpr (D < NC) pin(c);
                acc ^= c.x ^ c.y ^ c.z ^ c.w;
            }
            if constexpr (D < NC) {
                asm volatile("" : "+v"(acc)::"memory");  // (the next chunk is asked for when one is used up)
                if (j + D < NC) {
#pragma unroll
                    for (int r = 0; r < R; r++) load(r, j + D);
                }
            }
        }
    }
    if (acc == 0x9E3779B9u && sink) sink[0] = acc;  // (never true for the patterns the benchmark fills in; keeps the loads)
}
template <int R, int NC, int D = NC>
static int launch_read_probe(const int8_t *wq, uint32_t *sink, int N, int K, bool empty, hipStream_t s) {
    const int groups = (N + R - 1) / R;
    const int max_waves = 256 * 16;
    const int passes = (groups + max_waves - 1) / max_waves;
    int waves = (groups + passes - 1) / passes;
    const int blocks = (waves + kGemvWaves - 1) / kGemvWaves;
    waves = blocks * kGemvWaves;
    MYNN_LAUNCH((gemv_read_probe_kernel<R, NC, D>), dim3(blocks), dim3(kGemvThreads), 0, s, wq, sink, N, K, empty ? 0 : groups, waves);
    return launch_status("gemv_read_probe_kernel");
}

template <typename T>
int gemv_norm(void *out, const void *x, const void *norm_w, float eps, const int8_t *wq, const void *scale,
              int N, int K, hipStream_t s) {
    GemvParams p{};
    p.out = out; p.act = x; p.wq = wq; p.scale = scale; p.norm_w = norm_w; p.eps = eps; p.N = N; p.K = K;
    p.act_stride = K; p.out_stride = N;
    int rc = check_gemv(p, 1);
    if (rc) return rc;
    return gemv1_dispatch<T, EPI_PLAIN, true>(p, s);
}
// the decode step's lm_head: RMSNorm + GEMV + greedy token + loop state in one launch (cand: (N / 2 + 3) / 4 + 1
// words at most, all ~0 on entry and again on exit)
bool gemv_norm_argmax_supported(const void *x, const void *norm_w, const int8_t *wq, int N, int K) {
    return aligned16(x) && aligned16(norm_w) && aligned16(wq) && K % 16 == 0 && (K + 1023) / 1024 <= 14 && N > 0 &&
           (size_t)K * sizeof(float) <= 64 * 1024;
}
template <typename T>
int gemv_norm_argmax(void *out, const void *x, const void *norm_w, float eps, const int8_t *wq, const void *scale, int N, int K,
                     uint64_t *cand, int32_t *next, AdvanceState adv, int *err, int spin_limit, hipStream_t s) {
    GemvParams p{};
    p.out = out; p.act = x; p.wq = wq; p.scale = scale; p.norm_w = norm_w; p.eps = eps; p.N = N; p.K = K;
    p.act_stride = K; p.out_stride = N;
    p.cand = cand; p.next = next; p.adv = adv; p.err = err; p.spin_limit = spin_limit;
    MYNN_REQUIRE(cand && next && err && gemv_norm_argmax_supported(x, norm_w, wq, N, K), MYNN_ERR_UNSUPPORTED,
                 "gemv_norm_argmax: N=%d K=%d", N, K);
    const int nc = (K + 1023) / 1024;
    // (rows per wave and chunks in flight as gemv1_dispatch has them.  us a step of two layers over a long cache, vocabulary 128256, two rows per
    // wave / four: fp16, hidden 512 62.6 / 55.0, 1024 70.9 / 62.8; all chunks of a row at once / in a ring, bf16, hidden 5120 229 / 227, 6144 332 / 329)
    if (nc <= 1) return launch_gemv1<T, 4, 1, EPI_PLAIN, true, true>(p, s);
    if (nc <= 2) return launch_gemv1<T, 4, 2, EPI_PLAIN, true, true>(p, s);
    if (nc <= 4) return launch_gemv1<T, 2, 4, EPI_PLAIN, true, true>(p, s);
    if (nc <= 6) return launch_gemv1<T, 2, 6, EPI_PLAIN, true, true, 3>(p, s);
    if (nc <= 8) return launch_gemv1<T, 2, 8, EPI_PLAIN, true, true, 4>(p, s);
    return launch_gemv1<T, 2, 14, EPI_PLAIN, true, true, 5>(p, s);
}
template int gemv_norm_argmax<bf16_t>(void *, const void *, const void *, float, const int8_t *, const void *, int, int, uint64_t *,
                                      int32_t *, AdvanceState, int *, int, hipStream_t);
template int gemv_norm_argmax<f16_t>(void *, const void *, const void *, float, const int8_t *, const void *, int, int, uint64_t *,
                                     int32_t *, AdvanceState, int *, int, hipStream_t);

template <typename T>
int gemv_residual(void *out, const void *act, const int8_t *wq, const void *scale, const void *residual,
                  int N, int K, hipStream_t s) {
    GemvParams p{};
    p.out = out; p.act = act; p.wq = wq; p.scale = scale; p.residual = residual; p.N = N; p.K = K;
    p.act_stride = K; p.out_stride = N;
    int rc = check_gemv(p, 1);
    if (rc) return rc;
    return gemv1_dispatch<T, EPI_RESIDUAL, false>(p, s);
}
// wq/scale hold gate and up rows interleaved (row 2i = gate_i, row 2i+1 = up_i); N = 2*ffn
template <typename T>
int gemv_norm_swiglu(void *out, const void *x, const void *norm_w, float eps, const int8_t *wq,
                     const void *scale, int N, int K, hipStream_t s, uint64_t *fill, int fill_words) {
    GemvParams p{};
    p.out = out; p.act = x; p.wq = wq; p.scale = scale; p.norm_w = norm_w; p.eps = eps; p.N = N; p.K = K;
    p.act_stride = K; p.out_stride = N / 2;
    p.fill = fill; p.fill_words = fill_words;
    MYNN_REQUIRE(!fill || (aligned16(x) && aligned16(norm_w) && K % 8 == 0 && (K + 1023) / 1024 <= 14), MYNN_ERR_UNSUPPORTED,
                 "gemv_norm_swiglu: the fill rides on the decode kernel only");
    MYNN_REQUIRE(N % 2 == 0, MYNN_ERR_INVALID, "gate/up rows must come in pairs (N=%d)", N);
    int rc = check_gemv(p, 1);
    if (rc) return rc;
    return gemv1_dispatch<T, EPI_SWIGLU, true>(p, s);
}

template int gemv_norm<bf16_t>(void *, const void *, const void *, float, const int8_t *, const void *, int, int, hipStream_t);
template int gemv_norm<f16_t>(void *, const void *, const void *, float, const int8_t *, const void *, int, int, hipStream_t);
template int gemv_residual<bf16_t>(void *, const void *, const int8_t *, const void *, const void *, int, int, hipStream_t);
template int gemv_residual<f16_t>(void *, const void *, const int8_t *, const void *, const void *, int, int, hipStream_t);
template int gemv_norm_swiglu<bf16_t>(void *, const void *, const void *, float, const int8_t *, const void *, int, int, hipStream_t, uint64_t *, int);
template int gemv_norm_swiglu<f16_t>(void *, const void *, const void *, float, const int8_t *, const void *, int, int, hipStream_t, uint64_t *, int);

}  // namespace mynn

extern "C" int mynn_dequant_gemv(void *out, const void *act, const int8_t *wq, const void *scale, int N, int K,
                                 int act_dtype, int out_dtype, mynn_stream s) {
    MYNN_REQUIRE(K > 0 && K % 16 == 0, MYNN_ERR_UNSUPPORTED, "dequant_gemv: K=%d is not a multiple of 16", K);
    MYNN_REQUIRE(mynn::aligned16(wq), MYNN_ERR_INVALID, "dequant_gemv: wq must be 16-byte aligned");
    MYNN_REQUIRE((size_t)K * sizeof(float) <= 64 * 1024, MYNN_ERR_UNSUPPORTED, "dequant_gemv: K=%d exceeds the LDS stage", K);
    return mynn::dequant_gemv_dispatch(out, act, wq, scale, 1, N, K, act_dtype, out_dtype, mynn::as_stream(s));
}

extern "C" int mynn_gemv_read_probe(const int8_t *wq, void *sink, int N, int K, int empty, mynn_stream s) {
    using namespace mynn;
    MYNN_REQUIRE(wq && N > 0 && K > 0 && K % 16 == 0 && aligned16(wq), MYNN_ERR_INVALID, "gemv_read_probe: N=%d K=%d", N, K);
    const int nc = (K + 1023) / 1024;
    MYNN_REQUIRE(nc <= 14, MYNN_ERR_UNSUPPORTED, "gemv_read_probe: K=%d (the decode GEMV's row limit is 14336)", K);
    hipStream_t st = as_stream(s);
    // the geometry of gemv1_dispatch: four rows per wave for K <= 2048, two beyond
    if (nc <= 1) return launch_read_probe<4, 1>(wq, (uint32_t *)sink, N, K, empty != 0, st);
    if (nc <= 2) return launch_read_probe<4, 2>(wq, (uint32_t *)sink, N, K, empty != 0, st);
    if (nc <= 4) return launch_read_probe<2, 4>(wq, (uint32_t *)sink, N, K, empty != 0, st);
    if (nc <= 6) return launch_read_probe<2, 6, 3>(wq, (uint32_t *)sink, N, K, empty != 0, st);
    if (nc <= 8) return launch_read_probe<2, 8, 4>(wq, (uint32_t *)sink, N, K, empty != 0, st);
    return launch_read_probe<2, 14, 5>(wq, (uint32_t *)sink, N, K, empty != 0, st);
}
