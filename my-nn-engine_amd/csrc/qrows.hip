// QuantizedMatMul of 2 .. 128 rows, one launch without scratch memory: the streams of rowblock.hip with int8 on both sides.
//
//   out[m,n] = T((acc * a_scale[m]) * b_scale[n]), acc = sum_k lhs[m,k] * rhs[n,k] in exact int32 (the order does not matter)
//
// A workgroup owns 16 .. 64 rows of rhs and up to 32 of lhs (grid y) over all of K; its waves take steps of 128 k in turn.  A step is 128 bytes of every row, whole lines:
// both operands go global -> LDS by the load unit into rings that no other wave touches and are waited for by count; nobody meets
// anybody before the sums of the waves, in LDS at the end.  v_mfma_i32_16x16x64_i8: lane l holds row l % 16, k = 16 * (l / 16) .. +15.
//
// What bounds it: few rows, the weights; many, the lhs rows that every workgroup reads in full (some 80 KB a microsecond and CU).  As
// tiles of 32 x 64 (stages of 72 KB, up to 112 steps in series behind a barrier each) the same calls took, us, before / now: 8 rows,
// 2048 x 5632 8.3 / 5.2, 4096 x 4096 8.2 / 5.5, 4096 x 14336 16.7 / 11.1, 28672 x 4096 29.6 / 22.9; 32 rows 9.2 / 7.4, 8.5 / 6.8, 17.0 / 16.0, 29.8 / 28.3.
#include <type_traits>

#include "kernels.h"
#include "mfma.h"
#include "wave_ring.h"

namespace mynn {

// NB row blocks of 16 per workgroup, A8 groups of 8 lhs rows, ND stages, WAVES waves
template <int NB_, int A8_, int ND_, int WAVES_> struct QrShape {
    static constexpr int NB = NB_, A8 = A8_, ND = ND_, WAVES = WAVES_, MT = (A8 + 1) / 2;
    static constexpr int STAGE = (2 * NB + A8) * 1024, RED = 16 + 4;
    static size_t lds(int M) {
        const size_t st = (size_t)WAVES * ND * STAGE, red = (size_t)WAVES * NB * M * RED * 4;
        return st > red ? st : red;
    }
    static_assert(WAVES * ND * STAGE <= 160 * 1024 && WAVES * NB * A8 * 8 * RED * 4 <= 160 * 1024 && ND >= 2 && ND <= 8, "");
};
typedef int qi4_t __attribute__((ext_vector_type(4)));

template <typename T, typename S>
__global__ __launch_bounds__(S::WAVES * 64) void qrows_gemm_kernel(const int8_t *lhs, const int8_t *rhs, int M, int N, int K, const T *a_scale,
                                                                  const T *b_scale, T *out, int32_t *acc_out) {
    constexpr int NB = S::NB, A8 = S::A8, ND = S::ND, MT = S::MT, WAVES = S::WAVES, RS = S::RED;
    extern __shared__ __align__(16) char lds[];
    const int tid = threadIdx.x, lane = tid & 63, kw = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, h = lane >> 4;
    const int b0 = (int)blockIdx.x * NB, n0 = b0 * 16, m0 = (int)blockIdx.y * A8 * 8;
    lhs += (size_t)m0 * K;
    M = min(M - m0, A8 * 8);
    const int steps = K / 128, n = __builtin_amdgcn_readfirstlane((steps - kw + WAVES - 1) / WAVES);  // in all, of this wave
    char *ring = lds + kw * ND * S::STAGE;
    uint32_t aoff[A8], woff[2 * NB];
#pragma unroll
    for (int i = 0; i < A8; i++) aoff[i] = ring_chunk(lane, i, M - 1, K);
#pragma unroll
    for (int i = 0; i < 2 * NB; i++) woff[i] = ring_chunk(lane, i, N - 1 - n0, K);
    auto request = [&](int i, int slot) {
        const size_t k = (size_t)(i * WAVES + kw) * 128;
        const char *a = (const char *)lhs + k - 4096, *w = (const char *)rhs + (size_t)n0 * K + k - 4096;
        const uint32_t to = lds_offset(ring) + slot * S::STAGE;
        load_group_to_lds<(NB < 2 ? 2 : 4), true>(w, woff, to);
        if constexpr (NB > 2) load_group_to_lds<2 * NB - 4, true>(w, woff + 4, to + 4096);
        load_group_to_lds<A8>(a, aoff, to + 2 * NB * 1024);
    };
    qi4_t acc[NB][MT];
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int t = 0; t < MT; t++) acc[b][t] = qi4_t{0, 0, 0, 0};
    const int fr = A8 == 1 ? r & 7 : r;  // (rows past the loaded ones: columns that are not stored)
    qi4_t w[2][NB], a[2][MT];
    auto use = [&](int slot) {
        const char *st = ring + slot * S::STAGE;
#pragma unroll
        for (int x = 0; x < 2; x++) {
#pragma unroll
            for (int b = 0; b < NB; b++) w[x][b] = *(const qi4_t *)(st + b * 2048 + r * 128 + (((4 * x + h) ^ (r & 7)) << 4));
#pragma unroll
            for (int t = 0; t < MT; t++) a[x][t] = *(const qi4_t *)(st + 2 * NB * 1024 + t * 2048 + fr * 128 + (((4 * x + h) ^ (fr & 7)) << 4));
        }
    };
    auto multiply = [&]() {
#pragma unroll
        for (int x = 0; x < 2; x++)
#pragma unroll
            for (int b = 0; b < NB; b++)
#pragma unroll
                for (int t = 0; t < MT; t++) acc[b][t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(w[x][b], a[x][t], acc[b][t], 0, 0, 0);
    };
    constexpr int C = A8 + 2 * NB;  // loads of a step
    int i = 0, slot = 0;
#pragma unroll
    for (int d = 0; d < ND - 1; d++)
        if (d < n) request(d, d);
    for (; i + ND - 1 < n; i++) {
        wait_for_loads<(ND - 2) * C>();
        use(slot);
        request(i + ND - 1, slot == 0 ? ND - 1 : slot - 1);  // (the stage that the step before was read from)
        multiply();
        slot = slot + 1 == ND ? 0 : slot + 1;
    }
    // the last ND - 1 steps, with nothing left to ask for
    auto rest = [&](auto left) {
        constexpr int L = decltype(left)::value;
        if constexpr (L < ND) {
            if (n - i != L) return;
            wait_for_loads<(L - 1) * C>();
            use(slot);
            multiply();
            slot = slot + 1 == ND ? 0 : slot + 1;
            i++;
        }
    };
    rest(std::integral_constant<int, 7>{});
    rest(std::integral_constant<int, 6>{});
    rest(std::integral_constant<int, 5>{});
    rest(std::integral_constant<int, 4>{});
    rest(std::integral_constant<int, 3>{});
    rest(std::integral_constant<int, 2>{});
    rest(std::integral_constant<int, 1>{});
    __syncthreads();  // the rings are done with: their memory takes the sums
    int *red = (int *)lds;
#pragma unroll
    for (int b = 0; b < NB; b++)
#pragma unroll
        for (int t = 0; t < MT; t++) {
            const int m = t * 16 + r;
            if (m < M) *(qi4_t *)(red + ((size_t)(kw * NB + b) * M + m) * RS + 4 * h) = acc[b][t];
        }
    __syncthreads();
    for (int o = tid; o < NB * M * 16; o += WAVES * 64) {
        const int c = o % 16, m = (o / 16) % M, b = o / (16 * M), col = (b0 + b) * 16 + c;
        if (col >= N) continue;
        int t = 0;
#pragma unroll
        for (int k = 0; k < WAVES; k++) t += red[((size_t)(k * NB + b) * M + m) * RS + c];
        const size_t at = (size_t)(m0 + m) * N + col;
        if (acc_out) acc_out[at] = t;
        if (out) Elem<T>::st(out, at, ((float)t * Elem<T>::ld(a_scale, m0 + m)) * Elem<T>::ld(b_scale, col));
    }
}

// One workgroup per CU of as many row blocks as that takes up to 12288 rows of rhs (up to 16 rows of lhs: 16384); beyond, four waves, two
// workgroups per CU, whose ramps and stores overlap (us, eight waves / four: 28672 x 4096, 8 rows 23.8 with 64 rows each / 22.9, 32 rows
// 30.7 with 48 / 28.3 with 32; 14336 x 4096, 8 rows 12.4 / 14.3 with 64, 32 rows 19.6 with 48 / 14.9 with 32).
template <typename F> static int qr_shape(int M, int N, F &&f) {
    auto form = [&](auto b, auto waves, auto groups) {
        constexpr int NB = decltype(b)::value, A8 = decltype(groups)::value, D = 20 / (2 * NB + A8);
        return f(QrShape<NB, A8, D < 8 ? D : 8, decltype(waves)::value>{});
    };
    using std::integral_constant;
    const long cols = (long)N * ((M + 31) / 32);  // (as many workgroups as one group of rows of a matrix so wide)
    auto by_columns = [&](auto groups) {
        constexpr integral_constant<int, 8> eight;
        constexpr integral_constant<int, 4> four;
        if (cols <= 256 * 16) return form(integral_constant<int, 1>{}, eight, groups);
        if (cols <= 256 * 32) return form(integral_constant<int, 2>{}, eight, groups);
        if (cols <= 256 * 48) return form(integral_constant<int, 3>{}, eight, groups);
        if constexpr (decltype(groups)::value <= 2) return cols <= 256 * 64 ? form(four, eight, groups) : form(four, four, groups);
        else return form(integral_constant<int, 2>{}, four, groups);
    };
    if (M <= 8) return by_columns(integral_constant<int, 1>{});
    if (M <= 16) return by_columns(integral_constant<int, 2>{});
    return by_columns(integral_constant<int, 4>{});
}
template <typename T, typename S>
static int qr_go(const int8_t *lhs, const int8_t *rhs, const void *a_scale, const void *b_scale, void *out, int32_t *acc_out, int M, int N, int K, hipStream_t s) {
    static size_t lds_set = 64 * 1024;
    const size_t lds = S::lds(M < S::A8 * 8 ? M : S::A8 * 8);
    if (lds > lds_set) {
        MYNN_HIP(hipFuncSetAttribute((const void *)qrows_gemm_kernel<T, S>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
        lds_set = 160 * 1024;
    }
    MYNN_LAUNCH((qrows_gemm_kernel<T, S>), dim3((N + S::NB * 16 - 1) / (S::NB * 16), (M + S::A8 * 8 - 1) / (S::A8 * 8)), dim3(S::WAVES * 64), lds, s, lhs, rhs, M, N, K, (const T *)a_scale,
                (const T *)b_scale, (T *)out, acc_out);
    return launch_status("qrows_gemm_kernel");
}

bool qrows_supported(int M, int N, int K) { return M >= 2 && M <= 128 && N >= 1 && K >= 128 && K % 128 == 0; }
// Where it is the form to take (us a call with weights that are not cached, dot products (two rows) or tiles / so; profiles/few_row_times.csv has
// both over 4000 shapes; a call of tiles costs the host some 5.4 us, of the streams 4.4).
//   Two rows: up to 4096 weight rows (2048 x 5632 6.2 / 5.0, 4096 x 4096 6.1 / 5.3), beyond, not where rows of whole 8192 bytes (8192 x 8192 14.5 / 16.8;
//   but three row blocks of 16: 10240 x 8192 16.7 / 15.6), with two workgroups of streams per CU whole 4096, meet at the same channels of the
//   memory (16384 x 16384 44.9 / 52.5); more than 16384 weight rows where rows are short (28672 x 1024 8.8 / 6.8, x 4096 21.5 / 22.2).
//   Few weight rows leave most CUs without a workgroup, and what one reads for itself, 16 weight rows and the lhs rows over all of K, outlasts K
//   ranges over the device from some 500 KB on (8 rows, 500 x 14336 9.8 / 8.5, x 32768 12.8 / 15.3; 32 rows, 1024 x 6144 8.8 / 7.8, x 32768 15.5 /
//   26.6); with 1536 weight rows 650, and with up to 16 of lhs 1000 KB; a workgroup on every CU, 32 rows, 4096 x 14336 16.8 / 15.6, x 32768 32.1 / 32.0.
//   17 .. 32 rows otherwise: 5120 x 14336 18.8 / 20.9; with three row blocks, and beyond 12288 weight rows where rows are below 8192 bytes (32 rows, 9216 x
//   1024 6.3 / 5.6, 12288 x 4096 13.7 / 12.4, 14336 x 2048 8.6 / 8.9, 32000 x 4096 33.4 / 28.9, x 8192 56.6 / 65.6; ragged rows of the output cost the tiles
//   more: 9219 x 1024 6.9 / 5.8).
//   More: groups of 32 rows where a narrow matrix leaves CUs for them (64 rows, 2048 x 4096 8.1 / 6.0, x 6144 9.4 / 7.7, 2560 x 4096 8.6 / 7.7, x 5632
//   9.3 / 9.4; 128 rows, 2048 x 5632 10.0 / 9.1, 1024 x 6144 9.1 / 7.3, but 160 x 6144 8.2 / 8.6; with weights that are still cached, 73 rows, 2048 x 5632 8.5 /
//   6.3), or rows are so short that the host's time decides.
bool qrows_first(int M, int N, int K) {
    if (!qrows_supported(M, N, K)) return false;
    const long reads = (16 + 2l * M) * K, cols = (long)N * ((M + 31) / 32);
    if (M == 2) {
        if (N <= 256 * 32) return N <= 256 * 16 || K % 8192 != 0;
        return N <= 256 * 48 || (N <= 256 * 64 ? K % 4096 != 0 : K <= 2560);
    }
    if (M <= 16) return N >= 2304 || reads <= (N < 1536 ? 525000 : 1000000);
    if (M <= 32) {
        if (N < 3072) return reads <= (N < 1536 ? 525000 : 650000);
        if (N <= 256 * 16) return reads <= 1700000;
        if (N <= 256 * 32) return N > 256 * 22 || K <= 8192;
        return N <= 256 * 48 || K < 8192;
    }
    if (cols <= 256 * 16) return K <= (N >= 256 ? 8192 : 4096);
    return cols <= 256 * 32 ? K <= 6144 : cols <= 256 * 64 && K <= 640;
}
int qrows_gemm(void *out, int32_t *acc_out, const int8_t *lhs, const void *a_scale, const int8_t *rhs, const void *b_scale, int M, int N, int K, int dtype,
               hipStream_t s) {
    MYNN_REQUIRE((out || acc_out) && lhs && rhs && (!out || (a_scale && b_scale)), MYNN_ERR_INVALID, "qrows_gemm: null operand");
    MYNN_REQUIRE(qrows_supported(M, N, K) && K <= 131071, MYNN_ERR_UNSUPPORTED, "qrows_gemm: M=%d N=%d K=%d", M, N, K);
    MYNN_REQUIRE(aligned16(lhs) && aligned16(rhs), MYNN_ERR_INVALID, "qrows_gemm: operands must be 16-byte aligned");
    return dispatch_dtype(dtype, [&](auto *t) {
        using T = std::remove_pointer_t<decltype(t)>;
        return qr_shape(M, N, [&](auto shape) { return qr_go<T, decltype(shape)>(lhs, rhs, a_scale, b_scale, out, acc_out, M, N, K, s); });
    });
}

}  // namespace mynn

// For the tests and for measuring: the two forms of a product of few rows side by side; not part of the library's interface.
extern "C" int mynn_few_rows_first(int int8_lhs, int M, int N, int K) { return int8_lhs ? mynn::qrows_first(M, N, K) : mynn::rowblock_rows_first(M, N, K); }
