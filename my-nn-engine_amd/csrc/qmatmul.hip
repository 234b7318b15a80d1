// QuantizedMatMul (W8A8): acc[m,n] = sum_k lhs[m,k] * rhs[n,k] in exact int32, then
// out[m,n] = T((f32)acc * lhs_scale[m] * rhs_scale[n]) with the products taken left to right.
//
// Replaces quantized_gemv_int8.cuh:13-51 (one 32-lane warp per row, __dp4a) and
// quantized_matmul_int8.cuh:112-269 (mma.m16n8k32.s8, 3-stage cp.async); CPU twin
// src/codegen/cpu/kernels/qgemv_i8i8.rs:38-80.
//   2 .. 32 rows (narrow matrices 128), K % 128 == 0, by qrows_first: v_mfma_i32_16x16x64_i8, a stream per wave (qrows.hip)
//   M < 3  : wave64 rows, 16 int8 per lane per load, v_dot4_i32_i8, integer butterfly (this file)
//   else   : v_mfma_i32_32x32x32_i8 with tiles of 32 .. 128 rows (tile_gemm.hip) or 256 (gemm.hip)
// Integer accumulation is associative, so both are bit-exact whatever the order.
#include "kernels.h"

namespace mynn {

// ---- small M: one wave per (R rows of rhs) x (MB rows of lhs)
template <typename T, int R, int MB>
__global__ __launch_bounds__(256) void qgemv_i8_kernel(T *out, int32_t *acc_out, const int8_t *lhs, const T *lhs_scale,
                                                       const int8_t *rhs, const T *rhs_scale, int m_base, int N, int K) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int row0 = (blockIdx.x * 4 + wave) * R;
    if (row0 >= N) return;
    int acc[R][MB];
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int m = 0; m < MB; m++) acc[r][m] = 0;
    const int nchunks = K >> 4;
    for (int c = lane; c < nchunks; c += 64) {
        U4 a[MB];
#pragma unroll
        for (int m = 0; m < MB; m++) a[m] = *((const U4 *)(lhs + (size_t)(m_base + m) * K) + c);
#pragma unroll
        for (int r = 0; r < R; r++) {
            const int row = row0 + r < N ? row0 + r : N - 1;
            const U4 w = __builtin_nontemporal_load((const U4 *)(rhs + (size_t)row * K) + c);
#pragma unroll
            for (int m = 0; m < MB; m++) {
                acc[r][m] = __builtin_amdgcn_sdot4((int)a[m].x, (int)w.x, acc[r][m], false);
                acc[r][m] = __builtin_amdgcn_sdot4((int)a[m].y, (int)w.y, acc[r][m], false);
                acc[r][m] = __builtin_amdgcn_sdot4((int)a[m].z, (int)w.z, acc[r][m], false);
                acc[r][m] = __builtin_amdgcn_sdot4((int)a[m].w, (int)w.w, acc[r][m], false);
            }
        }
    }
#pragma unroll
    for (int r = 0; r < R; r++)
#pragma unroll
        for (int m = 0; m < MB; m++) acc[r][m] = wave_sum_i32(acc[r][m]);
#pragma unroll
    for (int r = 0; r < R; r++) {
        if (lane == r && row0 + r < N) {
#pragma unroll
            for (int m = 0; m < MB; m++) {
                const size_t o = (size_t)(m_base + m) * N + row0 + r;
                if (acc_out) acc_out[o] = acc[r][m];
                if (out) {
                    const float asc = Elem<T>::ld(lhs_scale, m_base + m), wsc = Elem<T>::ld(rhs_scale, row0 + r);
                    Elem<T>::st(out, o, ((float)acc[r][m] * asc) * wsc);
                }
            }
        }
    }
}

template <typename T>
static int qmatmul_launch(void *out, int32_t *acc_out, const int8_t *lhs, const void *ls, const int8_t *rhs,
                          const void *rs, int M, int N, int K, hipStream_t s) {
    const int R = 2;
    const dim3 grid((N + 4 * R - 1) / (4 * R));
    int m = 0;
    while (m < M) {
        const int mb = M - m >= 4 ? 4 : (M - m >= 2 ? 2 : 1);
        if (mb == 4)
            MYNN_LAUNCH((qgemv_i8_kernel<T, R, 4>), grid, dim3(256), 0, s, (T *)out, acc_out, lhs, (const T *)ls, rhs,
                               (const T *)rs, m, N, K);
        else if (mb == 2)
            MYNN_LAUNCH((qgemv_i8_kernel<T, R, 2>), grid, dim3(256), 0, s, (T *)out, acc_out, lhs, (const T *)ls, rhs,
                               (const T *)rs, m, N, K);
        else
            MYNN_LAUNCH((qgemv_i8_kernel<T, R, 1>), grid, dim3(256), 0, s, (T *)out, acc_out, lhs, (const T *)ls, rhs,
                               (const T *)rs, m, N, K);
        int rc = launch_status("qgemv_i8_kernel");
        if (rc) return rc;
        m += mb;
    }
    return 0;
}

}  // namespace mynn

extern "C" int mynn_quantized_matmul(void *out, int32_t *acc_out, const int8_t *lhs, const void *lhs_scale,
                                     const int8_t *rhs, const void *rhs_scale, int M, int N, int K, int dtype,
                                     mynn_stream s) {
    using namespace mynn;
    MYNN_REQUIRE(lhs && rhs && (out || acc_out), MYNN_ERR_INVALID, "quantized_matmul: null operand");
    MYNN_REQUIRE(!out || (lhs_scale && rhs_scale), MYNN_ERR_INVALID, "quantized_matmul: scales are needed for the float output");
    MYNN_REQUIRE(M > 0 && N > 0 && K > 0, MYNN_ERR_INVALID, "quantized_matmul: M=%d N=%d K=%d", M, N, K);
    MYNN_REQUIRE(K % 32 == 0, MYNN_ERR_UNSUPPORTED, "quantized_matmul: K=%d is not a multiple of 32", K);
    MYNN_REQUIRE(aligned16(lhs) && aligned16(rhs), MYNN_ERR_INVALID, "quantized_matmul: operands must be 16-byte aligned");
    // int32 accumulators hold the exact sum as long as K * 128 * 128 < 2^31
    MYNN_REQUIRE(K <= 131071, MYNN_ERR_UNSUPPORTED, "quantized_matmul: K=%d could overflow the int32 accumulator", K);
    // rows by the streams of qrows.hip where K is whole steps of them and they are the faster form
    if (qrows_first(M, N, K)) return qrows_gemm(out, acc_out, lhs, lhs_scale, rhs, rhs_scale, M, N, K, dtype, as_stream(s));
    // else matrix cores from three rows on (two rows of 4096 x 4096: 6.2 us as dot products, 8.1 as tiles; three: 10 and 8),
    // with the 256-row tiles of gemm.hip where enough of them make that the faster one; the output may lie anywhere (their
    // store writes element by element where it is not 16-byte aligned)
    if (M >= 3) {
        const TgPlan plan = tile_gemm_plan(TG_I8, dtype, M, N, K, kTgScratchMax);
        if (dtype != MYNN_F32 && qgemm_dma_us(M, N, K) < plan.us)
            return qgemm_dma(out, acc_out, lhs, lhs_scale, rhs, rhs_scale, nullptr, M, N, K, dtype, GEMM_PLAIN, as_stream(s));
        // (captured, a product whose K ranges would be side by side takes them as one: the streams, which need no memory for the sums.  us
        // captured, tiles / so: 8 x 500 x 32768 41.6 / 8.1, 32 x 1024 x 32768 41.9 / 25.7, 40 x 2048 x 14336 20.6 / 12.9, 64 x 4096 x 14336 21.2 / 18.8)
        if (plan.ks > 1 && qrows_supported(M, N, K) && stream_capturing(as_stream(s)))
            return qrows_gemm(out, acc_out, lhs, lhs_scale, rhs, rhs_scale, M, N, K, dtype, as_stream(s));
        return tile_gemm_on_stream(TG_I8, plan, out, acc_out, lhs, rhs, lhs_scale, rhs_scale, M, N, K, dtype, as_stream(s));
    }
    return dispatch_dtype(dtype, [&](auto *t) {
        using T = std::remove_pointer_t<decltype(t)>;
        return qmatmul_launch<T>(out, acc_out, lhs, lhs_scale, rhs, rhs_scale, M, N, K, as_stream(s));
    });
}
