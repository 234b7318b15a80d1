// Streaming decode attention: the merge as a launch of its own, the plan of the key ranges and the entry (the kernel:
// attention_stream.h).
#include "attention_stream.h"

namespace mynn {

// (sequences x kv heads x keys) from which the operator takes this kernel instead of the latency kernel of
// attention_decode.hip.  Latency / streaming, us a call, 16-bit caches (profiles/attention_routes.md): from 8192 on this one is the
// faster at every shape measured (D = 64: 16 x 128 keys 7.2 / 5.2, 2 x 1024 13.0 / 6.7, 4 x 2048 20.5 / 8.3; D = 128: 1 x 1024 12.7 / 7.5,
// 4 x 256 9.2 / 6.1).  The line was drawn when 4096 went either way; with eight waves and one wait in the merge it does no longer
// (D = 64, 4 x 256 7.0 / 5.3; D = 128, 2 x 256 7.3 / 6.2, 1 x 512 10.5 / 7.3), and it could come down.  An executor's fused form, which
// saves the RoPE + append launch as well, takes this kernel for every batch of two and more whatever the length.
constexpr long kStreamMinKeys = 8192;

// ---- merge of key ranges: out[row, d] = sum_s o_s * exp(m_s - m) / sum_s l_s * exp(m_s - m).
// A launch of its own, for callers whose scratch memory has no arrival counters and for the per-slice kernel.
template <typename T>
__global__ __launch_bounds__(256) void attn_merge_kernel(AttnParams p, int D) {
    const size_t idx = (size_t)blockIdx.x * 256 + threadIdx.x;  // (b, head, sq, d)
    const size_t rows = (size_t)p.B * p.Hq * p.Sq;
    if (idx >= rows * D) return;
    const size_t row = idx / D;
    const int d = (int)(idx % D);
    const float *ml = p.part_ml + row * p.nsplit * 2;
    const float *po = p.part_o + row * p.nsplit * D;
    float mt = -INFINITY;
#pragma unroll 8
    for (int s = 0; s < p.nsplit; s++) mt = fmaxf(mt, ml[2 * s]);
    float lt = 0.f, ot = 0.f;
#pragma unroll 8
    for (int s = 0; s < p.nsplit; s++) {
        const float ms = ml[2 * s];
        const float c = (ms == -INFINITY) ? 0.f : fast_exp(ms - mt);
        lt = fmaf(ml[2 * s + 1], c, lt);
        ot = fmaf(po[s * D + d], c, ot);
    }
    const size_t sq = row % p.Sq, bh = row / p.Sq, h = bh % p.Hq, b = bh / p.Hq;
    Elem<T>::st((T *)p.out, b * p.o_bs + h * p.o_hs + sq * p.o_rs + d, ot / lt);
}

int attention_merge_launch(const AttnParams &p, int D, int dtype, hipStream_t s) {
    const size_t n = (size_t)p.B * p.Hq * p.Sq * D;
    return dispatch_dtype(dtype, [&](auto *t) {
        using T = std::remove_pointer_t<decltype(t)>;
        MYNN_LAUNCH(attn_merge_kernel<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, D);
        return launch_status("attn_merge_kernel");
    });
}

// ---- host side ---------------------------------------------------------------------------------
bool attn_stream_eligible(int B, int Sq, int Hq, int Hkv, int D, int dtype, int kv_int8, int kv_len, int cache_len) {
    const int G = Hq / Hkv;
    return Sq == 1 && dtype != MYNN_F32 && (!kv_int8 || cache_len % kStreamTile == 0) && (D == 64 || D == 128) &&
           (G == 1 || G == 2 || G == 4 || G == 8) && cache_len >= kStreamTile && (long)B * Hkv * kv_len >= kStreamMinKeys;
}

// key rows per workgroup and number of key ranges: ONE workgroup per CU (its four waves keep eight tiles in flight,
// which is enough to stream; measured over batch x kv-head counts of 8 .. 384 and contexts of 512 .. 8192, two to
// four workgroups per CU -- what the register count allows -- were 0-25 % slower: shorter sequential runs, more partial
// results to write and to merge, and with at least one (sequence, kv head) per CU the merge launch disappears
// altogether); ranges a multiple of the 128 keys a workgroup takes per step
static int stream_slots() {
    static int slots = 0;
    if (!slots) {
        int dev = 0, cus = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) {
            (void)hipGetLastError();
            cus = 256;
        }
        slots = cus;
    }
    return slots;
}
void attn_stream_plan(int B, int Hkv, int kv_len, int *slice, int *nsplit) {
    const int step = 4 * kStreamTile, pairs = B * Hkv;
    int n = stream_slots() / pairs;
    const int nmax = (kv_len + 127) / 128;
    if (n > nmax) n = nmax;
    if (n < 1) n = 1;
    int rows = ((kv_len + n - 1) / n + step - 1) / step * step;
    // Eight waves to a workgroup and ranges of twice the length where that leaves nothing to merge, or where four would make so
    // many ranges that their arrivals and the merge, beyond eight of them two waits for memory instead of one, are most of the launch:
    // more than 16, or more than 8 that fill most of the CUs.  Us of an operator call, four / eight waves, fp16, 32 query heads:
    //   nothing left to merge    D = 64: 16 x 250 keys 6.0 / 4.6, 32 x 200 5.9 / 4.5; D = 128: 8 x 250 7.1 / 6.2; but 8 x 500 6.1 / 6.8
    //   16 pairs of (sequence, kv head), by keys          1000        1100        1200        1400        1700        1900        2048
    //     D = 64, 4 kv heads                         7.0 / 7.4   7.7 / 7.4   8.1 / 7.4   8.4 / 7.5   8.6 / 7.6   8.8 / 7.8   9.1 / 7.9
    //     D = 128, 8 kv heads                        8.0 / 8.7   8.3 / 9.0   8.7 / 8.9   9.2 / 9.1   9.8 / 9.4  10.3 / 9.6  10.7 / 9.6
    //   8 pairs:  D = 64, 4 kv heads                             7.0 / 7.1   7.0 / 7.2   7.3 / 6.9   7.3 / 7.2   7.6 / 7.1   7.6 / 7.5
    //     D = 128, 8 kv heads                                    7.8 / 8.3   7.8 / 8.4   7.9 / 8.4   8.1 / 8.7   8.2 / 8.7   8.5 / 8.7
    //   more than 16 ranges      8 pairs x 3000: D = 64 9.5 / 8.2, D = 128 10.7 / 9.6; 4 pairs x 4000: 9.8 / 7.8, 14.6 / 10.6
    const int ranges = (kv_len + rows - 1) / rows;
    if (rows == step && (ranges == 2 || ranges > 16 || (ranges > 8 && pairs * ranges * 8 >= stream_slots() * 5))) rows = 2 * step;
    *slice = rows;
    *nsplit = (kv_len + rows - 1) / rows;
}
// The number of key ranges is not monotonic in the length (a longer cache can round to fewer, longer ranges), so a
// workspace is sized for the most ranges ANY length up to kv_len_max can be planned with.
int attn_stream_max_ranges(int B, int Hkv, int kv_len_max) {
    int n = stream_slots() / (B * Hkv);
    const int nmax = (kv_len_max + 127) / 128;
    if (n > nmax) n = nmax;
    return n < 1 ? 1 : n;
}
// Paged caches: the pages of a key range travel in one vector register, a lane each, so a range spans at most 62
// pages (one more at either end for ranges that start inside a page); longer ranges are cut into more of them.
static int paged_slice_cap(int page_shift) {
    const int step = 4 * kStreamTile;
    return ((62 << page_shift) / step) * step;
}
void attn_stream_plan_paged(int B, int Hkv, int kv_len, int page_shift, int *slice, int *nsplit) {
    attn_stream_plan(B, Hkv, kv_len, slice, nsplit);
    const int cap = paged_slice_cap(page_shift);
    if (*slice > cap) {
        *slice = cap;
        *nsplit = (kv_len + cap - 1) / cap;
    }
}
int attn_stream_max_ranges_paged(int B, int Hkv, int kv_len_max, int page_shift) {
    const int a = attn_stream_max_ranges(B, Hkv, kv_len_max), cap = paged_slice_cap(page_shift);
    const int b = (kv_len_max + cap - 1) / cap;
    return a > b ? a : b;
}
// the conditions of attn_stream_eligible that do not depend on the length of one call
bool attn_stream_possible(int B, int Sq, int Hq, int Hkv, int D, int dtype, int cache_len) {
    const int G = Hq / Hkv;
    return Sq == 1 && dtype != MYNN_F32 && (D == 64 || D == 128) && (G == 1 || G == 2 || G == 4 || G == 8) &&
           cache_len >= kStreamTile && (long)B * Hkv * cache_len >= kStreamMinKeys;
}

// what the paged form needs whatever the sizes: one query row, a 16-bit type, head_dim 64 or 128, 1/2/4/8 query heads
// per kv head, pages of a power of two >= 32 rows
bool attn_stream_paged_supported(int Sq, int Hq, int Hkv, int D, int dtype, int page_rows) {
    const int G = Hkv > 0 ? Hq / Hkv : 0;
    return Sq == 1 && (dtype == MYNN_F16 || dtype == MYNN_BF16) && (D == 64 || D == 128) && (G == 1 || G == 2 || G == 4 || G == 8) &&
           page_rows >= kStreamTile && (page_rows & (page_rows - 1)) == 0;
}

int attention_stream_launch(const AttnParams &p, int D, int dtype, int kv_int8, hipStream_t s) {
    MYNN_REQUIRE(!kv_int8 || (p.k_scale && p.v_scale && p.cache_len % kStreamTile == 0), MYNN_ERR_INVALID,
                 "streaming attention: int8 KV needs scales and a cache length that is a multiple of %d", kStreamTile);
    MYNN_REQUIRE(p.q_rs >= 0 && aligned16(p.qkv ? p.qkv : p.q) && aligned16(p.k) && aligned16(p.v) && p.q_bs % 8 == 0 && p.q_hs % 8 == 0,
                 MYNN_ERR_INVALID, "streaming attention: q, k, v must be 16-byte aligned");
    MYNN_REQUIRE(p.nsplit == 1 || (p.part_o && p.part_ml), MYNN_ERR_INVALID,
                 "streaming attention: no scratch for %d key ranges", p.nsplit);
    MYNN_REQUIRE(p.slice % (4 * kStreamTile) == 0 && p.nsplit <= 65535, MYNN_ERR_INVALID,
                 "streaming attention: slice %d, %d ranges", p.slice, p.nsplit);
    if (p.page_table) {
        MYNN_REQUIRE(attn_stream_paged_supported(p.Sq, p.Hq, p.Hkv, D, dtype, 1 << p.page_shift), MYNN_ERR_UNSUPPORTED,
                     "paged attention: one query row, 16-bit type, head_dim 64/128, 1/2/4/8 heads per kv head, pages of 2^n >= %d rows",
                     kStreamTile);
        MYNN_REQUIRE(p.cache_len == p.pages_per_seq << p.page_shift, MYNN_ERR_INVALID,
                     "paged attention: cache length %d is not %d pages of %d rows", p.cache_len, p.pages_per_seq, 1 << p.page_shift);
        // a key range's pages travel in one register, a lane each
        MYNN_REQUIRE((p.slice >> p.page_shift) + 2 <= 64, MYNN_ERR_UNSUPPORTED,
                     "paged attention: a key range of %d rows spans more than 62 pages of %d rows", p.slice, 1 << p.page_shift);
    }
    const bool fuse = p.qkv != nullptr;
    MYNN_REQUIRE(!fuse || (p.nsplit == 1 || p.arrive), MYNN_ERR_INVALID, "streaming attention: the fused form merges its own key ranges");
    const StreamParams sp{{p.out, p.k_scale, p.v_scale, p.cos_t, p.sin_t, p.page_table, p.part_o, p.part_ml,
                           p.nsplit > 1 && p.B * p.Hkv <= kAttnArrive ? p.arrive : nullptr, fuse ? (long)(p.Hq + 2 * p.Hkv) * D : p.q_bs,
                           fuse ? (long)D : p.q_hs, p.o_bs, p.o_hs, p.scale, p.Hq, p.cache_len, p.active, p.nsplit, p.page_shift, p.pages_per_seq},
                          fuse ? p.qkv : p.q, p.k, p.v, p.d_active, p.d_past, p.d_pos, p.Hkv, p.slice};
    const int rc = dtype == MYNN_F16 ? attn_stream_go<f16_t>(sp, p.B, D, kv_int8, fuse, s) : attn_stream_go<bf16_t>(sp, p.B, D, kv_int8, fuse, s);
    if (sp.arrive) return rc;
    if (rc || p.nsplit == 1) return rc;
    return attention_merge_launch(p, D, dtype, s);
}

}  // namespace mynn
