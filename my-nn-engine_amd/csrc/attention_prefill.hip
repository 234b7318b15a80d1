// Causal / full prefill attention on the matrix cores (flash-attention form), replacing the
// reference's attention_tc (attention.cuh:45-314: mma.m16n8k16, S and P round-tripping through
// shared memory, 16 lanes doing the softmax serially).
//
// One workgroup = QW x KW waves: QW blocks of 32 query rows of one (batch, query head), the key tiles dealt out over KW
// groups of QW waves whose results are merged at the end.  Many rows: 4 x 1, two workgroups per CU (two waves per SIMD, up
// to 256 registers a lane: at three the kernel spilled into scratch inside the key loop).  A tile is a serial chain (scores,
// maximum, exponentials, product) of some 2 us at D = 128, so where the rows do not fill the device the tiles of a row run
// side by side instead of after each other.  Workgroups are dispatched longest first: grid y = query block, last first.
// Per 64-key tile (staged once in LDS for the waves of a group, K row-major, V transposed; two 32-key S^T tiles):
//   S^T = K . Q^T      v_mfma_f32_32x32x16: A = K rows from LDS, B = Q kept in registers
//   softmax            each lane owns ONE query column and 16 of the 32 keys of each S^T tile, so the
//                      row max / sum are in-lane plus a single exchange with lane ^ 32
//   O^T += V^T . P^T   the D-layout of S^T is already the B-operand layout of P^T (keys are
//                      contracted in the permuted order 4g+0..3, 8+4g+0..3), so P never leaves
//                      registers; A = V^T read from LDS with two 8-byte reads
// The rescale factor of the online softmax is a per-lane scalar because O^T keeps the same query
// column per lane; the rescale is skipped when no lane of the wave moved its maximum (most tiles after the
// first few).  Key tiles past a wave's last causal position are skipped.
// rope_q: the queries are read un-rotated from the projection's output and rotated in registers (the RoPE launch
// then only has the keys and values left to do).
// A thread stages CH neighbouring keys of the same 8 dims, so V^T goes to LDS CH keys at a time (4- or 8-byte
// writes of values gathered with v_perm) instead of one 2-byte write per value.
#include <type_traits>

#include "attention.h"
#include "mfma.h"

namespace mynn {

constexpr int kPfKeys = 64;

template <int D, int QW, int KW> constexpr int pf_buffers() { return KW == 1 ? 2 : 1; }  // LDS tiles per group
template <int D, int QW, int KW> constexpr size_t pf_group_bytes() {
    return (size_t)pf_buffers<D, QW, KW>() * (kPfKeys * (D + 8) + D * (kPfKeys + 4)) * 2 + 2 * kPfKeys * sizeof(float);
}
template <int D, int QW, int KW> constexpr size_t pf_lds() {
    const size_t tiles = KW * pf_group_bytes<D, QW, KW>(), merge = (size_t)(KW - 1) * QW * 64 * (D / 2 + 2) * sizeof(float);
    return tiles > merge ? tiles : merge;
}

// PAGED: K/V rows are found through a page table (AttnParams::page_table) of at most 64 pages per sequence, each a
// power of two >= 64 rows: a 64-key tile lies in one page, and the sequence's table row sits in one register (lane i =
// page i) from which a tile picks its entry with v_readlane.
// KV8: an int8 cache with a scale per row.  The codes enter both products exactly; a key's scale multiplies its score, its
// value's scale its weight.  (fp16: in units of the largest scale so far, times 2^12, so that small weights stay normal
// numbers and none overflows; a larger scale rescales O^T as a larger maximum does, and the unit is put back at the end.)
// The weights enter as several values of T each, rounded and rest: the row-at-a-time kernel, which also takes these calls,
// keeps them in f32.  Two of fp16 (22 bits: as near to the result in 64 bits as f32 is), three of bf16: with two, 0.2 % of the
// outputs were not the nearest bf16 value where f32 weights leave 0.01 - 0.03 % (32 heads, 128 rows behind 500 keys: two values
// 22.3 us, three 23.5 at D = 128, 13.9 and 14.3 at D = 64; one prompt of 128 rows 9.2 and 9.4).
template <typename T, int D, bool PAGED, bool KV8, int QW, int KW>
__global__ __launch_bounds__(QW *KW * 64, 2) void attn_prefill_kernel(AttnParams p) {
    constexpr int kPfThreads = QW * 64, kPfRows = QW * 32;  // threads of a group, query rows of the workgroup
    constexpr int NBUF = pf_buffers<D, QW, KW>();
    constexpr bool UNITS = KV8 && std::is_same<T, f16_t>::value;
    constexpr int LDK = D + 8;          // K tile row stride (elements): conflict-free 16-byte reads
    constexpr int LDV = kPfKeys + 4;    // V^T tile row stride
    constexpr int KS = D / 16;          // k-steps of the S^T product
    constexpr int DT = D / 32;          // 32-row tiles of O^T
    constexpr int CH = (kPfKeys * D / 8) / kPfThreads;  // 16-byte chunks per thread and tile (2 or 4): neighbouring keys
    constexpr int NPF = D == 64 && KW == 1 ? 2 : 1;     // tiles in flight in registers ahead of the one in LDS
    static_assert(CH == 2 || CH % 4 == 0, "a thread stages 2 or a multiple of 4 neighbouring keys");
    extern __shared__ __align__(16) char lds[];
    const int kg = threadIdx.x / kPfThreads;  // key group
    uint16_t(*Ks)[kPfKeys * LDK] = (uint16_t(*)[kPfKeys * LDK])(lds + kg * pf_group_bytes<D, QW, KW>());
    uint16_t(*Vt)[D * LDV] = (uint16_t(*)[D * LDV])(Ks + NBUF);
    float *ksc = (float *)(Vt + NBUF), *vsc = ksc + kPfKeys;  // KV8 (one tile's: written and read between two barriers)
    static_assert(!KV8 || KW > 1, "one buffer of scales, units left before the merge");

    const int tid = threadIdx.x % kPfThreads, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 31, g = lane >> 5;
    const int bh = blockIdx.x, b = bh / p.Hq, h = bh % p.Hq;
    const int G = p.Hq / p.Hkv, hkv = h / G;
    const int Sq = p.Sq;
    const int active = p.d_active ? *p.d_active : p.active;
    const int qoff = p.d_active ? active - Sq : p.q_pos_offset;
    const int kv_bound = min(active, p.cache_len);

    const int q_blk = ((int)gridDim.y - 1 - (int)blockIdx.y) * kPfRows;  // the blocks with the most keys are dispatched first
    const int qrow = q_blk + wave * 32 + col;           // this lane's query row
    const int qrow_c = min(qrow, Sq - 1);
    // keys this lane's query may see, and the furthest any row of the wave / workgroup may see
    const int my_bound = p.is_causal ? min(kv_bound, qoff + qrow_c + 1) : kv_bound;
    const int wave_last = min(q_blk + wave * 32 + 31, Sq - 1);
    const int wave_bound = p.is_causal ? min(kv_bound, qoff + wave_last + 1) : kv_bound;
    const int blk_last = min(q_blk + kPfRows - 1, Sq - 1);
    const int blk_bound = p.is_causal ? min(kv_bound, qoff + blk_last + 1) : kv_bound;
    const int ntiles = (blk_bound + kPfKeys - 1) / kPfKeys;

    using TKV = std::conditional_t<KV8, int8_t, T>;
    using Chunk = std::conditional_t<KV8, uint2, U4>;  // 8 elements of a cached row
    const size_t kv_row0 = PAGED ? 0 : (size_t)(b * p.Hkv + hkv) * p.cache_len;
    const TKV *Kg = (const TKV *)p.k + kv_row0 * D, *Vg = (const TKV *)p.v + kv_row0 * D;
    const int psh = p.page_shift, pmask = (1 << psh) - 1;
    int pg_reg = 0;
    if constexpr (PAGED) {
        if (lane < p.pages_per_seq) pg_reg = p.page_table[(size_t)b * p.pages_per_seq + lane];
    }
    // a tile travels global -> registers (NPF iterations ahead of) -> LDS (one iteration ahead of) the MFMAs.
    // Thread t stages the keys CH * (t / (D/8)) + 0 .. CH-1 of a tile, dims 8 * (t % (D/8)) .. +7.
    // Rows past the end are clamped to the last visible key: whatever they hold is masked out.
    const int key0 = (tid / (D / 8)) * CH, dd = (tid % (D / 8)) * 8;
    Chunk rk[NPF][CH], rv[NPF][CH];
    T rs = T{};  // KV8: the scale of key tid % 64, of K (tid < 64) or V
    auto load_tile = [&](int t, Chunk *k_, Chunk *v_) {
        size_t po = 0;  // PAGED: first row of the tile's page, in rows of one head of the pool
        if constexpr (PAGED) {
            const int pg = __builtin_amdgcn_readlane(pg_reg, __builtin_amdgcn_readfirstlane((t * kPfKeys) >> psh));
            po = ((size_t)pg * p.Hkv + hkv) << psh;
        }
#pragma unroll
        for (int c = 0; c < CH; c++) {
            const int key = min(t * kPfKeys + key0 + c, blk_bound - 1);
            const size_t row = PAGED ? po + (size_t)(key & pmask) : (size_t)key;
            k_[c] = *(const Chunk *)(Kg + row * D + dd);
            v_[c] = *(const Chunk *)(Vg + row * D + dd);
        }
        if constexpr (KV8) {
            if (tid < 128) rs = ((const T *)(tid < 64 ? p.k_scale : p.v_scale))[kv_row0 + min(t * kPfKeys + (tid & 63), blk_bound - 1)];
        }
    };
    auto operand = [](const Chunk &c) -> U4 {
        if constexpr (KV8) return i8x8_to_operand<T>(c.x, c.y);
        else return c;
    };
    auto store_tile = [&](int buf, const Chunk *k_, const Chunk *v8) {
        U4 v_[CH];
#pragma unroll
        for (int c = 0; c < CH; c++) v_[c] = operand(v8[c]);
        if constexpr (KV8) {
            if (tid < 128) ksc[tid] = Elem<T>::ld(&rs, 0);
        }
#pragma unroll
        for (int c = 0; c < CH; c++) *(U4 *)&Ks[buf][(key0 + c) * LDK + dd] = operand(k_[c]);
        // V^T[d][key0 .. key0 + CH - 1] for the 8 dims: dword i of a chunk holds dims 2i (low half) and 2i + 1
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t w[CH];
#pragma unroll
            for (int c = 0; c < CH; c++) w[c] = i == 0 ? v_[c].x : i == 1 ? v_[c].y : i == 2 ? v_[c].z : v_[c].w;
            uint16_t *lo = &Vt[buf][(dd + 2 * i) * LDV + key0], *hi = &Vt[buf][(dd + 2 * i + 1) * LDV + key0];
            if constexpr (CH == 2) {
                *(uint32_t *)lo = __builtin_amdgcn_perm(w[1], w[0], 0x05040100u);
                *(uint32_t *)hi = __builtin_amdgcn_perm(w[1], w[0], 0x07060302u);
            } else {
#pragma unroll
                for (int c = 0; c < CH; c += 4) {
                    *(uint2 *)(lo + c) = uint2{__builtin_amdgcn_perm(w[c + 1], w[c], 0x05040100u), __builtin_amdgcn_perm(w[c + 3], w[c + 2], 0x05040100u)};
                    *(uint2 *)(hi + c) = uint2{__builtin_amdgcn_perm(w[c + 1], w[c], 0x07060302u), __builtin_amdgcn_perm(w[c + 3], w[c + 2], 0x07060302u)};
                }
            }
        }
    };

    // the first tile's loads are on their way before the queries (and their RoPE table rows) are asked for
    if (kg < ntiles) load_tile(kg, rk[0], rv[0]);
    // Q^T fragments: B operand, lane (query col, g): d = 16*ks + 8*g .. +7
    const T *Q = (const T *)p.q + (size_t)b * p.q_bs + (size_t)h * p.q_hs + (size_t)qrow_c * p.q_rs;
    U4 qf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) qf[ks] = *(const U4 *)(Q + 16 * ks + 8 * g);
    if (p.rope_q) {
        // the query rows arrive un-rotated (straight from the projection): RoPE by the row's position, the arithmetic of
        // rope.cuh:18-46 -- lo' = lo*cos[j] - hi*sin[j], hi' = hi*cos[j + D/2] + lo*sin[j + D/2], separate products, one
        // rounding.  Dims d and d + D/2 sit in fragments ks and ks + KS/2 of the same lane.
        const size_t tab = (size_t)p.d_pos[qrow_c] * D;
        const T *cs = (const T *)p.cos_t + tab, *sn = (const T *)p.sin_t + tab;
#pragma unroll
        for (int ks = 0; ks < KS / 2; ks++) {
            const int d0 = 16 * ks + 8 * g;
            float xl[8], xh[8], cl[8], ch[8], sl[8], sh[8], ol[8], oh[8];
            widen8<T>(qf[ks], xl);
            widen8<T>(qf[ks + KS / 2], xh);
            widen8<T>(*(const U4 *)(cs + d0), cl);
            widen8<T>(*(const U4 *)(cs + d0 + D / 2), ch);
            widen8<T>(*(const U4 *)(sn + d0), sl);
            widen8<T>(*(const U4 *)(sn + d0 + D / 2), sh);
#pragma unroll
            for (int i = 0; i < 8; i++) {
                ol[i] = xl[i] * cl[i] - xh[i] * sl[i];
                oh[i] = xh[i] * ch[i] + xl[i] * sh[i];
            }
            qf[ks] = U4{pack2<T>(ol[0], ol[1]), pack2<T>(ol[2], ol[3]), pack2<T>(ol[4], ol[5]), pack2<T>(ol[6], ol[7])};
            qf[ks + KS / 2] = U4{pack2<T>(oh[0], oh[1]), pack2<T>(oh[2], oh[3]), pack2<T>(oh[4], oh[5]), pack2<T>(oh[6], oh[7])};
        }
    }

    f16x_t o[DT];
#pragma unroll
    for (int t = 0; t < DT; t++)
#pragma unroll
        for (int e = 0; e < 16; e++) o[t][e] = 0.f;
    // running max in units of log2: scores are turned into exponents of two with one FMA each,
    // p = 2^(s * scale * log2(e) - m); the softmax scale is positive, so the max may be taken on raw scores
    float m = -INFINITY, l = 0.f;
    float unit = 0x1p-60f;  // UNITS: O^T is kept divided by it, a power of two
    const float scale2 = p.scale * 1.4426950408889634f;
    // keys every query row of this wave may see: tiles that end at or below it need no masking
    const int wave_first = min(q_blk + wave * 32, Sq - 1);
    const int wave_all = p.is_causal ? min(kv_bound, qoff + wave_first + 1) : kv_bound;

    // one tile of 64 keys = two S^T tiles (rows = keys, cols = queries), one softmax update, 4 k-steps of P.V
    auto tile = [&](int buf, int k0, auto masked) {
        constexpr bool MASKED = decltype(masked)::value;
        f16x_t s[2];
#pragma unroll
        for (int hf = 0; hf < 2; hf++)
#pragma unroll
            for (int e = 0; e < 16; e++) s[hf][e] = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
            for (int hf = 0; hf < 2; hf++) {
                const U4 a = *(const U4 *)&Ks[buf][(32 * hf + col) * LDK + 16 * ks + 8 * g];
                s[hf] = Mfma<T>::run(a, qf[ks], s[hf]);
            }
        if constexpr (KV8) {
#pragma unroll
            for (int hf = 0; hf < 2; hf++)
#pragma unroll
                for (int e4 = 0; e4 < 4; e4++) {
                    const float4 f = *(const float4 *)&ksc[32 * hf + 8 * e4 + 4 * g];
                    s[hf][4 * e4] *= f.x; s[hf][4 * e4 + 1] *= f.y; s[hf][4 * e4 + 2] *= f.z; s[hf][4 * e4 + 3] *= f.w;
                }
        }
        // ---- online softmax for this lane's query over its 32 keys (+ partner lane's 32)
        float mloc = -INFINITY;
#pragma unroll
        for (int hf = 0; hf < 2; hf++)
#pragma unroll
            for (int e = 0; e < 16; e++) {
                if (MASKED) {
                    const int key = k0 + 32 * hf + 8 * (e >> 2) + 4 * g + (e & 3);
                    if (key >= my_bound) s[hf][e] = -INFINITY;
                }
                mloc = fmaxf(mloc, s[hf][e]);
            }
        mloc = fmaxf(mloc, __shfl_xor(mloc, 32, 64));  // (the row swap instruction measured slower here)
        const float mn = fmaxf(m, mloc * scale2);
        float corr = 1.f;
        if (MASKED && mn == -INFINITY) {
#pragma unroll
            for (int hf = 0; hf < 2; hf++)
#pragma unroll
                for (int e = 0; e < 16; e++) s[hf][e] = 0.f;
        } else {
            corr = __builtin_amdgcn_exp2f(m - mn);
            float ls = 0.f;
#pragma unroll
            for (int hf = 0; hf < 2; hf++)
#pragma unroll
                for (int e = 0; e < 16; e++) {
                    s[hf][e] = __builtin_amdgcn_exp2f(fmaf(s[hf][e], scale2, -mn));
                    ls += s[hf][e];
                }
            l = fmaf(l, corr, ls);
            m = mn;
        }
        float4 vs[KV8 ? 8 : 1];
        float to_unit = 1.f;
        if constexpr (KV8) {
#pragma unroll
            for (int i = 0; i < 8; i++) vs[i] = *(const float4 *)&vsc[32 * (i >> 2) + 8 * (i & 3) + 4 * g];
        }
        if constexpr (UNITS) {
            float vm = 0.f;
#pragma unroll
            for (int i = 0; i < 8; i++) vm = fmaxf(fmaxf(fmaxf(vm, fabsf(vs[i].x)), fmaxf(fabsf(vs[i].y), fabsf(vs[i].z))), fabsf(vs[i].w));
            vm = fmaxf(vm, __shfl_xor(vm, 32, 64));
            const float un = fmaxf(unit, __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, vm) & 0x7F800000u));
            corr *= unit * __builtin_amdgcn_rcpf(un);  // (of a power of two: exact)
            unit = un;
            to_unit = 4096.f * __builtin_amdgcn_rcpf(un);
        }
        // (a factor of exactly 1 in every lane leaves O^T as it is: the multiplications are skipped)
        if (__builtin_amdgcn_ballot_w64(corr != 1.f) != 0) {
#pragma unroll
            for (int t2 = 0; t2 < DT; t2++)
#pragma unroll
                for (int e = 0; e < 16; e++) o[t2][e] *= corr;
        }
        if constexpr (KV8) {
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float f[4] = {vs[i].x, vs[i].y, vs[i].z, vs[i].w};
#pragma unroll
                for (int e = 0; e < 4; e++) s[i >> 2][4 * (i & 3) + e] *= f[e] * to_unit;
            }
        }
        // ---- O^T += V^T . P^T, keys contracted in the order the D-layout delivers them
#pragma unroll
        for (int st = 0; st < 4; st++) {
            const f16x_t &ph = s[st >> 1];
            const int e0 = 8 * (st & 1);
            constexpr int PARTS = KV8 ? kParts<T> : 1;
            U4 pf[PARTS];
            if constexpr (KV8) {
                float w[8];
#pragma unroll
                for (int e = 0; e < 8; e++) w[e] = ph[e0 + e];
#pragma unroll
                for (int part = 0; part < PARTS; part++) {
                    pf[part].x = take_part<T>(w[0], w[1]);
                    pf[part].y = take_part<T>(w[2], w[3]);
                    pf[part].z = take_part<T>(w[4], w[5]);
                    pf[part].w = take_part<T>(w[6], w[7]);
                }
            } else
                pf[0] = U4{pack2<T>(ph[e0 + 0], ph[e0 + 1]), pack2<T>(ph[e0 + 2], ph[e0 + 3]),
                           pack2<T>(ph[e0 + 4], ph[e0 + 5]), pack2<T>(ph[e0 + 6], ph[e0 + 7])};
#pragma unroll
            for (int t2 = 0; t2 < DT; t2++) {
                const uint16_t *vr = &Vt[buf][(32 * t2 + col) * LDV + 16 * st + 4 * g];
                const uint2 lo = *(const uint2 *)vr, hi = *(const uint2 *)(vr + 8);
#pragma unroll
                for (int part = 0; part < PARTS; part++) o[t2] = Mfma<T>::run(U4{lo.x, lo.y, hi.x, hi.y}, pf[part], o[t2]);
            }
        }
    };
    auto compute = [&](int t, int buf) {
        const int k0 = t * kPfKeys;
        if (k0 + kPfKeys <= wave_all) tile(buf, k0, std::false_type{});
        else if (k0 < wave_bound) tile(buf, k0, std::true_type{});
    };

    // O^T in plain values again
    auto leave_unit = [&]() {
        if constexpr (UNITS) {
            unit *= 1.f / 4096.f;
#pragma unroll
            for (int t2 = 0; t2 < DT; t2++)
#pragma unroll
                for (int e = 0; e < 16; e++) o[t2][e] *= unit;
        }
    };

    if constexpr (KW == 1) {
        // tile 0 goes straight to LDS; tiles 1 .. NPF wait in registers (slot j holds tile 1 + j, then 1 + j + NPF, ..)
        if (ntiles > 0) {
            store_tile(0, rk[0], rv[0]);
#pragma unroll
            for (int j = 0; j < NPF; j++) load_tile(min(1 + j, ntiles - 1), rk[j], rv[j]);
        }
        __syncthreads();
        int t = 0;
        // groups of NPF iterations that all still issue a load (unconditional, so the waits on older loads can be counted)
        for (; t + 2 * NPF < ntiles; t += NPF) {
#pragma unroll
            for (int j = 0; j < NPF; j++) {
                store_tile((t + j + 1) & 1, rk[j], rv[j]);  // tile t + j + 1, loaded NPF iterations ago; its buffer was released by the last barrier
                load_tile(t + j + 1 + NPF, rk[j], rv[j]);   // (< ntiles by the loop bound)
                compute(t + j, (t + j) & 1);
                __syncthreads();
            }
        }
        // the rest: every tile still missing from LDS is in registers already or on its way
        for (; t < ntiles; t += NPF) {
#pragma unroll
            for (int j = 0; j < NPF; j++) {
                if (t + j < ntiles) {
                    if (t + j + 1 < ntiles) store_tile((t + j + 1) & 1, rk[j], rv[j]);
                    if (t + j + 1 + NPF < ntiles) load_tile(t + j + 1 + NPF, rk[j], rv[j]);
                    compute(t + j, (t + j) & 1);
                    __syncthreads();
                }
            }
        }
    } else {
        // group kg takes tiles kg, kg + KW, ..: one LDS tile per group, the next one in registers meanwhile
        for (int t = kg; t - kg < ntiles; t += KW) {  // (the same number of rounds for every group)
            if (t < ntiles) store_tile(0, rk[0], rv[0]);
            __syncthreads();
            if (t + KW < ntiles) load_tile(t + KW, rk[0], rv[0]);
            if (t < ntiles) compute(t, 0);
            __syncthreads();
        }
        leave_unit();
        // the groups' results meet in group 0, in their order: (m, l, O^T) of a lane, [word][lane] per wave
        constexpr int WORDS = D / 2 + 2;
        float *mine = (float *)lds + (size_t)((kg - 1) * QW + wave) * 64 * WORDS + lane;
        if (kg > 0) {
            mine[0] = m;
            mine[64] = l;
#pragma unroll
            for (int t2 = 0; t2 < DT; t2++)
#pragma unroll
                for (int e = 0; e < 16; e++) mine[(2 + t2 * 16 + e) * 64] = o[t2][e];
        }
        __syncthreads();
        if (kg > 0) return;
#pragma unroll
        for (int k = 1; k < KW; k++) {
            const float *from = (const float *)lds + (size_t)((k - 1) * QW + wave) * 64 * WORDS + lane;
            const float mo = from[0], mn = fmaxf(m, mo);
            const float ca = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mn), cb = mo == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mo - mn);
            l = l * ca + from[64] * cb;
            m = mn;
#pragma unroll
            for (int t2 = 0; t2 < DT; t2++)
#pragma unroll
                for (int e = 0; e < 16; e++) o[t2][e] = o[t2][e] * ca + from[(2 + t2 * 16 + e) * 64] * cb;
        }
    }

    // ---- out[query, d] = O^T[d, query] / l
    l += __shfl_xor(l, 32, 64);
    if (qrow < Sq) {
        T *out = (T *)p.out + (size_t)b * p.o_bs + (size_t)h * p.o_hs + (size_t)qrow * p.o_rs;
        const float inv = 1.0f / l;
#pragma unroll
        for (int t2 = 0; t2 < DT; t2++)
#pragma unroll
            for (int e4 = 0; e4 < 4; e4++) {
                const int d = 32 * t2 + 8 * e4 + 4 * g;
                uint2 w;
                w.x = pack2<T>(o[t2][4 * e4 + 0] * inv, o[t2][4 * e4 + 1] * inv);
                w.y = pack2<T>(o[t2][4 * e4 + 2] * inv, o[t2][4 * e4 + 3] * inv);
                *(uint2 *)(out + d) = w;
            }
    }
}

bool attention_prefill_supported(const AttnParams &p, int D, int dtype, int kv_int8) {
    if (dtype != MYNN_F16 && dtype != MYNN_BF16) return false;
    if (D != 64 && D != 128) return false;
    if (p.Sq < 16) return false;  // a handful of rows: the per-row kernel wastes less
    if (kv_int8) {
        // The conversion of a tile makes the chain longer, 8 us for one tile at D = 128, so the per-row kernel goes further:
        // as long as all rows together are few, fewer with many keys where the caller says how many (32 heads, D = 128, us,
        // per row / here: 64 rows 6.5 / 8.9, 96 rows 10.4 / 9.0, 4 x 24 rows 7.0 / 8.2, 4 x 32 rows 8.3 / 8.4, 4 x 64 rows
        // 17.5 / 9.3; behind 500 keys 32 rows 28 / 22, 64 rows 42 / 23, 128 rows 76 / 23).
        const long rows = (long)p.B * p.Hq * p.Sq;
        if (rows <= 3072 && !(rows >= 1536 && !p.d_active && p.active >= 256)) return false;
    }
    if (!(p.scale > 0.f)) return false;  // the running max is taken on unscaled scores
    // 16-byte loads of Q rows and 8-byte stores of out rows
    if ((p.q_rs % 8) || (p.q_hs % 8) || (p.q_bs % 8) || (p.o_rs % 4) || (p.o_hs % 4) || (p.o_bs % 4)) return false;
    if (((uintptr_t)p.q & 15) || ((uintptr_t)p.out & 7) || ((uintptr_t)p.k & 15) || ((uintptr_t)p.v & 15)) return false;
    return true;
}

template <typename T, int D, bool PAGED, bool KV8, int QW, int KW> static int pf_go(const AttnParams &p, hipStream_t s) {
    static bool lds_set = false;
    constexpr size_t lds = pf_lds<D, QW, KW>();
    if (!lds_set && lds > 64 * 1024) {
        MYNN_HIP(hipFuncSetAttribute((const void *)attn_prefill_kernel<T, D, PAGED, KV8, QW, KW>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        lds_set = true;
    }
    MYNN_LAUNCH((attn_prefill_kernel<T, D, PAGED, KV8, QW, KW>), dim3(p.B * p.Hq, (p.Sq + QW * 32 - 1) / (QW * 32)), dim3(QW * KW * 64), lds, s, p);
    return launch_status("attn_prefill_kernel");
}
// Which split, by the workgroups that 128 rows each would make (32 heads, causal; microseconds at 4 x 1 / 2 x 2 / 4 x 2):
// D = 64:  128 rows 6.6 / 5.3 / 6.5, 500: 12.6 / 9.4 / 11.4, 777: 16.9 / 13.4 / 15.2, 1200: 23.6 / 18.5 / 20.5, 2 x 936: 20.7 / 22.8
// D = 128: 128 rows 9.6 / 8.8 / 9.6, 500: 20.9 / 17.5 / 18.8, 777: 29.4 / 27.1 / 26.0, 1200: 43 / 38 / 36, 2048: 76 / 82 / 65,
// 2 x 936: 40.7 / 49.0 / 42.4.  Up to 64 rows there is one tile and nothing to split.
template <typename T, int D, bool PAGED, bool KV8> static int pf_pick(const AttnParams &p, hipStream_t s) {
    if constexpr (KV8) return pf_go<T, D, PAGED, KV8, 2, 2>(p, s);
    else {
        const long wgs = (long)p.B * p.Hq * ((p.Sq + 127) / 128);
        if constexpr (D == 64) {
            if (p.Sq > kPfKeys && wgs <= 320) return pf_go<T, D, PAGED, KV8, 2, 2>(p, s);
        } else {
            if (p.Sq > kPfKeys && wgs <= 128) return pf_go<T, D, PAGED, KV8, 2, 2>(p, s);
            if (p.Sq > kPfKeys && (wgs <= 320 || (wgs <= 512 && p.Sq >= 2000))) return pf_go<T, D, PAGED, KV8, 4, 2>(p, s);
        }
        return pf_go<T, D, PAGED, KV8, 4, 1>(p, s);
    }
}

int attention_prefill_launch(const AttnParams &p, int D, int dtype, int kv_int8, hipStream_t s) {
    MYNN_REQUIRE((p.Sq + 31) / 32 <= 65535, MYNN_ERR_UNSUPPORTED, "attention: Sq = %d exceeds the grid", p.Sq);
    if (p.page_table) {
        const int P = 1 << p.page_shift;
        MYNN_REQUIRE(!kv_int8 && P >= kPfKeys && p.pages_per_seq <= 64 && p.cache_len == p.pages_per_seq << p.page_shift, MYNN_ERR_UNSUPPORTED,
                     "paged prefill attention: %d pages of %d rows per sequence (at most 64 pages of 2^n >= %d rows, 16-bit)",
                     p.pages_per_seq, P, kPfKeys);
    }
    return dispatch_dtype16(dtype, [&](auto *t) {
        using T = std::remove_pointer_t<decltype(t)>;
        if (p.page_table) return D == 64 ? pf_pick<T, 64, true, false>(p, s) : pf_pick<T, 128, true, false>(p, s);
        if (kv_int8) return D == 64 ? pf_pick<T, 64, false, true>(p, s) : pf_pick<T, 128, false, true>(p, s);
        return D == 64 ? pf_pick<T, 64, false, false>(p, s) : pf_pick<T, 128, false, false>(p, s);
    });
}

}  // namespace mynn
