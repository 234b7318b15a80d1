// Causal / full prefill attention on the matrix cores (flash-attention form), replacing the
// reference's attention_tc (attention.cuh:45-314: mma.m16n8k16, S and P round-tripping through
// shared memory, 16 lanes doing the softmax serially).
//
// One workgroup = QW x KW waves: QW blocks of 32 query rows of one (batch, query head), the key tiles dealt out over KW
// groups of QW waves whose results are merged at the end.  Many rows: 4 x 1, two or three workgroups per CU.  A tile is a serial
// chain (scores, maximum, exponentials, product), so where the rows do not fill the device the tiles of a row run side by side
// instead of after each other.  Workgroups are dispatched longest first: grid y = query block, last first.
// Per tile of 64 or 32 keys (32-key S^T tiles):
//   S^T = K . Q^T      v_mfma_f32_32x32x16: A = K rows from LDS, B = Q kept in registers
//   softmax            each lane owns ONE query column and 16 of the 32 keys of each S^T tile, so the
//                      row max / sum are in-lane plus a single exchange with lane ^ 32
//   O^T += V^T . P^T   the D-layout of S^T is already the B-operand layout of P^T (keys are
//                      contracted in the permuted order 4g+0..3, 8+4g+0..3), so P never leaves
//                      registers; A = V^T read from the row-major V tile with two transposing 8-byte reads
// K and V go global -> LDS as they lie in memory (global_load_lds, two stages, one barrier per tile; chunks of a row placed so that
// both kinds of read fall into different banks: SQ_LDS_BANK_CONFLICT reads 0).  Through registers, with V^T written to LDS as such
// and two barriers per tile, the same launches took (bf16, us) D = 64: 1 x 777 14.1, 2 x 936 21.4, 8 x 1024 70, 4 x 2048 116;
// D = 128: 1 x 500 18.6, 1 x 777 26.0, 2 x 936 39, 8 x 1024 140.  Now (table at pf_pick) D = 64 keeps the vector units 74 % busy
// (8 x 1024: a quarter-rate exponential, an FMA, an addition, half a maximum and half a conversion per score and the rescaling of
// O^T), the matrix cores 35 %; D = 128 has two waves per SIMD and waits on the chain (vector 45 %, matrix 35 %).  Making the
// scores of the next tile between the exponentials of this one was 2 - 8 % slower (32 more registers, copies), wave priorities
// around the products 0 - 6 %.
// The rescale factor of the online softmax is a per-lane scalar because O^T keeps the same query
// column per lane; the rescale is skipped when no lane of the wave moved its maximum.  Rounds of tiles that every row sees in
// full run without masking, the last ones with; tiles past a wave's last causal position are skipped.
// rope_q: the queries are read un-rotated from the projection's output and rotated in registers (the RoPE launch
// then only has the keys and values left to do).
// PAGED: K/V rows are found through a page table (AttnParams::page_table) of at most 64 pages per sequence, each a
// power of two >= 64 rows: a tile lies in one page, and the sequence's table row sits in one register (lane i =
// page i) from which a tile picks its entry with v_readlane.
#include <type_traits>

#include "attention.h"
#include "mfma.h"

namespace mynn {

constexpr int kPfPage = 64;  // fewest rows of a page: a tile lies in one

// Rotates a query row in registers: RoPE by the row's position, the arithmetic of rope.cuh:18-46 -- lo' = lo*cos[j] - hi*sin[j],
// hi' = hi*cos[j + D/2] + lo*sin[j + D/2], separate products, one rounding.  Dims d and d + D/2 sit in fragments ks and
// ks + KS/2 of the same lane.
template <typename T, int D> __device__ __forceinline__ void pf_rotate(const AttnParams &p, int row, int g, U4 *qf) {
    constexpr int KS = D / 16;
    const size_t tab = (size_t)p.d_pos[row] * D;
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

// Which rows of the problem a workgroup has, and which keys they may see.
struct PfRows {
    int b, h, hkv, Sq, q_blk, qoff, kv_bound, blk_bound;
    __device__ __forceinline__ PfRows(const AttnParams &p, int rows) {
        const int bh = blockIdx.x;
        b = bh / p.Hq;
        h = bh % p.Hq;
        hkv = h / (p.Hq / p.Hkv);
        Sq = p.Sq;
        const int active = p.d_active ? *p.d_active : p.active;
        qoff = p.d_active ? active - Sq : p.q_pos_offset;
        kv_bound = min(active, p.cache_len);
        q_blk = ((int)gridDim.y - 1 - (int)blockIdx.y) * rows;  // the blocks with the most keys are dispatched first
        blk_bound = bound(p, min(q_blk + rows - 1, Sq - 1));
    }
    // keys that query row `row` may see
    __device__ __forceinline__ int bound(const AttnParams &p, int row) const { return p.is_causal ? min(kv_bound, qoff + row + 1) : kv_bound; }
};

template <int D, int KEYS, int QW, int KW> struct PfTile {
    static constexpr int ROWB = D * 2, TILEB = KEYS * ROWB, STAGE = 2 * TILEB, GROUP = 2 * STAGE;  // bytes: row, K or V tile, both, two stages
    static constexpr int THREADS = QW * KW * 64, ROWS = QW * 32;
    static constexpr int LOADS = TILEB / 1024 / QW;  // 1 KB loads per wave, of K and of V
    static constexpr int WORDS = D / 2 + 2;          // of a lane's result: maximum, sum, O^T
    static constexpr int MERGE = KW > 1 ? QW * KW * 64 * WORDS * 4 : 0;
    static constexpr int LDS = KW * GROUP > MERGE ? KW * GROUP : MERGE;
    static_assert(TILEB % (1024 * QW) == 0, "whole loads per wave");
    static_assert(KW == 1 || (D / 2 / KW) % 4 == 0, "a wave stores whole groups of four dims");
};

template <typename T, int D, bool PAGED, int KEYS, int QW, int KW>
__global__ __launch_bounds__(QW *KW * 64, 2) void attn_prefill_kernel(AttnParams p) {
    using G = PfTile<D, KEYS, QW, KW>;
    constexpr int KS = D / 16, DT = D / 32, NH = KEYS / 32;  // k-steps of S^T, 32-dim tiles of O^T, 32-key tiles of S^T
    constexpr int CPR = D / 8;                               // 16-byte chunks of a row
    extern __shared__ __align__(16) char lds[];
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wave = w % QW, kg = w / QW;  // block of 32 rows, key group
    const int col = lane & 31, g = lane >> 5;
    const PfRows R(p, G::ROWS);
    const int qrow = R.q_blk + wave * 32 + col, qrow_c = min(qrow, R.Sq - 1);  // this lane's query row
    const int my_bound = R.bound(p, qrow_c);
    const int wave_bound = R.bound(p, min(R.q_blk + wave * 32 + 31, R.Sq - 1));
    const int ntiles = (R.blk_bound + KEYS - 1) / KEYS;

    const size_t kv_row0 = PAGED ? 0 : (size_t)(R.b * p.Hkv + R.hkv) * p.cache_len;
    const char *Kg = (const char *)p.k + kv_row0 * G::ROWB, *Vg = (const char *)p.v + kv_row0 * G::ROWB;
    int pg_reg = 0;
    if constexpr (PAGED) {
        if (lane < p.pages_per_seq) pg_reg = p.page_table[(size_t)R.b * p.pages_per_seq + lane];
    }
    // this lane's chunks of a tile: LDS position P = (LOADS * wave + i) * 64 + lane, row P / CPR
    auto k_swz = [](int r) { return D == 128 ? r & 15 : (r >> 1) & 7; };
    auto v_swz = [](int r) { return D == 128 ? (r & 3) << 2 : (((r >> 1) ^ r) & 1) << 2; };
    uint32_t koff[G::LOADS], voff[G::LOADS];
    auto offsets = [&](int last) {  // rows past `last` repeat it: whatever they hold is masked out
#pragma unroll
        for (int i = 0; i < G::LOADS; i++) {
            const int P = (G::LOADS * wave + i) * 64 + lane, r = P / CPR, c = P % CPR;
            const uint32_t row = (uint32_t)min(r, last) * G::ROWB;
            koff[i] = row + ((c ^ k_swz(r)) << 4);
            voff[i] = row + ((c ^ v_swz(r)) << 4);
        }
    };
    offsets(KEYS - 1);
    char *grp = lds + kg * G::GROUP;
    auto issue = [&](int t, int stage) {
        size_t first = (size_t)t * KEYS;
        if constexpr (PAGED) {
            const int psh = p.page_shift;
            const int pg = __builtin_amdgcn_readlane(pg_reg, __builtin_amdgcn_readfirstlane((t * KEYS) >> psh));
            first = (((size_t)pg * p.Hkv + R.hkv) << psh) + ((t * KEYS) & ((1 << psh) - 1));
        }
        if ((t + 1) * KEYS > R.blk_bound) offsets(R.blk_bound - 1 - t * KEYS);  // (the last tile of the group)
        const char *kt = Kg + first * G::ROWB, *vt = Vg + first * G::ROWB;
        const uint32_t dst = lds_offset(grp + stage * G::STAGE + G::LOADS * wave * 1024);
#pragma unroll
        for (int i = 0; i < G::LOADS; i++) load_to_lds(kt, koff[i], dst + i * 1024);
#pragma unroll
        for (int i = 0; i < G::LOADS; i++) load_to_lds(vt, voff[i], dst + G::TILEB + i * 1024);
    };
    // the first tile's loads are on their way before the queries (and their RoPE table rows) are asked for
    if (kg < ntiles) issue(kg, 0);
    // Q^T fragments: B operand, lane (query col, g): d = 16*ks + 8*g .. +7
    const T *Q = (const T *)p.q + (size_t)R.b * p.q_bs + (size_t)R.h * p.q_hs + (size_t)qrow_c * p.q_rs;
    U4 qf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) qf[ks] = *(const U4 *)(Q + 16 * ks + 8 * g);
    if (p.rope_q) pf_rotate<T, D>(p, qrow_c, g, qf);

    f16x_t o[DT];
#pragma unroll
    for (int t = 0; t < DT; t++)
#pragma unroll
        for (int e = 0; e < 16; e++) o[t][e] = 0.f;
    // running reference in units of log2: scores are turned into exponents of two with one FMA each,
    // p = 2^(s * scale * log2(e) - m); the softmax scale is positive, so the max may be taken on raw scores
    float m = -INFINITY, l = 0.f;
    const float scale2 = p.scale * 1.4426950408889634f;

    const int krow = col * G::ROWB + ((g ^ k_swz(col)) << 4);
    int vrow[DT];
    {
        const int i = lane & 15, r = 4 * g + (i >> 2);
#pragma unroll
        for (int t2 = 0; t2 < DT; t2++)
            vrow[t2] = r * G::ROWB + (((4 * t2 + 2 * ((lane >> 4) & 1) + ((i & 3) >> 1)) ^ v_swz(r)) << 4) + 8 * (i & 1);
    }
    auto tile = [&](const char *kt, int k0, auto masked) {
        constexpr bool MASKED = decltype(masked)::value;
        const char *vt = kt + G::TILEB;
        f16x_t s[NH];
#pragma unroll
        for (int hf = 0; hf < NH; hf++)
#pragma unroll
            for (int e = 0; e < 16; e++) s[hf][e] = 0.f;
#pragma unroll
        for (int ks = 0; ks < KS; ks++)
#pragma unroll
            for (int hf = 0; hf < NH; hf++) s[hf] = Mfma<T>::run(*(const U4 *)(kt + (krow ^ (32 * ks)) + 32 * hf * G::ROWB), qf[ks], s[hf]);
        // ---- online softmax for this lane's query over its half of the keys (the partner lane l ^ 32 has the others)
        float mloc = -INFINITY;
#pragma unroll
        for (int hf = 0; hf < NH; hf++)
#pragma unroll
            for (int e = 0; e < 16; e++) {
                if (MASKED) {
                    if (32 * hf + 8 * (e >> 2) + (e & 3) >= my_bound - k0 - 4 * g) s[hf][e] = -INFINITY;
                }
                mloc = fmaxf(mloc, s[hf][e]);
            }
        const float mt = fmaxf(mloc, __shfl_xor(mloc, 32, 64)) * scale2;
        // (the largest weight so far is 1, which T holds exactly: a reference that may lag behind the maximum was 1 - 5 % further from
        // the result in 64 bits)
        const bool up = mt > m;
        if (__builtin_amdgcn_ballot_w64(up) != 0) {
            const float mn = up ? mt : m, corr = up ? __builtin_amdgcn_exp2f(m - mn) : 1.f;
            m = mn;
            l *= corr;
#pragma unroll
            for (int t2 = 0; t2 < DT; t2++)
#pragma unroll
                for (int e = 0; e < 16; e++) o[t2][e] *= corr;
        }
        const float mref = MASKED && m == -INFINITY ? 0.f : m;  // (no key seen yet: every exponential is of -inf)
        // (the tile's weights among themselves first: each one straight into the row's sum, a chain as long as the row of keys, was
        // further from it in 64 bits -- 777 keys 3e-7 of it against 7e-8, 32768 keys 1.7e-6 against 3.4e-7 -- and lost weights below 2^-24)
        float lt = 0.f;
#pragma unroll
        for (int hf = 0; hf < NH; hf++)
#pragma unroll
            for (int e = 0; e < 16; e++) {
                s[hf][e] = __builtin_amdgcn_exp2f(fmaf(s[hf][e], scale2, -mref));
                lt += s[hf][e];
            }
        l += lt;
        // ---- O^T += V^T . P^T, keys contracted in the order the D-layout delivers them
#pragma unroll
        for (int st = 0; st < 2 * NH; st++) {
            const f16x_t &ph = s[st >> 1];
            const int e0 = 8 * (st & 1);
            // (results of an exponential: no product that the conversion could be folded into)
            const U4 pf = U4{cvt2<T>(ph[e0 + 0], ph[e0 + 1]), cvt2<T>(ph[e0 + 2], ph[e0 + 3]), cvt2<T>(ph[e0 + 4], ph[e0 + 5]), cvt2<T>(ph[e0 + 6], ph[e0 + 7])};
#pragma unroll
            for (int t2 = 0; t2 < DT; t2++) {
                const char *vr = vt + vrow[t2] + 16 * st * G::ROWB;
                const uint2 lo = lds_read_tr16(vr), hi = lds_read_tr16(vr + 8 * G::ROWB);
                o[t2] = Mfma<T>::run(U4{lo.x, lo.y, hi.x, hi.y}, pf, o[t2]);
            }
        }
    };

    // one barrier per tile: behind it the tile is whole and the other stage free
    int t0 = 0, stage = 0;
    auto next = [&]() {
        // vmcnt(0) lgkmcnt(0): this wave's share of the tile is in LDS, and its reads of the stage that is filled next are through
        __builtin_amdgcn_s_waitcnt(0x0070);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (t0 + kg + KW < ntiles) issue(t0 + kg + KW, stage ^ 1);
    };
    // the rounds whose tiles every row of the workgroup sees in full, then those that need masking
    const int full = R.bound(p, min(R.q_blk, R.Sq - 1)) / KEYS - (KW - 1);
    for (; t0 < full; t0 += KW, stage ^= 1) {
        next();
        tile(grp + stage * G::STAGE, 0, std::false_type{});
    }
    for (; t0 < ntiles; t0 += KW, stage ^= 1) {
        next();
        if ((t0 + kg) * KEYS < wave_bound) tile(grp + stage * G::STAGE, (t0 + kg) * KEYS, std::true_type{});
    }

    l += __shfl_xor(l, 32, 64);
    T *out = (T *)p.out + (size_t)R.b * p.o_bs + (size_t)R.h * p.o_hs + (size_t)qrow * p.o_rs;
    if constexpr (KW == 1) {
        if (qrow >= R.Sq) return;
        const float inv = 1.0f / l;
#pragma unroll
        for (int t2 = 0; t2 < DT; t2++)
#pragma unroll
            for (int e4 = 0; e4 < 4; e4++) {
                const int d = 32 * t2 + 8 * e4 + 4 * g;
                *(uint2 *)(out + d) = uint2{pack2<T>(o[t2][4 * e4 + 0] * inv, o[t2][4 * e4 + 1] * inv),
                                            pack2<T>(o[t2][4 * e4 + 2] * inv, o[t2][4 * e4 + 3] * inv)};
            }
    } else {
        // the groups' results meet in LDS, [word][lane] per wave; group kg adds up its share of the dims, in the order of the groups
        __syncthreads();
        float *mine = (float *)lds + (size_t)w * 64 * G::WORDS + lane;
        mine[0] = m;
        mine[64] = l;
#pragma unroll
        for (int t2 = 0; t2 < DT; t2++)
#pragma unroll
            for (int e = 0; e < 16; e++) mine[(2 + t2 * 16 + e) * 64] = o[t2][e];
        __syncthreads();
        if (qrow >= R.Sq) return;
        constexpr int NE = D / 2 / KW;
        const float *from = (const float *)lds + (size_t)wave * 64 * G::WORDS + lane;
        constexpr int STEP = QW * 64 * G::WORDS;  // to the same wave of the next group
        float mk[KW], mm = -INFINITY, ll = 0.f;
#pragma unroll
        for (int k = 0; k < KW; k++) {
            mk[k] = from[k * STEP];
            mm = fmaxf(mm, mk[k]);
        }
#pragma unroll
        for (int k = 0; k < KW; k++) {
            mk[k] = mk[k] == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mk[k] - mm);
            ll += from[k * STEP + 64] * mk[k];
        }
        const float inv = 1.0f / ll;
        const float *fe = from + (2 + kg * NE) * 64;
#pragma unroll
        for (int q = 0; q < NE / 4; q++) {
            float v[4];
#pragma unroll
            for (int x = 0; x < 4; x++) {
                v[x] = 0.f;
#pragma unroll
                for (int k = 0; k < KW; k++) v[x] += fe[k * STEP + (4 * q + x) * 64] * mk[k];
            }
            const int e4 = kg * (NE / 4) + q, d = 8 * e4 + 4 * g;  // (32 * (e4 / 4) + 8 * (e4 % 4) + 4 * g)
            *(uint2 *)(out + d) = uint2{pack2<T>(v[0] * inv, v[1] * inv), pack2<T>(v[2] * inv, v[3] * inv)};
        }
    }
}

// The same over an int8 cache with a scale per row: 2 x 2 waves, the codes converted on the way to LDS (registers, the next tile's
// loads in flight meanwhile), V^T written there as it is read.  The codes enter both products exactly; a key's scale multiplies its
// score, its value's scale its weight.  (fp16: in units of the largest scale so far, times 2^12, so that small weights stay normal
// numbers and none overflows; a larger scale rescales O^T as a larger maximum does, and the unit is put back at the end.)
// The weights enter as several values of T each, rounded and rest: the row-at-a-time kernel, which also takes these calls,
// keeps them in f32.  Two of fp16 (22 bits: as near to the result in 64 bits as f32 is), three of bf16: with two, 0.2 % of the
// outputs were not the nearest bf16 value where f32 weights leave 0.01 - 0.03 % (32 heads, 128 rows behind 500 keys: two values
// 22.3 us, three 23.5 at D = 128, 13.9 and 14.3 at D = 64; one prompt of 128 rows 9.2 and 9.4).
// A thread stages CH neighbouring keys of the same 8 dims, so V^T goes to LDS CH keys at a time (4- or 8-byte
// writes of values gathered with v_perm) instead of one 2-byte write per value.
constexpr int kPf8Waves = 2, kPf8Groups = 2, kPf8Keys = 64;
template <int D> constexpr size_t pf8_group_bytes() { return (size_t)(kPf8Keys * (D + 8) + D * (kPf8Keys + 4)) * 2 + 2 * kPf8Keys * sizeof(float); }
template <int D> constexpr size_t pf8_lds() {
    const size_t tiles = kPf8Groups * pf8_group_bytes<D>(), merge = (size_t)(kPf8Groups - 1) * kPf8Waves * 64 * (D / 2 + 2) * sizeof(float);
    return tiles > merge ? tiles : merge;
}

template <typename T, int D> __global__ __launch_bounds__(kPf8Waves *kPf8Groups * 64, 2) void attn_prefill_kv8_kernel(AttnParams p) {
    constexpr int QW = kPf8Waves, KW = kPf8Groups, kPfKeys = kPf8Keys;
    constexpr int kPfThreads = QW * 64;  // threads of a group
    constexpr bool UNITS = std::is_same<T, f16_t>::value;
    constexpr int LDK = D + 8;          // K tile row stride (elements): conflict-free 16-byte reads
    constexpr int LDV = kPfKeys + 4;    // V^T tile row stride
    constexpr int KS = D / 16;          // k-steps of the S^T product
    constexpr int DT = D / 32;          // 32-row tiles of O^T
    constexpr int CH = (kPfKeys * D / 8) / kPfThreads;  // 16-byte chunks per thread and tile (2 or 4): neighbouring keys
    static_assert(CH == 2 || CH % 4 == 0, "a thread stages 2 or a multiple of 4 neighbouring keys");
    extern __shared__ __align__(16) char lds[];
    const int kg = threadIdx.x / kPfThreads;  // key group
    uint16_t *Ks = (uint16_t *)(lds + kg * pf8_group_bytes<D>()), *Vt = Ks + kPfKeys * LDK;
    float *ksc = (float *)(Vt + D * LDV), *vsc = ksc + kPfKeys;  // (one tile's: written and read between two barriers)

    const int tid = threadIdx.x % kPfThreads, lane = tid & 63, wave = tid >> 6;
    const int col = lane & 31, g = lane >> 5;
    const PfRows R(p, QW * 32);
    const int Sq = R.Sq, q_blk = R.q_blk, blk_bound = R.blk_bound;
    const int qrow = q_blk + wave * 32 + col, qrow_c = min(qrow, Sq - 1);  // this lane's query row
    const int my_bound = R.bound(p, qrow_c);
    const int wave_bound = R.bound(p, min(q_blk + wave * 32 + 31, Sq - 1));
    const int wave_all = R.bound(p, min(q_blk + wave * 32, Sq - 1));  // tiles that end at or below it need no masking
    const int ntiles = (blk_bound + kPfKeys - 1) / kPfKeys;

    using Chunk = uint2;  // 8 elements of a cached row
    const size_t kv_row0 = (size_t)(R.b * p.Hkv + R.hkv) * p.cache_len;
    const int8_t *Kg = (const int8_t *)p.k + kv_row0 * D, *Vg = (const int8_t *)p.v + kv_row0 * D;
    // a tile travels global -> registers (a round ahead) -> LDS.
    // Thread t stages the keys CH * (t / (D/8)) + 0 .. CH-1 of a tile, dims 8 * (t % (D/8)) .. +7.
    // Rows past the end are clamped to the last visible key: whatever they hold is masked out.
    const int key0 = (tid / (D / 8)) * CH, dd = (tid % (D / 8)) * 8;
    Chunk rk[CH], rv[CH];
    T rs = T{};  // the scale of key tid % 64, of K (tid < 64) or V
    auto load_tile = [&](int t, Chunk *k_, Chunk *v_) {
#pragma unroll
        for (int c = 0; c < CH; c++) {
            const int key = min(t * kPfKeys + key0 + c, blk_bound - 1);
            k_[c] = *(const Chunk *)(Kg + (size_t)key * D + dd);
            v_[c] = *(const Chunk *)(Vg + (size_t)key * D + dd);
        }
        if (tid < 128) rs = ((const T *)(tid < 64 ? p.k_scale : p.v_scale))[kv_row0 + min(t * kPfKeys + (tid & 63), blk_bound - 1)];
    };
    auto operand = [](const Chunk &c) -> U4 { return i8x8_to_operand<T>(c.x, c.y); };
    auto store_tile = [&](const Chunk *k_, const Chunk *v8) {
        U4 v_[CH];
#pragma unroll
        for (int c = 0; c < CH; c++) v_[c] = operand(v8[c]);
        if (tid < 128) ksc[tid] = Elem<T>::ld(&rs, 0);
#pragma unroll
        for (int c = 0; c < CH; c++) *(U4 *)&Ks[(key0 + c) * LDK + dd] = operand(k_[c]);
        // V^T[d][key0 .. key0 + CH - 1] for the 8 dims: dword i of a chunk holds dims 2i (low half) and 2i + 1
#pragma unroll
        for (int i = 0; i < 4; i++) {
            uint32_t w[CH];
#pragma unroll
            for (int c = 0; c < CH; c++) w[c] = i == 0 ? v_[c].x : i == 1 ? v_[c].y : i == 2 ? v_[c].z : v_[c].w;
            uint16_t *lo = &Vt[(dd + 2 * i) * LDV + key0], *hi = &Vt[(dd + 2 * i + 1) * LDV + key0];
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
    if (kg < ntiles) load_tile(kg, rk, rv);
    // Q^T fragments: B operand, lane (query col, g): d = 16*ks + 8*g .. +7
    const T *Q = (const T *)p.q + (size_t)R.b * p.q_bs + (size_t)R.h * p.q_hs + (size_t)qrow_c * p.q_rs;
    U4 qf[KS];
#pragma unroll
    for (int ks = 0; ks < KS; ks++) qf[ks] = *(const U4 *)(Q + 16 * ks + 8 * g);
    if (p.rope_q) pf_rotate<T, D>(p, qrow_c, g, qf);

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
    // one tile of 64 keys = two S^T tiles (rows = keys, cols = queries), one softmax update, 4 k-steps of P.V
    auto tile = [&](int k0, auto masked) {
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
                const U4 a = *(const U4 *)&Ks[(32 * hf + col) * LDK + 16 * ks + 8 * g];
                s[hf] = Mfma<T>::run(a, qf[ks], s[hf]);
            }
#pragma unroll
        for (int hf = 0; hf < 2; hf++)
#pragma unroll
            for (int e4 = 0; e4 < 4; e4++) {
                const float4 f = *(const float4 *)&ksc[32 * hf + 8 * e4 + 4 * g];
                s[hf][4 * e4] *= f.x; s[hf][4 * e4 + 1] *= f.y; s[hf][4 * e4 + 2] *= f.z; s[hf][4 * e4 + 3] *= f.w;
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
        float4 vs[8];
        float to_unit = 1.f;
#pragma unroll
        for (int i = 0; i < 8; i++) vs[i] = *(const float4 *)&vsc[32 * (i >> 2) + 8 * (i & 3) + 4 * g];
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
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float f[4] = {vs[i].x, vs[i].y, vs[i].z, vs[i].w};
#pragma unroll
            for (int e = 0; e < 4; e++) s[i >> 2][4 * (i & 3) + e] *= f[e] * to_unit;
        }
        // ---- O^T += V^T . P^T, keys contracted in the order the D-layout delivers them
#pragma unroll
        for (int st = 0; st < 4; st++) {
            const f16x_t &ph = s[st >> 1];
            const int e0 = 8 * (st & 1);
            constexpr int PARTS = kParts<T>;
            U4 pf[PARTS];
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
#pragma unroll
            for (int t2 = 0; t2 < DT; t2++) {
                const uint16_t *vr = &Vt[(32 * t2 + col) * LDV + 16 * st + 4 * g];
                const uint2 lo = *(const uint2 *)vr, hi = *(const uint2 *)(vr + 8);
#pragma unroll
                for (int part = 0; part < PARTS; part++) o[t2] = Mfma<T>::run(U4{lo.x, lo.y, hi.x, hi.y}, pf[part], o[t2]);
            }
        }
    };
    auto compute = [&](int t) {
        const int k0 = t * kPfKeys;
        if (k0 + kPfKeys <= wave_all) tile(k0, std::false_type{});
        else if (k0 < wave_bound) tile(k0, std::true_type{});
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

    // group kg takes tiles kg, kg + KW, ..: one LDS tile per group, the next one in registers meanwhile
    for (int t = kg; t - kg < ntiles; t += KW) {  // (the same number of rounds for every group)
        if (t < ntiles) store_tile(rk, rv);
        __syncthreads();
        if (t + KW < ntiles) load_tile(t + KW, rk, rv);
        if (t < ntiles) compute(t);
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

    // ---- out[query, d] = O^T[d, query] / l
    l += __shfl_xor(l, 32, 64);
    if (qrow < Sq) {
        T *out = (T *)p.out + (size_t)R.b * p.o_bs + (size_t)R.h * p.o_hs + (size_t)qrow * p.o_rs;
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

template <typename F> static int pf_launch(F kernel, const AttnParams &p, int rows, int threads, size_t lds, bool &lds_set, hipStream_t s) {
    if (!lds_set && lds > 64 * 1024) {
        MYNN_HIP(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
        lds_set = true;
    }
    MYNN_LAUNCH(kernel, dim3(p.B * p.Hq, (p.Sq + rows - 1) / rows), dim3(threads), lds, s, p);
    return launch_status("attn_prefill_kernel");
}
template <typename T, int D, bool PAGED, int KEYS, int QW, int KW> static int pf_go(const AttnParams &p, hipStream_t s) {
    using G = PfTile<D, KEYS, QW, KW>;
    static bool lds_set = false;
    return pf_launch(attn_prefill_kernel<T, D, PAGED, KEYS, QW, KW>, p, G::ROWS, G::THREADS, G::LDS, lds_set, s);
}
template <typename T, int D> static int pf_go_kv8(const AttnParams &p, hipStream_t s) {
    static bool lds_set = false;
    return pf_launch(attn_prefill_kv8_kernel<T, D>, p, kPf8Waves * 32, kPf8Waves * kPf8Groups * 64, pf8_lds<D>(), lds_set, s);
}
// Which split, by the workgroups that 128 rows each would make (32 heads, causal, bf16; microseconds of an operator call, which is
// never below 6.5; keys per tile / waves of rows x key groups):
//   D = 64        64 / 4 x 1   64 / 2 x 2   32 / 2 x 2      D = 128        64 / 4 x 1   64 / 2 x 2   32 / 2 x 2   64 / 4 x 2
//   1 x  300             7.6          6.9          7.1      1 x  128              7.4          6.9          7.0          9.3
//   1 x  777            14.4         11.2         12.2      1 x  500             15.2         12.1         13.3         15.3
//   1 x 1200            20.0         15.8         17.8      1 x  777             20.5         18.8         18.2         19.3
//   1 x 1300            21.3         17.0         18.5      1 x 1200             30.1         34.8         26.3         25.9
//   1 x 1600            25.5         23.5         23.3      1 x 1300             32.0         38.2         27.9         28.6
//   1 x 1900            30.4         30.0         28.9      1 x 1600             38.9         47.0         37.4         36.4
//   1 x 2048            32.8         32.7         32.1      1 x 1900             47.9         61.5         50.4         44.7
//   2 x  936            17.9         20.1         17.9      1 x 2048             52.1         67.6         53.8         48.7
//   8 x 1024            56.8         84.4         69.3      2 x  936             27.6         41.8         33.6         32.9
// (4 x 1 and 32 / 2 x 2 share a CU with a second workgroup.)  Beyond 320 workgroups it is the heads that count, as a launch lasts as long
// as the last rows of one: up to 32 of them (over all sequences) the groups of keys pay, 48 heads x 1100 rows take 4 x 1 (D = 64 20.1 us
// against 21.0, D = 128 30.1 against 32.1), 40 are a tie.  Up to 64 rows there is one tile and nothing to split.
template <typename T, int D, bool PAGED> static int pf_pick(const AttnParams &p, hipStream_t s) {
    const long wgs = (long)p.B * p.Hq * ((p.Sq + 127) / 128);
    const bool few_heads = wgs <= 512 && (long)p.B * p.Hq <= 32;
    if (p.Sq > 64) {
        if constexpr (D == 64) {
            if (wgs <= 320 || few_heads) return pf_go<T, D, PAGED, 64, 2, 2>(p, s);
        } else {
            if (wgs <= 128) return pf_go<T, D, PAGED, 64, 2, 2>(p, s);
            if (p.Sq > 128 && wgs <= 320) return pf_go<T, D, PAGED, 32, 2, 2>(p, s);
            if (few_heads) return pf_go<T, D, PAGED, 64, 4, 2>(p, s);
        }
    }
    return pf_go<T, D, PAGED, 64, 4, 1>(p, s);
}

int attention_prefill_launch(const AttnParams &p, int D, int dtype, int kv_int8, hipStream_t s) {
    MYNN_REQUIRE((p.Sq + 31) / 32 <= 65535, MYNN_ERR_UNSUPPORTED, "attention: Sq = %d exceeds the grid", p.Sq);
    if (p.page_table) {
        const int P = 1 << p.page_shift;
        MYNN_REQUIRE(!kv_int8 && P >= kPfPage && p.pages_per_seq <= 64 && p.cache_len == p.pages_per_seq << p.page_shift, MYNN_ERR_UNSUPPORTED,
                     "paged prefill attention: %d pages of %d rows per sequence (at most 64 pages of 2^n >= %d rows, 16-bit)",
                     p.pages_per_seq, P, kPfPage);
    }
    return dispatch_dtype16(dtype, [&](auto *t) {
        using T = std::remove_pointer_t<decltype(t)>;
        if (kv_int8) return D == 64 ? pf_go_kv8<T, 64>(p, s) : pf_go_kv8<T, 128>(p, s);
        if (p.page_table) return D == 64 ? pf_pick<T, 64, true>(p, s) : pf_pick<T, 128, true>(p, s);
        return D == 64 ? pf_pick<T, 64, false>(p, s) : pf_pick<T, 128, false>(p, s);
    });
}

}  // namespace mynn
