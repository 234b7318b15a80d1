// Streaming GQA decode attention for large (batch x context) products: one query row per sequence,
// 16-bit or int8 (per-token scales) K/V, head_dim 64 or 128, up to 8 query heads per kv head.
//
// attention_decode.hip is built for latency (one pass, everything in flight at once, one workgroup
// per CU); with megabytes of K/V per launch the job is bandwidth instead, and this kernel
// keeps the loads streaming: a workgroup of 4 or 8 waves (see stream_eight_waves) walks its key range in tiles of 32 keys per wave,
// the next tile's K and V already in registers while the current one is used.  Both products run on
// the matrix cores (v_mfma_f32_16x16x32), with the query heads as the 16 columns (zero beyond G):
//   scores   S[keys x heads] = K_tile . Q^T; K rows are the A operand straight from global memory
//            (lane l holds key l%16, dims 8*(l/16)..+7 of each 32-dim block),
//   softmax  online, per head, f32; a lane holds one head (l%16), so rescaling its accumulators is
//            lane-local; the tile's p values go to LDS as [head][key] in the storage type,
//   P.V      O^T[dims x heads] += V^T . P; V needs its keys along the reduction, so the tile is parked
//            in LDS (row stride 136 bytes: conflict-free) and read back two dims at a time, each pair of
//            keys split into an "even dims" and an "odd dims" operand by one v_perm -- the 16 rows of
//            an MFMA tile are dims 32c + 2r (+1),
// then waves are combined through LDS, and key ranges by the workgroup of a (sequence, kv head) that arrives last
// (or by a second launch, attn_merge_kernel, where the caller's scratch memory has no arrival counters).
// P enters the second product as a sum of storage-type values (two of fp16, three of bf16).  Replaces the
// reference's attention_decode (attention.cuh:495-606) for these shapes.
#pragma once
#include <type_traits>

#include "attention.h"
#include "kernels.h"
#include "mfma.h"

namespace mynn {

typedef float f4_t __attribute__((ext_vector_type(4)));
template <typename T> struct Mfma16;
template <> struct Mfma16<f16_t> {
    __device__ static f4_t run(const U4 &a, const U4 &b, f4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(h8_t, a), __builtin_bit_cast(h8_t, b), c, 0, 0, 0);
    }
};
template <> struct Mfma16<bf16_t> {
    __device__ static f4_t run(const U4 &a, const U4 &b, f4_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(b8_t, a), __builtin_bit_cast(b8_t, b), c, 0, 0, 0);
    }
};

constexpr int kStreamTile = 32;
// KVI8: int8 caches with one scale per token row (QuantizingKVCacheUpdate): K and V are widened exactly to
// the 16-bit type in registers, the key's k scale multiplies its score and its v scale its p.
// PAGED: K/V rows are found through a page table (AttnParams::page_table).  A tile of 32 keys never crosses a page
// (pages hold a power of two >= 32 rows, tiles start at multiples of 32), so the page is a wave-uniform value per
// tile: the workgroup's part of the table sits in one register (lane i = the i-th page of its key range, at most 64)
// and a tile picks its entry with v_readlane -- no dependent load in the key loop.
// FUSE: q is the raw q|k|v projection row of the sequence; the kernel rotates the queries itself, and the wave whose tiles
// hold row *d_past makes the new key (rotated) and value, writes them to the cache and keeps them in LDS, where it takes
// them from when it comes to their tile: the RoPE + append launch in front of it disappears and nobody waits for a store.
// (Written first and read back like any other row, behind a barrier: 8 us more at 32 sequences x 2048 keys.)
// What the kernel needs of AttnParams (a launch pays for its argument bytes: 0.9 us of host time for 300 against 60).
struct StreamRest {
    void *out;
    const void *k_scale, *v_scale, *cos_t, *sin_t;
    const int32_t *page_table;
    float *part_o, *part_ml;
    int *arrive;
    long q_bs, q_hs, o_bs, o_hs;
    float scale;
    int Hq, cache_len, active, nsplit, page_shift, pages_per_seq;
};
// ... and what its first loads need: leading scalar arguments, which arrive preloaded with the wave, where members of a struct take a load first (4 sequences x 2048
// keys, D = 64: 7.66 -> 7.48 us)
struct StreamParams : StreamRest {
    const void *q, *k, *v;
    const int32_t *d_active, *d_past;
    const int64_t *d_pos;
    int Hkv, slice;
};
enum StreamForm { kOneTile, kTiles, kTilesOnce };
// LDS of a workgroup of W waves, in bytes: V tiles, p tiles, (m, l) of the waves, the new row and its scales
template <typename T, int D, int W> struct StreamLds {
    static constexpr int V = kStreamTile * (D + 4) * 2, P = kParts<T> * 16 * (kStreamTile + 8) * 2, ML = 8 * 4;
    static constexpr int P0 = W * V, M0 = P0 + W * P, L0 = M0 + W * ML, ROW0 = L0 + W * ML, SCALE0 = ROW0 + 2 * D * 2, BYTES = SCALE0 + 16;
};
// FORM: kOneTile where the key range has a tile per wave, kTiles where a wave walks several, the next one's loads in flight (with both
// in one kernel, chosen by the range, the walk is 1 - 2 % slower: 17 sequences x 1056 keys, D = 128, 14.7 us against 14.4; the walk
// over a single tile 5 %: 4 x 1000, D = 64, 7.2 against 6.9).
// kTilesOnce: value rows, whole lines per instruction, are read with the hint that they won't be wanted again (stream_once below).  Key
// rows are read 64 bytes at a time, a line by two instructions: the hint there gave 2.5 % of a decode step of 32 sequences x 2048
// keys where this one gives 3.2, both together 3.0.
__device__ __forceinline__ U4 load_once(const U4 *p) { return __builtin_nontemporal_load(p); }
template <typename T, int D, int G, bool KVI8, bool PAGED, bool FUSE, int W, int FORM>
__global__ __launch_bounds__(W * 64) void attn_stream_kernel(const void *q, const void *k, const void *v, const int32_t *d_active, const int32_t *d_past,
                                                               const int64_t *d_pos, int Hkv, int slice, StreamRest rest) {
    const StreamParams p{rest, q, k, v, d_active, d_past, d_pos, Hkv, slice};
    using Lds = StreamLds<T, D, W>;
    constexpr int kStreamWaves = W, kStreamThreads = W * 64;
    extern __shared__ __align__(16) char sm[];
    constexpr int KB = D / 32;              // 32-dim blocks of a key row
    constexpr int LPK = D / 8;              // lanes per key row when a tile is loaded 16 bytes per lane
    constexpr int KPP = 64 / LPK;           // key rows per load pass of a wave
    constexpr int NP = kStreamTile / KPP;   // load passes per tile (V)
    constexpr int VST = D + 4;              // V tile row stride in elements (D*2 + 8 bytes)
    constexpr int PST = kStreamTile + 8;    // p tile row stride in elements (16-byte aligned rows)
    uint16_t(*v_s)[kStreamTile * VST] = (uint16_t(*)[kStreamTile * VST])sm;
    static_assert(Lds::V == kStreamTile * VST * 2 && Lds::P == kParts<T> * 16 * PST * 2 && G <= 8, "the layout above");
    // the storage type keeps 8 (bf16) or 11 (fp16) bits of p, and over thousands of keys that rounding shows
    // in small outputs: further tiles hold the remainder p - T(p), and what its rounding leaves out, and feed products of
    // their own.  Two values of fp16 measure as f32 weights do against 64 bits; with two of bf16 0.15 - 0.3 % of the outputs
    // were not the nearest value, with f32 weights or three values 0 - 0.05 % (at no cost: 32 sequences x 2048 keys, D = 128,
    // 55.7 us with either, over an int8 cache 30.4 with two and 30.3 - 30.8 with three)
    constexpr int PARTS = kParts<T>;
    // fp16 has the bits but not the range: p of a far-away key is subnormal or zero in fp16 while
    // thousands of them still add up, so p is stored times 2^12 and the factor taken out at the end
    constexpr float kPScale = std::is_same<T, f16_t>::value ? 4096.f : 1.f;
    uint16_t(*p_s)[PARTS * 16 * PST] = (uint16_t(*)[PARTS * 16 * PST])(sm + Lds::P0);
    float(*m_s)[8] = (float(*)[8])(sm + Lds::M0), (*l_s)[8] = (float(*)[8])(sm + Lds::L0);
    // (a wave's results take the place of its own V tile once it is through)
    static_assert(G * D * sizeof(float) <= kStreamTile * VST * sizeof(uint16_t), "results of a wave fit its V tile");
    auto o_s = [&](int w) { return (float(*)[D])v_s[w]; };

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int bhkv = blockIdx.x, split = blockIdx.y;
    const int b = bhkv / p.Hkv, hkv = bhkv % p.Hkv;
    const int head0 = hkv * G;
    const int active = p.d_active ? *p.d_active : p.active;
    const int bound = min(active, p.cache_len);
    const int k0 = split * p.slice, k1 = min(bound, k0 + p.slice);
    // key ranges that hold a row; the launch is sized for the whole cache, the ranges past the context only leave
    const int n_act = p.arrive ? max(1, min(p.nsplit, (bound + p.slice - 1) / p.slice)) : p.nsplit;
    const int past = FUSE ? *p.d_past : 0;
    const bool owner = FUSE && split == min(past / p.slice, p.nsplit - 1);
    if (split >= n_act && !owner) return;
    const size_t kv_base = PAGED ? 0 : (size_t)bhkv * p.cache_len;
    using TKV = typename std::conditional<KVI8, int8_t, T>::type;
    using Chunk = typename std::conditional<KVI8, uint2, U4>::type;  // 8 elements of a cached row
    const TKV *Kp = (const TKV *)p.k + kv_base * D, *Vp = (const TKV *)p.v + kv_base * D;
    const T *ksc = (const T *)p.k_scale + kv_base, *vsc = (const T *)p.v_scale + kv_base;  // KVI8 only
    // PAGED: pool row (in units of rows of one head) of row `r` of the tile starting at t0 = page's first row + r % P
    const int psh = p.page_shift, pmask = (1 << psh) - 1, pg0 = k0 >> psh;
    int pg_reg = 0;
    if constexpr (PAGED) {
        if (pg0 + lane < p.pages_per_seq) pg_reg = p.page_table[(size_t)b * p.pages_per_seq + pg0 + lane];
    }
    auto page_rows0 = [&](int t0) -> size_t {
        const int pg = __builtin_amdgcn_readlane(pg_reg, __builtin_amdgcn_readfirstlane((t0 >> psh) - pg0));
        return ((size_t)pg * p.Hkv + hkv) << psh;
    };
    // FUSE: the new row as the cache holds it, and its scales (KVI8)
    TKV(*new_row)[D] = (TKV(*)[D])(sm + Lds::ROW0);
    T *new_scale = (T *)(sm + Lds::SCALE0);
    const bool new_here = FUSE && past >= k0 && past < k1;  // ... is one of this key range's
    const bool new_mine = owner && wave == (new_here ? ((past - k0) / kStreamTile) % kStreamWaves : 0);
    struct NewRow {
        T lo[2], hi[2], cl, ch, sl, sh;  // as loaded: k and v, cos and sin of this lane's pair (elements i and i + D/2)
    };
    auto request = [&](NewRow &r) {  // (in front of the first tile's loads: loads return in order)
        constexpr int half = D / 2;
        const T *src = (const T *)p.q + (size_t)b * p.q_bs + (size_t)(p.Hq + hkv) * D;
        const T *ct = (const T *)p.cos_t + (size_t)*p.d_pos * D, *st = (const T *)p.sin_t + (size_t)*p.d_pos * D;
        const int i = min(lane, half - 1);
#pragma unroll
        for (int v = 0; v < 2; v++) {
            r.lo[v] = src[(size_t)v * p.Hkv * D + i];
            r.hi[v] = src[(size_t)v * p.Hkv * D + i + half];
        }
        r.cl = ct[i];
        r.ch = ct[i + half];
        r.sl = st[i];
        r.sh = st[i + half];
    };
    auto append = [&](const NewRow &r) {
        constexpr int half = D / 2;
        const size_t tok = kv_cache_row(KvPaging{PAGED ? p.page_table : nullptr, p.page_shift, p.pages_per_seq}, b, hkv, past, p.Hkv, p.cache_len);
        const int i = min(lane, half - 1);
        auto f = [](const T &x) { return Elem<T>::ld(&x, 0); };
        float lo[2] = {f(r.lo[0]), f(r.lo[1])}, hi[2] = {f(r.hi[0]), f(r.hi[1])};
        const float rl = Elem<T>::rnd(lo[0] * f(r.cl) - hi[0] * f(r.sl));
        const float rh = Elem<T>::rnd(hi[0] * f(r.ch) + lo[0] * f(r.sh));
        lo[0] = rl;
        hi[0] = rh;
#pragma unroll
        for (int v = 0; v < 2; v++) {
            TKV *dst = (TKV *)(v ? p.v : p.k) + tok * D;
            if constexpr (KVI8) {  // the rule of rope_quant_kv_append_kernel
                const float amax = wave_max(fmaxf(fabsf(lo[v]), fabsf(hi[v])));
                const float inv = amax == 0.f ? 0.f : 127.0f / amax;
                auto code = [&](float x) -> int8_t {
                    const float a = x * inv;
                    const int q = (int)(a + (a >= 0.f ? 0.5f : -0.5f));
                    return (int8_t)(q < -128 ? -128 : (q > 127 ? 127 : q));
                };
                Elem<T>::st(&new_scale[v], 0, amax * (1.0f / 127.0f));
                if (lane == 0) Elem<T>::st((T *)(v ? p.v_scale : p.k_scale), tok, amax * (1.0f / 127.0f));
                new_row[v][i] = code(lo[v]);
                new_row[v][i + half] = code(hi[v]);
            } else {
                Elem<T>::st(new_row[v], i, lo[v]);
                Elem<T>::st(new_row[v], i + half, hi[v]);
            }
            if (lane < half) {
                dst[lane] = new_row[v][lane];
                dst[lane + half] = new_row[v][lane + half];
            }
        }
    };
    if constexpr (FUSE) {
        if (split >= n_act) {  // a range without rows that the new one is appended behind
            if (new_mine) {
                NewRow r;
                request(r);
                append(r);
            }
            return;
        }
    }
    auto operand = [](const Chunk &c) -> U4 {
        if constexpr (KVI8) return i8x8_to_operand<T>(c.x, c.y);
        else return c;
    };
    const int col = lane & 15, quad = lane >> 4;  // MFMA column (head) and row/k group of this lane

    // Q^T as the B operand of the score product: column = head, k = dims 8*quad..+7 of each block
    U4 qf[KB], cs[2][FUSE ? KB : 1];
    {
        const T *qrow = (const T *)p.q + (size_t)b * p.q_bs + (size_t)(head0 + (col < G ? col : 0)) * p.q_hs;
#pragma unroll
        for (int j = 0; j < KB; j++) {
            qf[j] = *(const U4 *)(qrow + j * 32 + quad * 8);
            if (col >= G) qf[j] = U4{0u, 0u, 0u, 0u};
            if constexpr (FUSE) {
                cs[0][j] = *(const U4 *)((const T *)p.cos_t + (size_t)*p.d_pos * D + j * 32 + quad * 8);
                cs[1][j] = *(const U4 *)((const T *)p.sin_t + (size_t)*p.d_pos * D + j * 32 + quad * 8);
            }
        }
    }

    // running state of head `col`: maximum, partial sum (the 4 quads hold parts), O^T accumulators
    // acc[c][par][e] = dim 32c + 2*(4*quad + e) + par
    float m_run = -INFINITY, l_run = 0.f;
    // UNITS: the scale of a value multiplies its key's weight, so with scales of 16 and more (values beyond 2000) the weights
    // would pass fp16's largest number: they and the accumulators are then kept divided by a power of two, one for the wave
    constexpr bool UNITS = KVI8 && std::is_same<T, f16_t>::value;
    float unit = 1.f, to_unit = kPScale;  // kPScale / unit
    f4_t acc[KB][2];
#pragma unroll
    for (int c = 0; c < KB; c++)
#pragma unroll
        for (int par = 0; par < 2; par++) acc[c][par] = f4_t{0.f, 0.f, 0.f, 0.f};

    const int vk = lane / LPK, vd = (lane % LPK) * 8;  // V load: key row within a pass, dim offset
    // (KVI8: the scales of the lane's 2 x 4 score keys travel with the tile, 8 bytes per load; the cache
    // length is a multiple of 32 there, so a tile never reaches past its row of scales)
    auto load_tile = [&](int t0, Chunk (*kr)[KB], Chunk *vr, uint2 *sr) {
        size_t po = 0;
        if constexpr (PAGED) po = page_rows0(t0);
        auto at = [&](int row) -> size_t {
            if constexpr (PAGED) return po + (size_t)(row & pmask);
            else return (size_t)row;
        };
        if constexpr (KVI8) {
#pragma unroll
            for (int a = 0; a < 2; a++) {
                sr[a] = *(const uint2 *)(ksc + at(t0 + a * 16 + quad * 4));
                sr[2 + a] = *(const uint2 *)(vsc + at(t0 + a * 16 + quad * 4));
            }
        }
        // rows past the range re-read the last valid row; their scores are masked below
#pragma unroll
        for (int a = 0; a < 2; a++) {
            const int krow = min(t0 + a * 16 + col, k1 - 1);
#pragma unroll
            for (int j = 0; j < KB; j++) kr[a][j] = *(const Chunk *)(Kp + at(krow) * D + j * 32 + quad * 8);
        }
#pragma unroll
        for (int q = 0; q < NP; q++) {
            const int vrow = min(t0 + q * KPP + vk, k1 - 1);
            const Chunk *src = (const Chunk *)(Vp + at(vrow) * D + vd);
            if constexpr (FORM == kTilesOnce) vr[q] = load_once(src);
            else vr[q] = *src;
        }
    };

    uint16_t *vt = v_s[wave], *pt = p_s[wave];
    auto scale_of = [](const uint2 &four, int e) -> float {  // element e of four packed storage-type values
        const uint32_t w = e < 2 ? four.x : four.y;
        const uint16_t b = (uint16_t)((e & 1) ? w >> 16 : w & 0xFFFFu);
        T v = __builtin_bit_cast(T, b);
        return Elem<T>::ld(&v, 0);
    };
    auto process = [&](int t, Chunk (*kr)[KB], Chunk *vr, uint2 *sr) {
        if constexpr (FUSE) {
            if (new_here && new_mine && past >= t && past < t + kStreamTile) {
                // (rows past the range stand for its last one, which may be the new row: no old content of it is used)
#pragma unroll
                for (int a = 0; a < 2; a++)
                    if (min(t + a * 16 + col, k1 - 1) == past) {
#pragma unroll
                        for (int j = 0; j < KB; j++) kr[a][j] = *(const Chunk *)&new_row[0][j * 32 + quad * 8];
                    }
#pragma unroll
                for (int q = 0; q < NP; q++)
                    if (min(t + q * KPP + vk, k1 - 1) == past) vr[q] = *(const Chunk *)&new_row[1][vd];
                if constexpr (KVI8) {
#pragma unroll
                    for (int a = 0; a < 2; a++) {
                        const int e = past - (t + a * 16 + quad * 4);
                        if (e >= 0 && e < 4) {
                            auto put = [&](uint2 &four, T v) {
                                const uint32_t bits = __builtin_bit_cast(uint16_t, v), keep = e & 1 ? 0xFFFFu : 0xFFFF0000u, sh = e & 1 ? 16 : 0;
                                if (e < 2) four.x = (four.x & keep) | bits << sh;
                                else four.y = (four.y & keep) | bits << sh;
                            };
                            put(sr[a], new_scale[0]);
                            put(sr[2 + a], new_scale[1]);
                        }
                    }
                }
            }
        }
        // ---- park V: [key][dim], two 8-byte stores per lane and pass
#pragma unroll
        for (int q = 0; q < NP; q++) {
            uint2 *dst = (uint2 *)&vt[(q * KPP + vk) * VST + vd];
            const U4 v = operand(vr[q]);
            dst[0] = uint2{v.x, v.y};
            dst[1] = uint2{v.z, v.w};
        }
        // ---- scores: lane = head col, keys 16a + 4*quad + e
        float sv[2][4], tmax = -INFINITY;
#pragma unroll
        for (int a = 0; a < 2; a++) {
            f4_t s4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int j = 0; j < KB; j++) s4 = Mfma16<T>::run(operand(kr[a][j]), qf[j], s4);
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int key = t + a * 16 + quad * 4 + e;
                float sc = s4[e];
                if constexpr (KVI8) sc *= scale_of(sr[a], e);
                sv[a][e] = key < k1 ? sc * p.scale : -INFINITY;
                tmax = fmaxf(tmax, sv[a][e]);
            }
        }
        tmax = fmaxf(tmax, __shfl_xor(tmax, 16, 64));
        tmax = fmaxf(tmax, __shfl_xor(tmax, 32, 64));
        const float m_new = fmaxf(m_run, tmax);  // finite: the tile has at least one key in range
        float alpha = fast_exp(m_run - m_new), back = 1.f;
        m_run = m_new;
        float psum = 0.f;
        if constexpr (UNITS) {
            float vm = 0.f;
#pragma unroll
            for (int a = 0; a < 2; a++)
#pragma unroll
                for (int e = 0; e < 4; e++) vm = fmaxf(vm, t + a * 16 + quad * 4 + e < k1 ? fabsf(scale_of(sr[2 + a], e)) : 0.f);
            if (__builtin_amdgcn_ballot_w64(vm > 8.f * unit) != 0) {
                vm = fmaxf(vm, __shfl_xor(vm, 16, 64));
                vm = fmaxf(vm, __shfl_xor(vm, 32, 64));
                // (its power of two; scales of fp16 end at 2^16)
                const float un = fmaxf(unit, __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, fminf(vm, 65536.f)) & 0x7F800000u));
                const float inv = __builtin_bit_cast(float, 0x7F000000u - __builtin_bit_cast(uint32_t, un));
                back = unit * inv;
                unit = un;
                to_unit = kPScale * inv;
            }
        }
#pragma unroll
        for (int a = 0; a < 2; a++) {
            float pe[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                pe[e] = fast_exp(sv[a][e] - m_new);  // 0 for keys past the range
                psum += pe[e];
                if constexpr (KVI8) pe[e] = t + a * 16 + quad * 4 + e < k1 ? pe[e] * scale_of(sr[2 + a], e) : 0.f;
            }
            // p[head][16a + 4*quad .. +3] in the storage type
#pragma unroll
            for (int e = 0; e < 4; e++) pe[e] *= UNITS ? to_unit : kPScale;
#pragma unroll
            for (int part = 0; part < PARTS; part++) {
                const uint32_t w0 = take_part<T>(pe[0], pe[1]), w1 = take_part<T>(pe[2], pe[3]);
                *(uint2 *)&pt[part * 16 * PST + col * PST + a * 16 + quad * 4] = uint2{w0, w1};
            }
        }
        l_run = l_run * alpha + psum;
        alpha *= back;
        if (alpha != 1.f) {
#pragma unroll
            for (int c = 0; c < KB; c++)
#pragma unroll
                for (int par = 0; par < 2; par++) acc[c][par] *= alpha;
        }
        __builtin_amdgcn_wave_barrier();
        // ---- O^T += V^T . P: B operand = p[head col][keys 8*quad..+7]; A operands from V dword pairs
        U4 pf[PARTS];
#pragma unroll
        for (int part = 0; part < PARTS; part++) pf[part] = *(const U4 *)&pt[part * 16 * PST + col * PST + quad * 8];
#pragma unroll
        for (int c = 0; c < KB; c++) {
            uint32_t w[8];
#pragma unroll
            for (int i = 0; i < 8; i++) w[i] = *(const uint32_t *)&vt[(quad * 8 + i) * VST + c * 32 + col * 2];
            U4 ev, od;  // keys 8*quad..+7 at dim 32c + 2*col and at the next dim
            ev.x = __builtin_amdgcn_perm(w[1], w[0], 0x05040100u); od.x = __builtin_amdgcn_perm(w[1], w[0], 0x07060302u);
            ev.y = __builtin_amdgcn_perm(w[3], w[2], 0x05040100u); od.y = __builtin_amdgcn_perm(w[3], w[2], 0x07060302u);
            ev.z = __builtin_amdgcn_perm(w[5], w[4], 0x05040100u); od.z = __builtin_amdgcn_perm(w[5], w[4], 0x07060302u);
            ev.w = __builtin_amdgcn_perm(w[7], w[6], 0x05040100u); od.w = __builtin_amdgcn_perm(w[7], w[6], 0x07060302u);
#pragma unroll
            for (int part = 0; part < PARTS; part++) {
                acc[c][0] = Mfma16<T>::run(ev, pf[part], acc[c][0]);
                acc[c][1] = Mfma16<T>::run(od, pf[part], acc[c][1]);
            }
        }
        __builtin_amdgcn_wave_barrier();
    };

    // two register sets, named so that the wait for one never covers the other; the load of the next tile
    // is issued unconditionally (after the last tile: that tile once more) to keep the loop free of branches
    // around loads
    Chunk kA[2][KB], vA[NP], kB[2][KB], vB[NP];
    uint2 sA[4], sB[4];
    const int tstep = kStreamWaves * kStreamTile;
    // The wave's tiles are k0 + 32 wave + 128 n, n < nt.  The workgroups of different sequences start their walk at
    // different n and wrap around, the kv heads of one sequence stay in step.  Measured over the batch-32 decode step
    // at context 2048 with a paged cache (pages of 256 rows, a sequence's heads 64 KB apart inside a page): every
    // workgroup from n = 0: 53 us per launch; starts one tile apart per sequence: 49 us; one tile apart per
    // workgroup (heads out of step as well): 60 us; a contiguous cache is indifferent to all three (50 us).  The
    // order of the tiles changes nothing but the rounding of the online softmax, and it is a fixed function of the
    // grid.
    const int nt = (k1 - k0 - wave * kStreamTile + tstep - 1) / tstep;  // (kOneTile: one, or none or fewer)
    NewRow fresh;
    if constexpr (FUSE) {
        if (new_mine) request(fresh);
        if (nt <= 0 && new_mine) append(fresh);
    }
    if (nt > 0) {
        const int rot = (int)((unsigned)(b + split) % (unsigned)nt);
        auto tile_at = [&](int n) {
            n = min(n, nt - 1) + rot;
            if (n >= nt) n -= nt;
            return k0 + wave * kStreamTile + n * tstep;
        };
        int n = 0;
        load_tile(tile_at(0), kA, vA, sA);
        if constexpr (FUSE) {
            // rotate the queries: dims d and d + D/2 of a pair are blocks j and j + KB/2 of the same lane
#pragma unroll
            for (int j = 0; j < KB / 2; j++) {
                float xl[8], xh[8], cl[8], ch[8], sl[8], sh[8], ol[8], oh[8];
                widen8<T>(qf[j], xl);
                widen8<T>(qf[j + KB / 2], xh);
                widen8<T>(cs[0][j], cl);
                widen8<T>(cs[0][j + KB / 2], ch);
                widen8<T>(cs[1][j], sl);
                widen8<T>(cs[1][j + KB / 2], sh);
#pragma unroll
                for (int i = 0; i < 8; i++) {
                    ol[i] = xl[i] * cl[i] - xh[i] * sl[i];
                    oh[i] = xh[i] * ch[i] + xl[i] * sh[i];
                }
                qf[j] = U4{pack2<T>(ol[0], ol[1]), pack2<T>(ol[2], ol[3]), pack2<T>(ol[4], ol[5]), pack2<T>(ol[6], ol[7])};
                qf[j + KB / 2] = U4{pack2<T>(oh[0], oh[1]), pack2<T>(oh[2], oh[3]), pack2<T>(oh[4], oh[5]), pack2<T>(oh[6], oh[7])};
            }
            if (new_mine) append(fresh);
            __builtin_amdgcn_wave_barrier();
        }
        if constexpr (FORM == kOneTile) process(tile_at(0), kA, vA, sA);
        else while (true) {
            load_tile(tile_at(n + 1), kB, vB, sB);
            process(tile_at(n), kA, vA, sA);
            if (++n >= nt) break;
            load_tile(tile_at(n + 1), kA, vA, sA);
            process(tile_at(n), kB, vB, sB);
            if (++n >= nt) break;
        }
    }

    // ---- this wave's results to LDS: l over the 4 quads of a head; lane (head col, quad) holds the
    // dims 32c + 2*(4*quad + e) + par of O^T
    l_run += __shfl_xor(l_run, 16, 64);
    l_run += __shfl_xor(l_run, 32, 64);
    if (lane < G) {
        m_s[wave][lane] = m_run;
        l_s[wave][lane] = l_run;
    }
    if (col < G) {
#pragma unroll
        for (int c = 0; c < KB; c++)
#pragma unroll
            for (int par = 0; par < 2; par++)
#pragma unroll
                for (int e = 0; e < 4; e++) o_s(wave)[col][c * 32 + 2 * (4 * quad + e) + par] = acc[c][par][e] * (UNITS ? unit * (1.0f / kPScale) : 1.0f / kPScale);
    }
    __syncthreads();

    // ---- combine the waves (a wave with no tile has m = -inf, l = 0, o = 0), two dims per thread
    T *out = (T *)p.out;
    for (int idx = tid; idx < G * D / 2; idx += kStreamThreads) {
        const int g = idx / (D / 2), d = idx % (D / 2) * 2;
        float mt = -INFINITY;
#pragma unroll
        for (int w = 0; w < kStreamWaves; w++) mt = fmaxf(mt, m_s[w][g]);
        float lt = 0.f, o0 = 0.f, o1 = 0.f;
#pragma unroll
        for (int w = 0; w < kStreamWaves; w++) {
            const float c = m_s[w][g] == -INFINITY ? 0.f : fast_exp(m_s[w][g] - mt);
            lt = fmaf(l_s[w][g], c, lt);
            o0 = fmaf(o_s(w)[g][d], c, o0);
            o1 = fmaf(o_s(w)[g][d + 1], c, o1);
        }
        const size_t row = (size_t)(b * p.Hq + head0 + g), at = (size_t)b * p.o_bs + (size_t)(head0 + g) * p.o_hs + d;
        if (n_act == 1) {
            Elem<T>::st(out, at, o0 / lt);
            Elem<T>::st(out, at + 1, o1 / lt);
        } else if (p.arrive) {
            // (past this XCD's L2: whoever arrives last reads them)
            auto word = [](float lo, float hi) { return (uint64_t)__builtin_bit_cast(uint32_t, lo) | ((uint64_t)__builtin_bit_cast(uint32_t, hi) << 32); };
            __hip_atomic_store((uint64_t *)(p.part_o + (row * p.nsplit + split) * D + d), word(o0, o1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if (d == 0) __hip_atomic_store((uint64_t *)(p.part_ml + (row * p.nsplit + split) * 2), word(mt, lt), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        } else {
            // merged by attn_merge_kernel in the next launch
            float *po = p.part_o + (row * p.nsplit + split) * D + d;
            po[0] = o0;
            po[1] = o1;
            if (d == 0) {
                p.part_ml[(row * p.nsplit + split) * 2] = mt;
                p.part_ml[(row * p.nsplit + split) * 2 + 1] = lt;
            }
        }
    }
    if (n_act == 1 || !p.arrive) return;

    // ---- the last key range to arrive merges them, in their order (the result does not depend on who was last)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // this range's results are written through before it counts itself in
    __syncthreads();
    int *flag = (int *)&p_s[0][0];
    if (tid == 0) {
        const int before = __hip_atomic_fetch_add(p.arrive + bhkv, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (before == n_act - 1) __hip_atomic_store(p.arrive + bhkv, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);  // ready for the next launch
        *flag = before;
    }
    __syncthreads();
    if (*flag != n_act - 1) return;
    auto merge = [&](auto ahead, auto all) {
        constexpr int AH = decltype(ahead)::value;      // ranges whose loads are in flight together
        constexpr bool ALL = decltype(all)::value;      // ... which are all of them: one wait for memory instead of two
        for (int idx = tid; idx < G * D / 2; idx += kStreamThreads) {
            const int g = idx / (D / 2), d = idx % (D / 2) * 2;
            const size_t row = (size_t)(b * p.Hq + head0 + g);
            const uint64_t *ml = (const uint64_t *)(p.part_ml + row * p.nsplit * 2), *po = (const uint64_t *)(p.part_o + row * p.nsplit * D + d);
            auto lo = [](uint64_t w) { return __builtin_bit_cast(float, (uint32_t)w); };
            auto hi = [](uint64_t w) { return __builtin_bit_cast(float, (uint32_t)(w >> 32)); };
            uint64_t w[AH], o[AH];
            auto fetch = [&](int s0, bool values) {
#pragma unroll
                for (int i = 0; i < AH; i++) {
                    const int sp = min(s0 + i, n_act - 1);
                    w[i] = __hip_atomic_load(ml + sp, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    if (values) o[i] = __hip_atomic_load(po + (size_t)sp * (D / 2), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
            };
            // the maximum of all ranges first, as attn_merge_kernel has it
            float mt = -INFINITY;
            for (int s0 = 0; s0 < (ALL ? 1 : n_act); s0 += AH) {
                fetch(s0, ALL);
#pragma unroll
                for (int i = 0; i < AH; i++) mt = fmaxf(mt, lo(w[i]));
            }
            float lt = 0.f, o0 = 0.f, o1 = 0.f;
            for (int s0 = 0; s0 < (ALL ? 1 : n_act); s0 += AH) {
                if constexpr (!ALL) fetch(s0, true);
#pragma unroll
                for (int i = 0; i < AH; i++) {
                    const float ms = lo(w[i]);
                    const float c = ms == -INFINITY || s0 + i >= n_act ? 0.f : fast_exp(ms - mt);
                    lt = fmaf(hi(w[i]), c, lt);
                    o0 = fmaf(lo(o[i]), c, o0);
                    o1 = fmaf(hi(o[i]), c, o1);
                }
            }
            const size_t at = (size_t)b * p.o_bs + (size_t)(head0 + g) * p.o_hs + d;
            Elem<T>::st(out, at, o0 / lt);
            Elem<T>::st(out, at + 1, o1 / lt);
        }
    };
    if (n_act <= 8) merge(std::integral_constant<int, 8>{}, std::true_type{});
    else if (n_act <= 16) merge(std::integral_constant<int, 16>{}, std::true_type{});
    else merge(std::integral_constant<int, 8>{}, std::false_type{});
}

// Waves of a workgroup, four or eight, from its key range: attn_stream_plan makes ranges of 256 rows where eight are wanted, one or five
// and more of them.  Where the pairs of (sequence, kv head) ask for 256 rows anyway, eight waves with a tile each are as fast as four
// with two or faster (us, four / eight: D = 64, 32 pairs x 1500 keys, int8 cache 8.3 / 7.9; D = 128, 36 x 1500 11.7 / 10.9, 40 x 1100 11.1 / 10.4).
inline bool stream_eight_waves(int slice, int nsplit) { return slice == 256 && (nsplit == 1 || nsplit >= 5); }

// Whether 16-bit value rows are read as not wanted again (four waves only: eight have little to read).  In an executor's step (the
// length in device memory) the other layers' caches and weights pass before the same rows are read again; an operator's caches
// may still be in the Infinity Cache, 256 MB, from the call before unless they are larger than it.  Us per launch without /
// with, D = 128, 8 kv heads: operator, 17 sequences x 1056 keys (74 MB) 14.7 / 16.2, 24 x 2000 29.9 / 31.0, 32 x 2000 (262 MB) 41.5 /
// 42.0, 32 x 3000 (393 MB) 68.8 / 57.9, 64 x 3000 133.5 / 122.7; step of an 8-layer executor, 16 x 1000 804 / 790, 32 x 1000 930 / 916,
// 64 x 3000 2020 / 1915; launch of 32 x 2048 in a 32-layer step, paged, 47.6 / 43.9.  (int8 caches, 32 x 3000: no difference.)
inline bool stream_once(const StreamParams &p, int B, size_t row_bytes) {
    return p.d_active || 2 * (size_t)B * p.Hkv * min(p.active, p.cache_len) * row_bytes > (320u << 20);
}

// by type, a translation unit each
template <typename T> int attn_stream_go(const StreamParams &p, int B, int D, int kv_int8, bool fuse, hipStream_t s);

}  // namespace mynn
