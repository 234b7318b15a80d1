// Which tile of tile_gemm_kernel (tile_gemm.h) a product takes, and over how many K ranges.
#include <algorithm>

#include "tile_gemm.h"

namespace mynn {

// ---- which tile, and over how many K ranges.
// The time of a launch, in microseconds, fitted per tile to measured times (every tile at 1 .. 16 ranges):
//
//   t = launch + steps per range * (a * rounds + b * workgroups on the fullest CU) + g * further workgroups + e * ranges
//       + partial sums at 4 TB/s
//
// a: what a step costs a CU however few workgroups it holds (latency); b: what each resident workgroup adds (LDS, MFMA and
// dequantisation work); rounds: how often a CU takes a new set of workgroups; g: what every workgroup on the fullest CU but
// the first adds outside its steps (ramp and store).  Never less than the weights' bytes at 4.6 TB/s or the tiles'
// operations at the rate the tile keeps up in long launches (padding included).  The constants are those that choose best, not
// those that predict best (some tiles have a `g` that only says that they are never taken for more than one workgroup per CU).
// How well (profiles/tile_gemm_plans.csv: matrices of the benchmark's models and as many others, tests/test_tile_plans.py): from 16 rows
// on 0.6 % above the best of all tiles and ranges on average over 660 shapes of each type, 6 % at the 97th percentile, one in 660 more
// than 15 % (16 and 24 rows of 15871 x 8096, bf16, where two plans meet the line of the weights' bytes, by 20 %).  Fewer than 16 rows 2.1
// and 2.8 %: launches alone; each further range of a call also costs its host path, so there the older constants stay.  int8 2.3 %, one
// in 25 more than 15 %: two tables, below and from 256 rows on, fitted to the models' matrices with an earlier form of the loop.  (Two
// columns where the conversion of the weights costs differ: it is 14 vector operations per 8 fp16 weights, 20 per 8 bf16 weights.)
// Of the tiles of fewer than 96 rows, 64 x 128 is the best at 1 in 10 shapes, by up to 13 % (fp16, 97 x 5476 x 7456 33.6 us without it, 29.6
// with; 255 x 4096 x 4096 22.9 / 19.7; 33 x 14336 x 4096 22.9 / 19.3), 64 x 64 where 32 x 128 and 64 x 128 leave CUs without a workgroup and
// there is too little K for ranges (300 x 2048 x 2048 12.7 / 11.8).
struct TgCost {
    int bm, bn, per_cu;  // rows and columns of the tile, workgroups a CU holds
    float launch[2], a[2], b[2], e[2], g[2], rate[2];  // [0] fp16, [1] bf16; rate: 10^9 operations per microsecond
};
// (the order of the tiles in tg_launch_w8 and tg_launch_i8)
constexpr TgCost kTgW8[] = {
    {32, 64, 3, {4.933f, 3.913f}, {0.155f, 0.274f}, {0.081f, 0.078f}, {0.215f, 0.357f}, {0.000f, 0.000f}, {0.400f, 0.673f}},
    {32, 128, 3, {4.207f, 3.940f}, {0.164f, 0.311f}, {0.128f, 0.088f}, {0.478f, 0.439f}, {0.524f, 1.596f}, {0.437f, 0.400f}},
    {64, 64, 2, {4.188f, 4.423f}, {0.140f, 0.200f}, {0.152f, 0.141f}, {0.478f, 0.479f}, {0.000f, 0.000f}, {0.458f, 0.412f}},
    {64, 128, 2, {4.556f, 4.389f}, {0.185f, 0.195f}, {0.144f, 0.208f}, {1.030f, 1.032f}, {3.900f, 2.289f}, {0.815f, 1.237f}},
    {96, 128, 2, {4.886f, 5.084f}, {0.033f, 0.239f}, {0.293f, 0.161f}, {1.153f, 1.268f}, {3.844f, 3.201f}, {0.861f, 0.805f}},
    {128, 128, 1, {5.311f, 5.250f}, {0.370f, 0.391f}, {0.095f, 0.108f}, {1.007f, 1.068f}, {9.915f, 8.787f}, {0.972f, 0.953f}},
    {160, 128, 1, {5.472f, 6.763f}, {0.398f, 0.468f}, {0.091f, 0.047f}, {2.595f, 1.541f}, {13.523f, 12.223f}, {0.973f, 0.979f}},
    {128, 256, 1, {6.476f, 5.986f}, {0.488f, 0.307f}, {0.208f, 0.444f}, {2.786f, 3.029f}, {7.963f, 6.760f}, {1.079f, 1.075f}},
    {160, 256, 1, {8.920f, 9.339f}, {0.821f, 0.251f}, {0.122f, 0.733f}, {1.187f, 0.037f}, {5.301f, 4.901f}, {1.131f, 1.162f}},
};
constexpr TgCost kTgW8S[] = {
    {32, 32, 3, {3.394f, 3.360f}, {0.190f, 0.203f}, {0.014f, 0.016f}, {0.504f, 0.503f}, {0.0f, 0.0f}, {0.90f, 0.90f}},
    {32, 64, 3, {3.231f, 3.192f}, {0.165f, 0.185f}, {0.060f, 0.061f}, {0.504f, 0.499f}, {0.0f, 0.0f}, {0.90f, 0.90f}},
    {32, 128, 3, {2.924f, 1.705f}, {0.101f, 0.134f}, {0.148f, 0.199f}, {0.744f, 0.879f}, {0.0f, 0.0f}, {0.90f, 0.90f}},
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

static const TgCost *tg_table(int kind, int M, int *n) {
    *n = kind == TG_W8S ? 3 : kind == TG_W8 ? 9 : 6;
    return kind == TG_W8S ? kTgW8S : kind == TG_W8 ? kTgW8 : M < 256 ? kTgI8Few : kTgI8;
}

bool tile_gemm_supported(int kind, int M, int N, int K) {
    return M >= 1 && N >= 1 && K >= 16 && K % (kind == TG_I8 ? 32 : 16) == 0 && (long)K * 256 * 2 < (1l << 31);
}

// seq: for a plan whose ranges one workgroup takes, which has two sets of sums in its registers
static TgPlan tg_choose(int kind, int dtype, int M, int N, int K, size_t scratch_bytes, bool seq) {
    int n_tiles;
    const TgCost *tab = tg_table(kind, M, &n_tiles);
    const int d = dtype == MYNN_BF16 ? 1 : 0;
    const int iters = (K * (kind == TG_I8 ? 1 : 2) + 127) / 128;
    const double weights_us = (double)N * K / 4.6e6;
    TgPlan best;
    best.us = 1e30;
    for (int t = 0; t < n_tiles; t++) {
        const TgCost &c = tab[t];
        if (seq && c.bm * c.bn > 128 * 128) continue;
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
static TgPlan tg_remembered(int kind, int dtype, int M, int N, int K, size_t scratch_bytes, bool seq) {
    struct Entry {
        int kind = -1, dtype, M, N, K;
        size_t scratch;
        bool seq;
        TgPlan plan;
    };
    thread_local Entry table[32];
    Entry &e = table[((unsigned)M * 31u + (unsigned)N * 17u + (unsigned)K * 7u + (unsigned)kind * 5u + (unsigned)dtype) % 32u];
    if (e.kind != kind || e.dtype != dtype || e.M != M || e.N != N || e.K != K || e.scratch != scratch_bytes || e.seq != seq)
        e = Entry{kind, dtype, M, N, K, scratch_bytes, seq, tg_choose(kind, dtype, M, N, K, scratch_bytes, seq)};
    return e.plan;
}

TgPlan tile_gemm_plan(int kind, int dtype, int M, int N, int K, size_t scratch_bytes) {
    return tg_remembered(kind, dtype, M, N, K, scratch_bytes, false);
}

TgPlan tile_gemm_plan_seq(int kind, int dtype, int M, int N, int K, int ks) {
    const bool i8 = kind == TG_I8;  // (int32 sums are the same in any order: one range)
    TgPlan plan = tg_remembered(kind, dtype, M, N, K, 0, !i8);
    plan.ks = i8 ? 1 : ks;
    plan.seq = plan.ks > 1;
    return plan;
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
        if (kind == TG_I8) return tg_launch_i8<T>(plan.tile, p, epi);
        if constexpr (sizeof(T) == 2) return tg_launch_w8<T>(kind, plan.tile, p, epi);
        return (int)MYNN_ERR_UNSUPPORTED;  // (f32: refused above)
    });
}

}  // namespace mynn

// For the tests, and for measuring what the constants above are fitted to; not part of the library's interface.
// plan[6] = tile, its rows and columns, K ranges, whether one workgroup takes them one after the other, bytes of partial sums.
// seq_ks > 0: the plan without scratch memory for the sums of seq_ks ranges
extern "C" int mynn_tile_gemm_plan(int kind, int dtype, int M, int N, int K, size_t scratch_bytes, int seq_ks, long *plan, double *us) {
    using namespace mynn;
    MYNN_REQUIRE(plan && kind >= TG_W8 && kind <= TG_I8 && tile_gemm_supported(kind, M, N, K), MYNN_ERR_UNSUPPORTED, "tile_gemm_plan: kind %d, M=%d N=%d K=%d", kind, M, N, K);
    const TgPlan p = seq_ks > 0 ? tile_gemm_plan_seq(kind, dtype, M, N, K, seq_ks) : tile_gemm_plan(kind, dtype, M, N, K, scratch_bytes);
    int n;
    const TgCost &c = tg_table(kind, M, &n)[p.tile];
    const long v[6] = {p.tile, c.bm, c.bn, p.ks, p.seq, (long)p.part_bytes};
    for (int i = 0; i < 6; i++) plan[i] = v[i];
    if (us) *us = p.us;
    return MYNN_OK;
}
// a product by the tile and the ranges given; part, counters (zero): for ranges that workgroups take side by side
extern "C" int mynn_tile_gemm(int kind, int tile, int ks, int seq, void *out, int32_t *acc_out, const void *act, const int8_t *wq, const void *a_scale, const void *w_scale,
                              const void *res, int M, int N, int K, int dtype, int epi, void *part, size_t part_bytes, int *counters, mynn_stream s) {
    using namespace mynn;
    MYNN_REQUIRE(kind >= TG_W8 && kind <= TG_I8 && tile_gemm_supported(kind, M, N, K), MYNN_ERR_UNSUPPORTED, "tile_gemm: kind %d, M=%d N=%d K=%d", kind, M, N, K);
    int n;
    const TgCost *tab = tg_table(kind, M, &n);
    MYNN_REQUIRE(tile >= 0 && tile < n, MYNN_ERR_INVALID, "tile_gemm: tile %d of %d", tile, n);
    const long tiles = (long)((M + tab[tile].bm - 1) / tab[tile].bm) * ((N + tab[tile].bn - 1) / tab[tile].bn);
    const int iters = (K * (kind == TG_I8 ? 1 : 2) + 127) / 128;
    MYNN_REQUIRE(ks >= 1 && ks <= iters && (ks == 1 || seq || (tiles <= kTgCounters && part_bytes >= (size_t)tiles * ks * tab[tile].bm * tab[tile].bn * 4)),
                 MYNN_ERR_INVALID, "tile_gemm: %d K ranges of %ld tiles", ks, tiles);
    TgPlan p;
    p.tile = tile;
    p.ks = ks;
    p.seq = seq != 0 && ks > 1;
    return tile_gemm(kind, p, out, acc_out, act, wq, a_scale, w_scale, res, M, N, K, dtype, epi, part, counters, as_stream(s));
}
