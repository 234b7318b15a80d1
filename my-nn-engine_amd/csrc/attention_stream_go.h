// Launches of attn_stream_kernel: every form for one type.
#pragma once
#include "attention_stream.h"

namespace mynn {

template <typename T, int D, int G, bool KVI8, bool PAGED, bool FUSE, int W, int FORM> static int stream_go(const StreamParams &p, int B, hipStream_t s) {
    constexpr int lds = StreamLds<T, D, W>::BYTES;
    static bool lds_set = false;
    if (!lds_set && lds > 64 * 1024) {
        MYNN_HIP(hipFuncSetAttribute((const void *)attn_stream_kernel<T, D, G, KVI8, PAGED, FUSE, W, FORM>, hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        lds_set = true;
    }
    MYNN_LAUNCH((attn_stream_kernel<T, D, G, KVI8, PAGED, FUSE, W, FORM>), dim3(B * p.Hkv, p.nsplit), dim3(W * 64), lds, s, p.q, p.k, p.v, p.d_active, p.d_past, p.d_pos, p.Hkv, p.slice, (const StreamRest &)p);
    return launch_status("attn_stream_kernel");
}
template <typename T, int D, int G, bool KVI8, bool PAGED, bool FUSE> static int stream_w(const StreamParams &p, int B, hipStream_t s) {
    // (eight waves: ranges of 256 keys)
    if (stream_eight_waves(p.slice, p.nsplit)) return stream_go<T, D, G, KVI8, PAGED, FUSE, 8, kOneTile>(p, B, s);
    if (p.slice == 4 * kStreamTile) return stream_go<T, D, G, KVI8, PAGED, FUSE, 4, kOneTile>(p, B, s);
    if constexpr (KVI8) {
        return stream_go<T, D, G, KVI8, PAGED, FUSE, 4, kTiles>(p, B, s);
    } else if constexpr (FUSE) {  // (executors only)
        return stream_go<T, D, G, KVI8, PAGED, FUSE, 4, kTilesOnce>(p, B, s);
    } else {
        if (stream_once(p, B, D * sizeof(T))) return stream_go<T, D, G, KVI8, PAGED, FUSE, 4, kTilesOnce>(p, B, s);
        return stream_go<T, D, G, KVI8, PAGED, FUSE, 4, kTiles>(p, B, s);
    }
}
template <typename T, int D, bool KVI8, bool PAGED, bool FUSE>
static int stream_g(const StreamParams &p, int B, hipStream_t s) {
    switch (p.Hq / p.Hkv) {
    case 1: return stream_w<T, D, 1, KVI8, PAGED, FUSE>(p, B, s);
    case 2: return stream_w<T, D, 2, KVI8, PAGED, FUSE>(p, B, s);
    case 4: return stream_w<T, D, 4, KVI8, PAGED, FUSE>(p, B, s);
    case 8: return stream_w<T, D, 8, KVI8, PAGED, FUSE>(p, B, s);
    default: return fail(MYNN_ERR_UNSUPPORTED, "streaming attention: %d query heads per kv head", p.Hq / p.Hkv);
    }
}

template <typename T, int D, bool FUSE>
static int stream_kv(const StreamParams &p, int B, int kv_int8, hipStream_t s) {
    if (p.page_table) return kv_int8 ? stream_g<T, D, true, true, FUSE>(p, B, s) : stream_g<T, D, false, true, FUSE>(p, B, s);
    return kv_int8 ? stream_g<T, D, true, false, FUSE>(p, B, s) : stream_g<T, D, false, false, FUSE>(p, B, s);
}
template <typename T> int attn_stream_go(const StreamParams &p, int B, int D, int kv_int8, bool fuse, hipStream_t s) {
    if (fuse) return D == 64 ? stream_kv<T, 64, true>(p, B, kv_int8, s) : stream_kv<T, 128, true>(p, B, kv_int8, s);
    return D == 64 ? stream_kv<T, 64, false>(p, B, kv_int8, s) : stream_kv<T, 128, false>(p, B, kv_int8, s);
}

}  // namespace mynn
