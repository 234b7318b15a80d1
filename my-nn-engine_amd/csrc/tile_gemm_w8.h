// The tiles of products of int8 weights with 16-bit activations, in the order of kTgW8 and kTgW8S (tile_gemm.hip).
#pragma once
#include "tile_gemm.h"

namespace mynn {

template <typename T> int tg_launch_w8(int kind, int tile, const TgArgs &p, int epi) {
    if (kind == TG_W8) {
        if (tile == 0) return tg_epi<T, TgTile<TG_W8, 32, 64, 1, 2, 6, 2, 1>>(p, epi);
        if (tile == 1) return tg_epi<T, TgTile<TG_W8, 32, 128, 1, 4, 4, 2, 1>>(p, epi);
        if (tile == 2) return tg_epi<T, TgTile<TG_W8, 64, 64, 2, 2, 6, 2, 2, false>>(p, epi);
        if (tile == 3) return tg_epi<T, TgTile<TG_W8, 64, 128, 1, 4, 4, 2, 1>>(p, epi);
        if (tile == 4) return tg_epi<T, TgTile<TG_W8, 96, 128, 1, 4, 4, 1, 1>>(p, epi);
        if (tile == 5) return tg_epi<T, TgTile<TG_W8, 128, 128, 1, 4, 6, 1, 1>>(p, epi);
        if (tile == 6) return tg_epi<T, TgTile<TG_W8, 160, 128, 1, 4, 5, 1, 1>>(p, epi);
        if (tile == 7) return tg_epi<T, TgTile<TG_W8, 128, 256, 1, 4, 4, 1, 1>>(p, epi);
        return tg_epi<T, TgTile<TG_W8, 160, 256, 1, 4, 4, 1, 1>>(p, epi);
    }
    if (tile == 0) return tg_epi<T, TgTile<TG_W8S, 32, 32, 1, 1, 8, 1, 1>>(p, epi);
    if (tile == 1) return tg_epi<T, TgTile<TG_W8S, 32, 64, 1, 2, 6, 2, 1>>(p, epi);
    return tg_epi<T, TgTile<TG_W8S, 32, 128, 1, 4, 4, 2, 1>>(p, epi);
}

}  // namespace mynn
