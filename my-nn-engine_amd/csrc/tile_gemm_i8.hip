// tile_gemm_kernel for int8 operands (QuantizedMatMul), the tiles in the order of kTgI8 (tile_gemm.hip).
#include "tile_gemm.h"

namespace mynn {

template <typename T> int tg_launch_i8(int tile, const TgArgs &p, int epi) {
    if (tile == 0) return tg_epi<T, TgTile<TG_I8, 32, 64, 1, 2, 6, 1, 1>>(p, epi);
    if (tile == 1) return tg_epi<T, TgTile<TG_I8, 64, 64, 2, 2, 6, 2, 1>>(p, epi);
    if (tile == 2) return tg_epi<T, TgTile<TG_I8, 64, 128, 2, 4, 6, 2, 2>>(p, epi);
    if (tile == 3) return tg_epi<T, TgTile<TG_I8, 64, 128, 2, 2, 3, 2, 1>>(p, epi);
    if (tile == 4) return tg_epi<T, TgTile<TG_I8, 128, 128, 2, 4, 4, 2, 1>>(p, epi);
    return tg_epi<T, TgTile<TG_I8, 128, 256, 2, 4, 3, 2, 1>>(p, epi);
}
template int tg_launch_i8<f16_t>(int, const TgArgs &, int);
template int tg_launch_i8<bf16_t>(int, const TgArgs &, int);
template int tg_launch_i8<float>(int, const TgArgs &, int);

}  // namespace mynn
