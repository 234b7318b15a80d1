// tile_gemm_kernel for bf16 activations and int8 weights.
#include "tile_gemm_w8.h"

namespace mynn {

template int tg_launch_w8<bf16_t>(int, int, const TgArgs &, int);

}  // namespace mynn
