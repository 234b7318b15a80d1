// attn_stream_kernel for fp16.
#include "attention_stream_go.h"

namespace mynn {

template int attn_stream_go<f16_t>(const StreamParams &, int, int, int, bool, hipStream_t);

}  // namespace mynn
