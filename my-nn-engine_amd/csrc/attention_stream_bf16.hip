// attn_stream_kernel for bf16.
#include "attention_stream_go.h"

namespace mynn {

template int attn_stream_go<bf16_t>(const StreamParams &, int, int, int, bool, hipStream_t);

}  // namespace mynn
