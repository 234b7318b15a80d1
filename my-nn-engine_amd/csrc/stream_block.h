// Scratch memory of the entry points that need some and are given none.
#pragma once
#include <map>
#include <memory>
#include <mutex>

#include "mynn_common.h"

namespace mynn {

// One block per stream, grown on demand, so that calls on different streams never share one.
//  - A lease holds the block's lock until the caller has launched everything that uses it: a second host thread on the
//    same stream can neither free the block between look-up and launch nor put its launches between two of the first's.
//  - A block handed to a call that is being captured belongs to the graph from then on, which may be replayed at any time:
//    it is kept when the stream's block grows.  Growing then at least doubles, so that all blocks kept of a stream are
//    together smaller than its present one.  (The graph's launches share the block with the stream's other calls: they
//    have to be ordered with those, as they are when it is replayed on that stream.)
//  - A block that no graph knows is freed when it grows, after the stream's work so far.
class StreamBlocks {
    struct Block {
        std::mutex mu;
        char *ptr = nullptr;
        size_t bytes = 0;
        bool in_graph = false;
    };
    std::mutex mu_;
    std::map<const void *, std::unique_ptr<Block>> blocks_;

public:
    struct Lease {
        std::unique_lock<std::mutex> held;
        char *ptr = nullptr;
    };

    // at least `need` bytes; `zeroed`: how many of the first ones are zero when the block is new; `capturing`:
    // stream_capturing(s), which callers have asked already (0.1 us)
    int lease(hipStream_t s, bool capturing, size_t need, size_t zeroed, const char *who, Lease *out) {
        Block *b;
        {
            // (this handle stands for another stream in every thread)
            static thread_local char own;
            std::lock_guard<std::mutex> lk(mu_);
            std::unique_ptr<Block> &slot = blocks_[s == hipStreamPerThread ? (const void *)&own : (const void *)s];
            if (!slot) slot.reset(new Block);
            b = slot.get();
        }
        std::unique_lock<std::mutex> held(b->mu);
        if (need > b->bytes) {
            MYNN_REQUIRE(!capturing, MYNN_ERR_STATE,
                         "%s: the library workspace cannot grow while the stream is being captured; call it once before, or pass a workspace", who);
            const size_t bytes = b->in_graph && need < 2 * b->bytes ? 2 * b->bytes : need;
            MYNN_HIP(hipStreamSynchronize(s));
            if (b->ptr && !b->in_graph) MYNN_HIP(hipFree(b->ptr));
            b->ptr = nullptr;
            b->bytes = 0;
            b->in_graph = false;
            MYNN_HIP(hipMalloc((void **)&b->ptr, bytes));
            if (zeroed) {
                const hipError_t e = hipMemsetAsync(b->ptr, 0, zeroed, s);
                if (e != hipSuccess) {
                    (void)hipFree(b->ptr);
                    b->ptr = nullptr;
                    return hip_fail(e, who);
                }
            }
            b->bytes = bytes;
        }
        b->in_graph = b->in_graph || capturing;
        out->held = std::move(held);
        out->ptr = b->ptr;
        return 0;
    }
};

}  // namespace mynn
