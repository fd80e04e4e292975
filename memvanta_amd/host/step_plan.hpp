// step_plan.hpp -- how many tokens a prefill step's buffers are made for.
#pragma once
#include <algorithm>
#include <cstddef>

namespace memvanta {
namespace hip {

// Whether consecutive chunks of `batch` tokens may share a step at all: in the
// fp32 numerics the last batch % 8 tokens of a chunk have arithmetic of their
// own, in the Q8 numerics a chunk of one has.
inline bool batch_joins(std::size_t batch, bool q8) { return q8 ? batch >= 2 : batch && batch % 8 == 0; }

// Tokens of a step of a model whose chunks have at most max_batch: as many as
// `joined` where some chunk size joins, fewer (down to 32) where the attention
// scores of a step, one float per token, head and position, would pass 512 MB.
// Never fewer than max_batch, whatever its scores take.
inline std::size_t step_tokens(std::size_t max_batch, std::size_t joined, std::size_t n_ctx, std::size_t n_head,
                               bool q8) {
    if (max_batch < (q8 ? 2u : 8u)) return max_batch;
    std::size_t s = std::min(joined, n_ctx);
    while (s > 32 && s * n_head * n_ctx * 4 > (std::size_t{512} << 20)) s /= 2;
    return std::max(max_batch, s);
}

// The largest step that alloc(tokens) finds room for: `step`, else halves of
// it, at last max_batch.  0: none.
template <typename Alloc>
std::size_t fit_step(std::size_t step, std::size_t max_batch, Alloc&& alloc) {
    for (;; step = std::max(max_batch, step / 2)) {
        if (alloc(step)) return step;
        if (step <= max_batch) return 0;
    }
}

}  // namespace hip
}  // namespace memvanta
