// What the router's forward kernel leaves in its workspace, shared with the sparse-map kernels that consume it, and the
// router's backward as the layer calls it.
#pragma once

#include <stddef.h>
#include <stdint.h>

namespace fm {

// Sums over all tokens, per routed expert and in total.
struct RouterStats {
    static __host__ __device__ int probability_sum(int e) { return e; }
    static __host__ __device__ int count(int experts, int e) { return experts + e; }
    static __host__ __device__ int z_sum(int experts) { return 2 * experts; }
    static __host__ __device__ int size(int experts) { return 2 * experts + 1; }
};

// One workgroup per CU at most: what a workgroup counts is read by every workgroup of the sparse map, so a finer cut
// costs there what it gains here.
constexpr int kMaxRouterBlocks = 256;
constexpr int kRouterTokensPerBlock = 16;

// Workgroups of the router's forward kernel; workgroup b handles the tokens
// [b * router_tokens_per_block, (b + 1) * router_tokens_per_block).
inline int router_blocks(int64_t tokens) {
    const int64_t blocks = (tokens + kRouterTokensPerBlock - 1) / kRouterTokensPerBlock;
    return static_cast<int>(blocks < kMaxRouterBlocks ? blocks : kMaxRouterBlocks);
}
inline int64_t router_tokens_per_block(int64_t tokens) {
    const int blocks = router_blocks(tokens);
    return blocks > 0 ? (tokens + blocks - 1) / blocks : 0;
}
// The workspace starts with int32 counts [workgroup][expert, the shared ones after the routed ones].
inline size_t router_counts_bytes(int64_t tokens, int64_t experts) {
    return sizeof(int32_t) * static_cast<size_t>(router_blocks(tokens)) * static_cast<size_t>(experts);
}

// `fm_router_backward`. With `round_grad_scores` the gradients of the scores are rounded to `dtype` first: the type in which
// the combine's backward hands them over where the layer runs one call after the other.
int router_backward(const void *grad_scores, const void *scores, const void *top_experts, const void *logits, const void *noise,
                    const void *lse, const void *statistics, void *grad_logits, double auxiliary_loss_grad, double z_loss_grad,
                    int64_t num_tokens, int64_t num_experts, int64_t experts_per_token, int64_t shared_experts, int dtype,
                    bool round_grad_scores, void *stream);

// `fm_router_linear_backward`. With `round_product` (half precision, up to 128 experts) what is added to grad_input is rounded to
// `dtype` first: the two gradients of the layer's input as autograd adds them where the layer runs one call after the other.
int router_linear_backward(const void *grad_logits, const void *input, const void *weight, void *grad_input, void *grad_weight,
                           bool round_product, int64_t num_tokens, int64_t num_experts, int64_t hidden, int dtype, void *workspace,
                           size_t workspace_size, void *stream);

}  // namespace fm
