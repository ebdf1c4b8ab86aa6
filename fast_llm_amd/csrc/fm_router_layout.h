// What the router's forward kernel leaves in its workspace, shared with the sparse-map kernels that consume it, and the
// router's backward as the layer calls it.
#pragma once

#include <hip/hip_runtime.h>
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

// What is left to do for the losses when the forward kernel has run: the sums over its workgroups.
struct RouterFinish {
    const int32_t *block_counts;  // as above
    const float *block_sums;      // [workgroup][expert, the z-loss after them]
    float *statistics, *losses;
    int blocks, experts, shared;
    int64_t tokens;
};
// The launch with the sums is the caller's if `finish` is false.
int router_forward(const void *logits, const void *noise, void *top_experts, void *scores, void *lse, void *statistics, void *losses,
                   void *workspace, size_t workspace_size, int64_t num_tokens, int64_t num_experts, int64_t experts_per_token,
                   int64_t shared_experts, int dtype, bool finish, void *stream);
RouterFinish router_finish_of(const void *workspace, void *statistics, void *losses, int64_t num_tokens, int64_t num_experts,
                              int64_t shared_experts);
// `fm_sparse_map_from_router`, with the router's sums in the same launch if `finish` is not null.
int sparse_map_from_router(const int64_t *top_experts, const void *router_workspace, size_t router_workspace_size,
                           int64_t num_tokens, int64_t num_experts, int64_t experts_per_token, int64_t shared_experts,
                           int64_t pad_to_multiple, int index_dtype, void *sparse_rows, void *expert_ends, void *expert_pad_begins,
                           void *workspace, size_t workspace_size, const RouterFinish *finish, void *stream);

// statistics = the sums over the workgroups of the forward kernel (softmax sums and z-loss sum as doubles: up to 256
// terms of similar size), losses[0] = load-balancing loss, losses[1] = z-loss. One workgroup of kFinishThreads: its threads are
// parts x columns (a power of two of them), so that all terms are requested at once whatever the number of experts. (16 threads per
// column, 64 columns at a time: 18 us at 128 experts and 256 workgroups; one thread per column that walked down 1024 workgroups 261.)
constexpr int kFinishThreads = 1024, kFinishWaves = kFinishThreads / 64;
struct FinishLds {
    double sums[kFinishThreads];
    double balances[kFinishWaves], z_sums[kFinishWaves];
    int32_t counts[kFinishThreads];
};

__device__ inline void finish_router(const RouterFinish &finish, FinishLds &lds) {
    constexpr int kBatch = 16;
    const int experts = finish.experts, blocks = finish.blocks, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    int columns = 8;
    while (columns < experts && columns < kFinishThreads) columns *= 2;
    const int column = threadIdx.x & (columns - 1), part = threadIdx.x / columns, parts = kFinishThreads / columns;
    const int per_part = (blocks + parts - 1) / parts;
    // A wavefront holds several parts of few columns; then `rows` sums per column are left, one per wavefront or part.
    const int rows = columns < 64 ? kFinishWaves : parts, row = columns < 64 ? wave : part;
    double z_sum = 0.0, balance = 0.0;
    for (int b = threadIdx.x; b < blocks; b += kFinishThreads) z_sum += finish.block_sums[static_cast<int64_t>(b) * (experts + 1) + experts];
    for (int base = 0; base < experts; base += columns) {
        const int c = base + column;
        double sum = 0.0;
        int32_t count = 0;
        for (int i0 = 0; i0 < per_part; i0 += kBatch) {
            float sums[kBatch];
            int32_t counts[kBatch];
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                const int b = part * per_part + i0 + i;
                const bool exists = i0 + i < per_part && b < blocks && c < experts;
                sums[i] = exists ? finish.block_sums[static_cast<int64_t>(b) * (experts + 1) + c] : 0.f;
                counts[i] = exists ? finish.block_counts[static_cast<int64_t>(b) * (experts + finish.shared) + c] : 0;
            }
#pragma unroll
            for (int i = 0; i < kBatch; ++i) sum += sums[i], count += counts[i];
        }
        for (int offset = columns; offset < 64; offset *= 2) {
            sum += __shfl_xor(sum, offset, 64);
            count += __shfl_xor(count, offset, 64);
        }
        if (columns >= 64 || lane < columns) {
            lds.sums[row * columns + column] = sum;
            lds.counts[row * columns + column] = count;
        }
        __syncthreads();
        if (static_cast<int>(threadIdx.x) < columns && c < experts) {
            sum = 0.0, count = 0;
            for (int r = 0; r < rows; ++r) sum += lds.sums[r * columns + column], count += lds.counts[r * columns + column];
            finish.statistics[RouterStats::probability_sum(c)] = static_cast<float>(sum);
            finish.statistics[RouterStats::count(experts, c)] = static_cast<float>(count);
            balance += sum * count;
        }
        __syncthreads();
    }
#pragma unroll
    for (int offset = 32; offset > 0; offset >>= 1) {
        balance += __shfl_xor(balance, offset, 64);
        z_sum += __shfl_xor(z_sum, offset, 64);
    }
    if (lane == 0) lds.balances[wave] = balance, lds.z_sums[wave] = z_sum;
    __syncthreads();
    if (threadIdx.x == 0) {
        balance = z_sum = 0.0;
        for (int w = 0; w < kFinishWaves; ++w) balance += lds.balances[w], z_sum += lds.z_sums[w];
        const double tokens = static_cast<double>(finish.tokens);
        finish.statistics[RouterStats::z_sum(experts)] = static_cast<float>(z_sum);
        finish.losses[0] = static_cast<float>(balance / tokens / tokens);
        finish.losses[1] = static_cast<float>(z_sum / tokens);
    }
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
