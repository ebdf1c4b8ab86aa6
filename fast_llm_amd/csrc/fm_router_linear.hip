// Backward of the router's linear layer, logits [tokens, experts] = input [tokens, hidden] x weight^T:
//   grad_weight [experts, hidden] = grad_logits^T x input     and     grad_input += grad_logits x weight.
//
// The weight gradient reduces over the tokens into a result of at most a few hundred KiB: one column of tiles. It runs as a
// row-sparse grouped product whose groups are pieces of the token axis, enough of them for a tile per CU, into fp32 partial
// results that a small kernel adds in their order. 16384 tokens of 2048 and 128 experts: 28 us with the addition; the device
// library's product of these operands takes 134 to 180.
// The input gradient is a grouped product without groups.
#include "fm_gemm_common.h"

namespace fm {

namespace router_linear {

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;

template <typename T>
__global__ __launch_bounds__(256) void router_add_pieces_kernel(const float *__restrict__ pieces, T *__restrict__ out, int count,
                                                               int64_t size) {
    const int64_t at = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) * 4;
    if (at >= size) return;
    f32x4_t sum{0.f, 0.f, 0.f, 0.f};
    constexpr int kBatch = 8;  // requested together
    for (int p0 = 0; p0 < count; p0 += kBatch) {
        f32x4_t piece[kBatch];
#pragma unroll
        for (int i = 0; i < kBatch; ++i)
            piece[i] = p0 + i < count ? *reinterpret_cast<const f32x4_t *>(pieces + (p0 + i) * size + at) : f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < kBatch; ++i) sum += piece[i];
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) out[at + c] = from_float<T>(sum[c]);
}

struct Pieces {
    int count;
    int64_t tokens;  // each
};

// A tile of 256 per CU, or eight of 32, in pieces of whole slices (64 tokens) and at least two of them.
static Pieces plan_pieces(int64_t tokens, int64_t experts, int64_t hidden, int dtype) {
    const int64_t tile = dtype == FM_DTYPE_F32 ? 32 : 256, shortest = 128;
    const int64_t tiles = (hidden + tile - 1) / tile * ((experts + tile - 1) / tile);
    const int64_t target = dtype == FM_DTYPE_F32 ? 2048 : 256;
    const int64_t wanted = max(int64_t(1), min((target + tiles - 1) / tiles, tokens / shortest));
    const int64_t each = ((tokens + wanted - 1) / wanted + 63) / 64 * 64;
    return {static_cast<int>((tokens + each - 1) / each), each};
}

}  // namespace router_linear

}  // namespace fm

using namespace fm;

extern "C" size_t fm_router_linear_backward_workspace_size(int64_t num_tokens, int64_t num_experts, int64_t hidden, int dtype) {
    if (!valid_dtype(dtype) || num_tokens <= 0 || num_experts <= 0 || hidden <= 0) return 0;
    const int vector = 16 / dtype_size(dtype);
    if (num_experts % vector != 0 || hidden % vector != 0 || num_experts > 4096 || hidden >= (1 << 20)) return 0;
    return sizeof(float) * router_linear::plan_pieces(num_tokens, num_experts, hidden, dtype).count * num_experts * hidden;
}

extern "C" int fm_router_linear_backward(const void *grad_logits, const void *input, const void *weight, void *grad_input,
                                         void *grad_weight, int64_t num_tokens, int64_t num_experts, int64_t hidden, int dtype,
                                         void *workspace, size_t workspace_size, void *stream_) {
    const char *name = "fm_router_linear_backward";
    const size_t needed = fm_router_linear_backward_workspace_size(num_tokens, num_experts, hidden, dtype);
    if (needed == 0)
        return fail(FM_ERR_UNSUPPORTED, "%s: experts and hidden must be multiples of 16 bytes, got %lld and %lld", name,
                    static_cast<long long>(num_experts), static_cast<long long>(hidden));
    FM_REQUIRE(grad_logits && aligned16(grad_logits), "%s: null or misaligned grad_logits", name);
    if (grad_weight) {
        FM_REQUIRE(input && aligned16(input) && workspace && aligned16(workspace) && workspace_size >= needed,
                   "%s: null or misaligned tensor, or a workspace of less than %zu bytes", name, needed);
        hipStream_t stream = static_cast<hipStream_t>(stream_);
        const router_linear::Pieces pieces = router_linear::plan_pieces(num_tokens, num_experts, hidden, dtype);
        GemmArgs args{grad_logits, input, workspace, nullptr, nullptr, 1, num_experts, hidden, 1, hidden, 1,
                      num_experts * pieces.count, hidden, num_tokens, num_experts, pieces.count, kInputRowSparse, 0, FM_INDEX_I32,
                      FM_DTYPE_F32};
        args.piece_length = pieces.tokens;
        if (int status = dtype == FM_DTYPE_F32 ? f32_gemm_launch(args, stream) : mfma_gemm_launch(args, dtype, nullptr, 0, stream))
            return status;
        const int64_t size = num_experts * hidden;
        FM_DISPATCH_DTYPE(dtype, T, {
            router_linear::router_add_pieces_kernel<T><<<static_cast<uint32_t>((size / 4 + 255) / 256), 256, 0, stream>>>(
                static_cast<const float *>(workspace), static_cast<T *>(grad_weight), pieces.count, size);
        });
        if (int status = check_launch(name)) return status;
    }
    if (grad_input == nullptr) return FM_OK;
    FM_REQUIRE(weight && aligned16(weight) && aligned16(grad_input), "%s: null or misaligned tensor", name);
    return fm_output_sparse_matmul(grad_logits, weight, grad_input, nullptr, num_tokens, hidden, num_experts, 1, num_experts, 1, hidden, 1,
                                   hidden, 1, 1, dtype, dtype, FM_INDEX_I32, nullptr, 0, stream_);
}
