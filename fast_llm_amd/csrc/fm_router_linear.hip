// The router's linear layer, logits [tokens, experts] = input [tokens, hidden] x weight^T, for few tokens, and its backward:
//   grad_weight [experts, hidden] = grad_logits^T x input     and     grad_input += grad_logits x weight.
//
// The weight gradient reduces over the tokens into a result of at most a few hundred KiB: one column of tiles. It runs as a
// row-sparse grouped product whose groups are pieces of the token axis, enough of them for a tile per CU, into fp32 partial
// results that a small kernel adds in their order. 16384 tokens of 2048 and 128 experts: 28 us with the addition; the device
// library's product of these operands takes 134 to 180.
// The input gradient is a grouped product without groups in fp32. In half precision it reduces over at most 128 experts: the bytes
// of the gradient that it is added to are the bound, which a kernel reads and writes once (see router_input_grad_kernel).
//
// The logits of few tokens are latency and nothing else: a workgroup computes 16 tokens x 16 experts, its wavefronts a part of the
// hidden axis each, fragments straight from memory into registers, all loads of eight steps under way at once, and one exchange
// through LDS at the end (twice the wavefronts are no faster). us on the device, the device library's product in brackets: one token of
// 4096 and 8 experts 4.8 (7.4), 64 tokens 7.6 (7.6), 96 of 2048 and 128 experts 5.5 (5.4), 512 of 256 and 8 experts in single
// precision 3.3 (3.7), operands in cache; from memory 1531 of 4096 and 8 experts 13.8 (20), 3001 of 1280 and 16 9.3 (13), 700 of 2048 and
// 64 9.8 (14.7), 1999 of 2048 and 128 21.8 (16.6). Calling that library takes 19 us of the host's time, this 8. Workgroups of 2 x 4 to
// 4 x 8 tiles, which read less, lose more to the fewer of them (5001 of 2048 and 64 experts 23 to 28 us, 28 so, 18.8).
#include "fm_gemm_common.h"
#include "fm_router_layout.h"

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

// ---- logits of few tokens -------------------------------------------------------------------------------------------------
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4_t;

constexpr int kLogitTile = 16, kLogitWaves = 8;

// A lane's 16 bytes of each operand: 8 (half precision) or 4 (fp32) consecutive elements of row lane % 16, the four groups of 16
// lanes one after the other along the hidden axis. Which element of a step is multiplied when is the same for both operands.
__device__ __forceinline__ f32x4_t multiply(bf16_t, u32x4_t a, u32x4_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4_t multiply(f16_t, u32x4_t a, u32x4_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4_t multiply(float, u32x4_t a, u32x4_t b, f32x4_t c) {
    const f32x4_t a_values = __builtin_bit_cast(f32x4_t, a), b_values = __builtin_bit_cast(f32x4_t, b);
#pragma unroll
    for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(a_values[i], b_values[i], c, 0, 0, 0);
    return c;
}

template <typename T>
__global__ __launch_bounds__(64 * kLogitWaves) void router_logits_kernel(const T *__restrict__ input, const T *__restrict__ weight,
                                                                        T *__restrict__ logits, int64_t tokens, int experts, int hidden) {
    constexpr int kVector = 16 / sizeof(T), kStep = 4 * kVector, kBatch = 8;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int64_t token0 = static_cast<int64_t>(blockIdx.x) * kLogitTile;
    const int expert0 = blockIdx.y * kLogitTile;
    // Rows past the last one are the last one: they are not stored.
    const T *x = input + min(token0 + (lane & 15), tokens - 1) * hidden;
    const T *w = weight + static_cast<int64_t>(min(expert0 + (lane & 15), experts - 1)) * hidden;
    const int steps = (hidden + kStep - 1) / kStep, each = (steps + kLogitWaves - 1) / kLogitWaves;
    const int first = wave * each, last = min(first + each, steps), offset = (lane >> 4) * kVector;
    f32x4_t sum{0.f, 0.f, 0.f, 0.f};
    for (int step = first; step < last; step += kBatch) {
        u32x4_t a[kBatch], b[kBatch];
#pragma unroll
        for (int i = 0; i < kBatch; ++i) {
            const int at = (step + i) * kStep + offset;
            a[i] = b[i] = u32x4_t{0, 0, 0, 0};
            if (step + i < last && at < hidden) {  // hidden is a multiple of kVector
                a[i] = *reinterpret_cast<const u32x4_t *>(w + at);
                b[i] = *reinterpret_cast<const u32x4_t *>(x + at);
            }
        }
#pragma unroll
        for (int i = 0; i < kBatch; ++i) sum = multiply(T(), a[i], b[i], sum);
    }
    // A lane holds four consecutive experts of one token; the wavefronts' parts add up in their order.
    __shared__ f32x4_t parts[kLogitWaves][64];
    parts[wave][lane] = sum;
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int other = 1; other < kLogitWaves; ++other) sum += parts[other][lane];
    const int64_t token = token0 + (lane & 15);
    if (token >= tokens) return;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        const int expert = expert0 + (lane >> 4) * 4 + c;
        if (expert < experts) logits[token * experts + expert] = from_float<T>(sum[c]);
    }
}

// ---- input gradient ------------------------------------------------------------------------------------------------------------
// grad_input += grad_logits x weight; with kRoundProduct the product is rounded before it is added, as where autograd adds the two
// gradients of a layer's input. A workgroup has 128 columns of the weight in LDS as the MFMAs want them (kSteps x 32 experts, a step
// per wavefront; the K-rows that a lane loads are transposed in blocks of 8 x 8, one v_perm_b32 per two values), and its wavefronts
// walk kInputGradTokens tokens each, 16 at a time: a lane holds eight consecutive columns of four of them, 16 lanes 256 bytes of a
// row. us, a product and an addition of torch in brackets: 16384 tokens of 2048 and 128 experts 31 (53), 64 experts 24 (48; 5.5
// TB/s), 8192 of 4096 and 8 experts 22 (54; 6 TB/s), 1999 of 2048 and 128 experts 9 (22), 512 of 512 and 8 experts 5 (22, the
// host's time). With the columns in registers there is one wavefront per SIMD from 65 experts on: 54 us for the first of these.
constexpr int kInputGradTokens = 64, kInputGradMaxExperts = 128;

template <typename T, int kSteps, bool kRoundProduct>
__global__ __launch_bounds__(256, 4) void router_input_grad_kernel(const T *__restrict__ grad_logits, const T *__restrict__ weight,
                                                                   T *__restrict__ grad_input, int64_t tokens, int experts, int hidden) {
    static_assert(kSteps <= 4, "a step per wavefront");
    __shared__ u32x4_t columns[kSteps][8][64];  // [step][i][lane]: column i of the lane's eight, experts 32 step + 8 group + 0 .. 7
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, group = lane >> 4;
    const int column = blockIdx.x * 128 + (lane & 15) * 8;
    const bool exists = column < hidden;  // a multiple of 8
    if (wave < kSteps) {
        u32x4_t raw[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int expert = wave * 32 + group * 8 + j;
            raw[j] = u32x4_t{0, 0, 0, 0};
            if (exists && expert < experts) raw[j] = *reinterpret_cast<const u32x4_t *>(weight + static_cast<int64_t>(expert) * hidden + column);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            u32x4_t one;
#pragma unroll
            for (int p = 0; p < 4; ++p)
                one[p] = __builtin_amdgcn_perm(raw[2 * p + 1][i / 2], raw[2 * p][i / 2], i % 2 ? 0x07060302u : 0x05040100u);
            columns[wave][i][lane] = one;
        }
    }
    __syncthreads();
    const int64_t first = (static_cast<int64_t>(blockIdx.y) * 4 + wave) * kInputGradTokens;
    for (int64_t token0 = first; token0 < min(first + kInputGradTokens, tokens); token0 += 16) {
        asm volatile("" ::: "memory");  // the columns are read from LDS every time, not kept in registers
        T *target = grad_input + (token0 + group * 4) * hidden + column;
        const T *row = grad_logits + min(token0 + (lane & 15), tokens - 1) * experts + group * 8;
        u32x4_t logits[kSteps], before[4];
#pragma unroll
        for (int step = 0; step < kSteps; ++step) {
            logits[step] = u32x4_t{0, 0, 0, 0};
            if (step * 32 + group * 8 < experts) logits[step] = *reinterpret_cast<const u32x4_t *>(row + step * 32);  // a multiple of 8
        }
        const int64_t left = exists ? tokens - token0 - group * 4 : 0;  // of the lane's four tokens
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (r < left) before[r] = *reinterpret_cast<const u32x4_t *>(target + static_cast<int64_t>(r) * hidden);
        f32x4_t sums[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) sums[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int step = 0; step < kSteps; ++step)
#pragma unroll
            for (int i = 0; i < 8; ++i) sums[i] = multiply(T(), logits[step], columns[step][i][lane], sums[i]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (r >= left) continue;
            Vec16<T> value = __builtin_bit_cast(Vec16<T>, before[r]);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const float product = kRoundProduct ? to_float(from_float<T>(sums[i][r])) : sums[i][r];
                value.v[i] = from_float<T>(to_float(value.v[i]) + product);
            }
            store16(target + static_cast<int64_t>(r) * hidden, value);
        }
    }
}

template <typename T, bool kRoundProduct>
static void launch_input_grad(const void *grad_logits, const void *weight, void *grad_input, int64_t tokens, int experts, int hidden,
                              hipStream_t stream) {
    const int64_t rows = 4 * kInputGradTokens;
    const dim3 grid((hidden + 127) / 128, static_cast<uint32_t>((tokens + rows - 1) / rows));
    const auto kernel = experts <= 32   ? router_input_grad_kernel<T, 1, kRoundProduct>
                        : experts <= 64 ? router_input_grad_kernel<T, 2, kRoundProduct>
                                        : router_input_grad_kernel<T, 4, kRoundProduct>;
    kernel<<<grid, 256, 0, stream>>>(static_cast<const T *>(grad_logits), static_cast<const T *>(weight), static_cast<T *>(grad_input),
                                     tokens, experts, hidden);
}

}  // namespace router_linear

}  // namespace fm

using namespace fm;

extern "C" int fm_router_linear_forward(const void *input, const void *weight, void *logits, int64_t num_tokens, int64_t num_experts,
                                        int64_t hidden, int dtype, void *stream) {
    using namespace router_linear;
    const char *name = "fm_router_linear_forward";
    FM_REQUIRE(valid_dtype(dtype), "%s: bad dtype", name);
    FM_REQUIRE(num_tokens >= 0 && num_experts > 0 && num_experts <= 4096 && hidden > 0 && hidden < (1 << 20), "%s: bad shape", name);
    if (hidden % (16 / dtype_size(dtype)) != 0)
        return fail(FM_ERR_UNSUPPORTED, "%s: hidden must be a multiple of 16 bytes, got %lld", name, static_cast<long long>(hidden));
    if (num_tokens == 0) return FM_OK;
    FM_REQUIRE(input && weight && logits && aligned16(input) && aligned16(weight), "%s: null or misaligned tensor", name);
    const int64_t blocks = (num_tokens + kLogitTile - 1) / kLogitTile;
    if (blocks >= (int64_t(1) << 31)) return fail(FM_ERR_UNSUPPORTED, "%s: too many tokens", name);
    const dim3 grid(static_cast<uint32_t>(blocks), static_cast<uint32_t>((num_experts + kLogitTile - 1) / kLogitTile));
    FM_DISPATCH_DTYPE(dtype, T, {
        router_logits_kernel<T><<<grid, 64 * kLogitWaves, 0, static_cast<hipStream_t>(stream)>>>(
            static_cast<const T *>(input), static_cast<const T *>(weight), static_cast<T *>(logits), num_tokens,
            static_cast<int>(num_experts), static_cast<int>(hidden));
    });
    return check_launch(name);
}

extern "C" size_t fm_router_linear_backward_workspace_size(int64_t num_tokens, int64_t num_experts, int64_t hidden, int dtype) {
    if (!valid_dtype(dtype) || num_tokens <= 0 || num_experts <= 0 || hidden <= 0) return 0;
    const int vector = 16 / dtype_size(dtype);
    if (num_experts % vector != 0 || hidden % vector != 0 || num_experts > 4096 || hidden >= (1 << 20)) return 0;
    return sizeof(float) * router_linear::plan_pieces(num_tokens, num_experts, hidden, dtype).count * num_experts * hidden;
}

int fm::router_linear_backward(const void *grad_logits, const void *input, const void *weight, void *grad_input, void *grad_weight,
                               bool round_product, int64_t num_tokens, int64_t num_experts, int64_t hidden, int dtype,
                               void *workspace, size_t workspace_size, void *stream_) {
    const char *name = "fm_router_linear_backward";
    const size_t needed = fm_router_linear_backward_workspace_size(num_tokens, num_experts, hidden, dtype);
    if (needed == 0)
        return fail(FM_ERR_UNSUPPORTED, "%s: experts and hidden must be multiples of 16 bytes, got %lld and %lld", name,
                    static_cast<long long>(num_experts), static_cast<long long>(hidden));
    FM_REQUIRE(grad_logits && aligned16(grad_logits), "%s: null or misaligned grad_logits", name);
    // fp32, more experts: a grouped product. Tokens: the grid's y.
    const bool own_input_grad =
        dtype != FM_DTYPE_F32 && num_experts <= router_linear::kInputGradMaxExperts && num_tokens < (int64_t(1) << 23);
    if (round_product && grad_input && !own_input_grad)
        return fail(FM_ERR_UNSUPPORTED, "%s: the product of this size is not rounded before it is added", name);
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
    if (own_input_grad) {
        const auto launch = [&](auto zero) {
            using T = decltype(zero);
            const auto run = round_product ? router_linear::launch_input_grad<T, true> : router_linear::launch_input_grad<T, false>;
            run(grad_logits, weight, grad_input, num_tokens, static_cast<int>(num_experts), static_cast<int>(hidden),
                static_cast<hipStream_t>(stream_));
        };
        dtype == FM_DTYPE_BF16 ? launch(bf16_t()) : launch(f16_t());
        return check_launch(name);
    }
    return fm_output_sparse_matmul(grad_logits, weight, grad_input, nullptr, num_tokens, hidden, num_experts, 1, num_experts, 1, hidden, 1,
                                   hidden, 1, 1, dtype, dtype, FM_INDEX_I32, nullptr, 0, stream_);
}

extern "C" int fm_router_linear_backward(const void *grad_logits, const void *input, const void *weight, void *grad_input,
                                         void *grad_weight, int64_t num_tokens, int64_t num_experts, int64_t hidden, int dtype,
                                         void *workspace, size_t workspace_size, void *stream) {
    return router_linear_backward(grad_logits, input, weight, grad_input, grad_weight, false, num_tokens, num_experts, hidden, dtype,
                                  workspace, workspace_size, stream);
}
