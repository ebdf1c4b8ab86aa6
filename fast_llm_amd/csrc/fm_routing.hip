// Top-k routing: for every token the k largest router logits, in descending order, their expert indices, and the
// softmax over just those k logits in fp32 (reference: MixtureOfExpertMLP._topk_routing,
// fast_llm/layers/decoder/mlp/mixture_of_experts.py:243-244, i.e. torch.topk followed by torch.softmax(dtype=fp32));
// the rest of the router's front end around it; and the backward of both with respect to the logits.
#include <type_traits>

#include "fm_gemm_common.h"
#include "fm_router_layout.h"

namespace fm {

constexpr int kRoutingThreads = 256;  // 4 tokens per workgroup
constexpr int kMaxPerLane = 16;       // experts <= 1024
constexpr int kMaxTopK = 64;
constexpr int kRouterMaxThreads = 1024;

// ---- the router front end: routing, auxiliary losses and shared experts in one pass ---------------------------
// Everything MixtureOfExpertMLP does between the router's logits and the sparse map (reference:
// fast_llm/layers/decoder/mlp/mixture_of_experts.py:146-171, 237-278) from one read of the logits:
//   * z-loss mean_t(logsumexp(logits_t)^2) on the logits as they come (:147-154, layers/language_model/loss/z_loss.py:88-92);
//   * jitter: the logits are multiplied by `noise` (drawn by the caller) and rounded to their type (:157-159, 234-235);
//   * top-k experts and the fp32 softmax over their logits (:243-244);
//   * the load-balancing loss sum_e mean_t(softmax(logits)[t, e]) * mean_t(selected[t, e]) (:245-254);
//   * shared experts, prepended to every token's slots with score 1 (:264-278).
// A workgroup walks a fixed range of tokens and keeps the per-expert sums of its tokens in registers; the sums of all
// workgroups are then added in a fixed order by a second kernel, so results do not depend on scheduling.
//
// What bounds it is the chain of dependent steps of a token: load a row, then k rounds of an arg-max. A token is
// therefore shared by no more lanes than it has experts (kGroup = 8 .. 64 lanes, 8 tokens per wavefront at 8
// experts), a lane holds no more logits than there are (kPerLane), and a round is a maximum of integer keys over the
// group in DPP and lane-swap instructions followed by one ballot. (A wavefront per token with 16 logits per lane at any
// number of experts and a butterfly of (value, index) pairs through LDS: 66 us forward, 100 us backward at 16384 tokens
// and 8 of 128 experts; now 17 and 11. 96 tokens: 42 us, now 5.)
template <int kGroup, int kPerLane>
struct RouterShape {
    static constexpr int kTokens = 64 / kGroup;  // tokens of a wavefront at a time
    static_assert(kGroup == 64 || kPerLane == 1, "more than one logit per lane: the whole wavefront shares a token");
};

// A float as an integer that orders like it (and -0 like +0); 0 is below -infinity. NaN is above every number, as in
// torch.topk: a token with a NaN logit selects that expert and gets NaN scores, so a broken router shows in the loss
// instead of silently losing a slot.
__device__ __forceinline__ uint32_t order_key(float value) {
    if (value != value) return 0xffffffffu;
    const uint32_t bits = __float_as_uint(value + 0.f);
    return bits & 0x80000000u ? ~bits : bits | 0x80000000u;
}
__device__ __forceinline__ float value_of_key(uint32_t key) {
    if (key == 0xffffffffu) return __uint_as_float(0x7fc00000u);
    return __uint_as_float(key & 0x80000000u ? key & 0x7fffffffu : ~key);
}
constexpr uint32_t kKeyOfMinusInfinity = 0x007fffffu;

// Reduction over the `kGroup` lanes that share a token; every lane gets the result.
template <int kGroup, typename V, typename Op>
__device__ __forceinline__ V group_reduce(V value, Op op) {
    static_assert(sizeof(V) == 4 && kGroup >= 8 && kGroup <= 64, "32-bit values, groups of 8 to 64 lanes");
    const auto dpp = [&](auto control) {
        return __builtin_bit_cast(V, __builtin_amdgcn_mov_dpp(__builtin_bit_cast(int, value), decltype(control)::value, 0xf, 0xf, true));
    };
    value = op(value, dpp(std::integral_constant<int, 0xB1>{}));   // lane ^ 1
    value = op(value, dpp(std::integral_constant<int, 0x4E>{}));   // lane ^ 2
    value = op(value, dpp(std::integral_constant<int, 0x141>{}));  // the other four of eight (mirrored)
    if constexpr (kGroup >= 16) value = op(value, dpp(std::integral_constant<int, 0x140>{}));  // the other eight of sixteen
    if constexpr (kGroup >= 32) {
        const uint32_t bits = __builtin_bit_cast(uint32_t, value);
        const auto rows = __builtin_amdgcn_permlane16_swap(bits, bits, false, false);
        value = op(__builtin_bit_cast(V, static_cast<uint32_t>(rows[0])), __builtin_bit_cast(V, static_cast<uint32_t>(rows[1])));
    }
    if constexpr (kGroup >= 64) {
        const uint32_t bits = __builtin_bit_cast(uint32_t, value);
        const auto halves = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
        value = op(__builtin_bit_cast(V, static_cast<uint32_t>(halves[0])), __builtin_bit_cast(V, static_cast<uint32_t>(halves[1])));
    }
    return value;
}
template <int kGroup>
__device__ __forceinline__ float group_sum(float value) {
    return group_reduce<kGroup>(value, [](float a, float b) { return a + b; });
}
template <int kGroup>
__device__ __forceinline__ uint32_t group_max(uint32_t value) {
    return group_reduce<kGroup>(value, [](uint32_t a, uint32_t b) { return a > b ? a : b; });
}

// The logits of a token as the router sees them: raw, and after the jitter (rounded to T like the reference's
// `logits * noise`). Lane l of the group holds experts l, l + kGroup, ...; absent ones are -infinity.
template <typename T, int kGroup, int kPerLane>
__device__ __forceinline__ void load_router_row(const T *logits, const T *noise, int64_t token, int experts, int lane,
                                                float (&raw)[kPerLane], float (&routed)[kPerLane],
                                                float (&factor)[kPerLane]) {
#pragma unroll
    for (int q = 0; q < kPerLane; ++q) {
        const int e = q * kGroup + lane;
        raw[q] = routed[q] = -INFINITY;
        factor[q] = 1.f;
        if (e < experts) {
            raw[q] = routed[q] = to_float(logits[token * experts + e]);
            if (noise != nullptr) {
                factor[q] = to_float(noise[token * experts + e]);
                routed[q] = to_float(from_float<T>(raw[q] * factor[q]));
            }
        }
    }
}

// log(sum_e exp(values[e])) over the experts of a token, given the largest of them.
template <int kGroup, int kPerLane>
__device__ __forceinline__ float group_logsumexp(const float (&values)[kPerLane], float maximum) {
    float sum = 0.f;
#pragma unroll
    for (int q = 0; q < kPerLane; ++q) sum += __expf(values[q] - maximum);
    return maximum + logf(group_sum<kGroup>(sum));
}

// `block_counts`: [workgroup][expert], may be null.
// kStatistics: also logsumexp, softmax sums and z-loss sums, which only the auxiliary losses and their gradients need.
template <typename T, int kGroup, int kPerLane, bool kStatistics>
__global__ __launch_bounds__(kRouterMaxThreads) void router_forward_kernel(
    const T *__restrict__ logits, const T *__restrict__ noise, int64_t *__restrict__ top_experts,
    float *__restrict__ scores, float *__restrict__ lse, int32_t *__restrict__ block_counts,
    float *__restrict__ block_sums, int64_t tokens, int64_t per_block, int experts, int k, int shared) {
    constexpr int kTokens = RouterShape<kGroup, kPerLane>::kTokens;
    extern __shared__ float lds_sums[];  // [waves][stats]
    const int wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const int lane = threadIdx.x & (kGroup - 1), group = (threadIdx.x & 63) / kGroup;
    const int64_t begin = blockIdx.x * per_block, end = min(begin + per_block, tokens);
    const int slots = shared + k;
    float probability_sum[kPerLane], z_sum = 0.f;
    int32_t count[kPerLane];
#pragma unroll
    for (int q = 0; q < kPerLane; ++q) probability_sum[q] = 0.f, count[q] = 0;

    for (int64_t first = begin + wave * kTokens; first < end; first += waves * kTokens) {
        // Lanes of groups past the last token work on the last one and keep nothing of it.
        const bool valid = first + group < end;
        const int64_t token = valid ? first + group : end - 1;
        float raw[kPerLane], values[kPerLane], factor[kPerLane];
        load_router_row<T, kGroup, kPerLane>(logits, noise, token, experts, lane, raw, values, factor);
        uint32_t key[kPerLane], best = 0;
#pragma unroll
        for (int q = 0; q < kPerLane; ++q) {
            key[q] = q * kGroup + lane < experts ? order_key(values[q]) : 0u;
            best = max(best, key[q]);
        }
        best = group_max<kGroup>(best);
        const float top_value = value_of_key(best);
        if constexpr (kStatistics) {
            const float lse_routed = group_logsumexp<kGroup, kPerLane>(values, top_value);
            float lse_raw = lse_routed;
            if (noise != nullptr) {
                uint32_t raw_best = 0;
#pragma unroll
                for (int q = 0; q < kPerLane; ++q)
                    raw_best = max(raw_best, q * kGroup + lane < experts ? order_key(raw[q]) : 0u);
                lse_raw = group_logsumexp<kGroup, kPerLane>(raw, value_of_key(group_max<kGroup>(raw_best)));
            }
            if (valid) {
                if (lane == 0) {
                    lse[2 * token] = lse_routed;
                    lse[2 * token + 1] = lse_raw;
                    z_sum += lse_raw * lse_raw;
                }
#pragma unroll
                for (int q = 0; q < kPerLane; ++q)
                    if (q * kGroup + lane < experts) probability_sum[q] += __expf(values[q] - lse_routed);
            }
        }

        float sum = 0.f, my_value = 0.f;
        int my_expert = 0;
        for (int j = 0; j < k; ++j) {
            if (j > 0) {
                best = 0;
#pragma unroll
                for (int q = 0; q < kPerLane; ++q) best = max(best, key[q]);
                best = group_max<kGroup>(best);
            }
            // The lowest expert with the largest key. A selected expert is then worth -infinity.
            int winner = -1;
#pragma unroll
            for (int q = 0; q < kPerLane; ++q) {
                uint64_t owners = __ballot(key[q] == best);
                if constexpr (kGroup < 64) owners = (owners >> (group * kGroup)) & ((1ull << kGroup) - 1);
                if (winner < 0 && owners != 0) winner = q * kGroup + __ffsll(static_cast<unsigned long long>(owners)) - 1;
            }
#pragma unroll
            for (int q = 0; q < kPerLane; ++q)
                if (q * kGroup + lane == winner) {
                    key[q] = kKeyOfMinusInfinity;
                    count[q] += valid ? 1 : 0;
                }
            const float shifted = __expf(value_of_key(best) - top_value);
            sum += shifted;
            if (lane == j) {  // lane j keeps slot j
                my_value = shifted;
                my_expert = winner;
            }
        }
        if (valid) {
            if (lane < k) {
                top_experts[token * slots + shared + lane] = my_expert;
                scores[token * slots + shared + lane] = my_value / sum;
            }
            for (int j = lane; j < shared; j += kGroup) {
                top_experts[token * slots + j] = experts + j;
                scores[token * slots + j] = 1.f;
            }
        }
    }

    if (block_counts == nullptr) return;
    // Sums of the workgroup's tokens: over the groups of a wavefront, then over the wavefronts in their order.
#pragma unroll
    for (int offset = kGroup; offset < 64; offset <<= 1) {
#pragma unroll
        for (int q = 0; q < kPerLane; ++q) {
            count[q] += __shfl_xor(count[q], offset, 64);
            if constexpr (kStatistics) probability_sum[q] += __shfl_xor(probability_sum[q], offset, 64);
        }
        if constexpr (kStatistics) z_sum += __shfl_xor(z_sum, offset, 64);
    }
    const int columns = kStatistics ? RouterStats::size(experts) : experts;
    int32_t *wave_counts = reinterpret_cast<int32_t *>(lds_sums) + wave * columns;
    float *wave_sums = lds_sums + wave * columns + experts;
    if (group == 0) {
#pragma unroll
        for (int q = 0; q < kPerLane; ++q) {
            const int e = q * kGroup + lane;
            if (e < experts) {
                wave_counts[e] = count[q];
                if constexpr (kStatistics) wave_sums[e] = probability_sum[q];
            }
        }
        if (kStatistics && lane == 0) wave_sums[experts] = z_sum;
    }
    __syncthreads();
    for (int c = threadIdx.x; c < columns; c += blockDim.x) {
        if (c < experts) {
            int32_t total = 0;
            for (int w = 0; w < waves; ++w) total += reinterpret_cast<const int32_t *>(lds_sums)[w * columns + c];
            block_counts[static_cast<int64_t>(blockIdx.x) * (experts + shared) + c] = total;
        } else {
            float total = 0.f;
            for (int w = 0; w < waves; ++w) total += lds_sums[w * columns + c];
            block_sums[static_cast<int64_t>(blockIdx.x) * (experts + 1) + c - experts] = total;
        }
    }
    // Every token of the range visits the shared experts.
    for (int j = threadIdx.x; j < shared; j += blockDim.x)
        block_counts[static_cast<int64_t>(blockIdx.x) * (experts + shared) + experts + j] = static_cast<int32_t>(max(end - begin, int64_t(0)));
}

__global__ __launch_bounds__(kFinishThreads) void router_finish_kernel(RouterFinish finish) {
    __shared__ FinishLds lds;
    finish_router(finish, lds);
}

// Gradient of the raw logits: through the top-k softmax,
//   scores[t, j] * (grad_scores[t, j] - sum_i scores[t, i] * grad_scores[t, i]) for the j-th selected expert of token t
// and 0 for an expert that was not selected; plus, scaled by the constant gradients the reference attaches to its auxiliary losses (functional/utils.py:63-71),
//   load balancing:  aux_scale * p[t, e] * (count[e] - sum_i p[t, i] * count[i]),  p = softmax of the routed logits
//   z-loss:          z_scale * lse_raw[t] * softmax(raw logits)[t, e]
// with aux_scale = aux_grad / tokens^2 and z_scale = 2 * z_grad / tokens; the routed part is multiplied by the jitter.
template <typename T, int kGroup, int kPerLane>
__global__ __launch_bounds__(kRoutingThreads) void router_backward_kernel(
    const float *__restrict__ grad_scores, const float *__restrict__ scores, const int64_t *__restrict__ top_experts,
    const T *__restrict__ logits, const T *__restrict__ noise, const float *__restrict__ lse,
    const float *__restrict__ statistics, T *__restrict__ grad_logits, float aux_scale, float z_scale, int64_t tokens,
    int experts, int k, int shared, bool round_grad_scores) {
    constexpr int kTokens = RouterShape<kGroup, kPerLane>::kTokens;
    const int lane = threadIdx.x & (kGroup - 1), group = (threadIdx.x & 63) / kGroup;
    const int64_t mine = (static_cast<int64_t>(blockIdx.x) * (kRoutingThreads / 64) + (threadIdx.x >> 6)) * kTokens + group;
    const bool valid = mine < tokens;
    const int64_t token = valid ? mine : tokens - 1;
    const int slots = shared + k;
    float raw[kPerLane], routed[kPerLane], factor[kPerLane], grad[kPerLane];
    // The logits are only needed for the losses and the jitter.
    const bool with_losses = aux_scale != 0.f || z_scale != 0.f;
    if (with_losses || noise != nullptr) {
        load_router_row<T, kGroup, kPerLane>(logits, noise, token, experts, lane, raw, routed, factor);
    } else {
#pragma unroll
        for (int q = 0; q < kPerLane; ++q) factor[q] = 1.f;
    }
    const float lse_routed = with_losses ? lse[2 * token] : 0.f, lse_raw = with_losses ? lse[2 * token + 1] : 0.f;
    const float score = lane < k ? scores[token * slots + shared + lane] : 0.f;
    float grad_score = lane < k ? grad_scores[token * slots + shared + lane] : 0.f;
    if (round_grad_scores) grad_score = to_float(from_float<T>(grad_score));
    const int expert = lane < k ? static_cast<int>(top_experts[token * slots + shared + lane]) : -1;

    // Load balancing.
    float weighted = 0.f;
#pragma unroll
    for (int q = 0; q < kPerLane; ++q) {
        const int e = q * kGroup + lane;
        grad[q] = 0.f;
        if (e < experts && aux_scale != 0.f) {
            const float probability = __expf(routed[q] - lse_routed);
            const float selected = statistics[RouterStats::count(experts, e)];
            grad[q] = probability * selected;  // finished below
            weighted += grad[q];
        }
    }
    if (aux_scale != 0.f) {
        weighted = group_sum<kGroup>(weighted);
#pragma unroll
        for (int q = 0; q < kPerLane; ++q) {
            const int e = q * kGroup + lane;
            if (e < experts) grad[q] = aux_scale * (grad[q] - __expf(routed[q] - lse_routed) * weighted);
        }
    }
    // Top-k softmax.
    const float dot = group_sum<kGroup>(score * grad_score);
    const float grad_selected = score * (grad_score - dot);
    for (int j = 0; j < k; ++j) {
        const int selected = __shfl(expert, j, kGroup);
        const float value = __shfl(grad_selected, j, kGroup);
#pragma unroll
        for (int q = 0; q < kPerLane; ++q)
            if (q * kGroup + lane == selected) grad[q] += value;
    }
    // Back through the jitter; z-loss.
#pragma unroll
    for (int q = 0; q < kPerLane; ++q) {
        const int e = q * kGroup + lane;
        if (valid && e < experts) {
            float value = grad[q] * factor[q];
            if (z_scale != 0.f) value += z_scale * lse_raw * __expf(raw[q] - lse_raw);
            grad_logits[token * experts + e] = from_float<T>(value);
        }
    }
}

// Runs the statement with kGroup and kPerLane: the fewest lanes per token that hold its logits, one each as long as a
// wavefront suffices.
#define FM_DISPATCH_ROUTER_SHAPE(experts, kGroup, kPerLane, ...)                                        \
    if (experts <= 8) { constexpr int kGroup = 8, kPerLane = 1; __VA_ARGS__; }                          \
    else if (experts <= 16) { constexpr int kGroup = 16, kPerLane = 1; __VA_ARGS__; }                   \
    else if (experts <= 32) { constexpr int kGroup = 32, kPerLane = 1; __VA_ARGS__; }                   \
    else if (experts <= 64) { constexpr int kGroup = 64, kPerLane = 1; __VA_ARGS__; }                   \
    else if (experts <= 128) { constexpr int kGroup = 64, kPerLane = 2; __VA_ARGS__; }                  \
    else if (experts <= 256) { constexpr int kGroup = 64, kPerLane = 4; __VA_ARGS__; }                  \
    else if (experts <= 512) { constexpr int kGroup = 64, kPerLane = 8; __VA_ARGS__; }                  \
    else { constexpr int kGroup = 64, kPerLane = kMaxPerLane; __VA_ARGS__; }

}  // namespace fm

using namespace fm;

extern "C" size_t fm_router_workspace_size(int64_t num_tokens, int64_t num_experts) {
    if (num_tokens <= 0 || num_experts <= 0) return 0;
    return router_counts_bytes(num_tokens, num_experts + kMaxTopK) +
           sizeof(float) * static_cast<size_t>(router_blocks(num_tokens)) * (num_experts + 1);
}

static int check_router_shape(const char *name, int64_t num_tokens, int64_t num_experts, int64_t experts_per_token,
                              int64_t shared_experts, int dtype) {
    FM_REQUIRE(valid_dtype(dtype), "%s: bad dtype %d", name, dtype);
    FM_REQUIRE(num_tokens >= 0 && num_experts > 0 && num_experts <= 64 * kMaxPerLane, "%s: %lld experts (1..%d)", name,
               static_cast<long long>(num_experts), 64 * kMaxPerLane);
    FM_REQUIRE(experts_per_token > 0 && experts_per_token <= num_experts && shared_experts >= 0 &&
                   experts_per_token + shared_experts <= kMaxTopK,
               "%s: experts_per_token %lld, shared_experts %lld", name, static_cast<long long>(experts_per_token),
               static_cast<long long>(shared_experts));
    FM_REQUIRE(num_tokens < (int64_t(1) << 31), "%s: too many tokens", name);
    return FM_OK;
}

namespace fm {

template <typename T, int kGroup, int kPerLane, bool kStatistics>
static int launch_router_forward(const void *logits, const void *noise, void *top_experts, void *scores, void *lse,
                                  int32_t *block_counts, float *block_sums, int64_t tokens, int experts, int k,
                                  int shared, hipStream_t stream) {
    constexpr int kTokens = RouterShape<kGroup, kPerLane>::kTokens;
    const auto kernel = router_forward_kernel<T, kGroup, kPerLane, kStatistics>;
    // Where nobody wants counts a wavefront has its tokens once and no workgroup is asked what it did: top 8 of 131072 tokens of
    // 512 experts 159 us, 971 when 256 workgroups of 4 wavefronts walked over them.
    int blocks = static_cast<int>((tokens + kTokens * 4 - 1) / (kTokens * 4)), threads = 256;
    int64_t per_block = kTokens * 4;
    size_t lds = 0;
    if (block_counts != nullptr) {
        // One workgroup per CU at most, so 16 wavefronts, whose sums take up to 131 KB of its 160 (1024 experts). 131072 tokens
        // of 512 experts 298 us, 1130 with 4 wavefronts.
        blocks = router_blocks(tokens), per_block = router_tokens_per_block(tokens), threads = kRouterMaxThreads;
        lds = sizeof(float) * (threads / 64) * (kStatistics ? RouterStats::size(experts) : experts);
    }
    if (lds > 64 * 1024) {
        static std::atomic<uint64_t> configured{0};
        constexpr int kMost = static_cast<int>(sizeof(float)) * (kRouterMaxThreads / 64) * (2 * 64 * kMaxPerLane + 1);
        if (int status = allow_lds(reinterpret_cast<const void *>(kernel), kMost, configured)) return status;
    }
    kernel<<<blocks, threads, lds, stream>>>(static_cast<const T *>(logits), static_cast<const T *>(noise),
                                             static_cast<int64_t *>(top_experts), static_cast<float *>(scores),
                                             static_cast<float *>(lse), block_counts, block_sums, tokens, per_block, experts, k, shared);
    return FM_OK;
}

static int run_router_backward(const char *name, const void *grad_scores, const void *scores, const void *top_experts,
                               const void *logits, const void *noise, const void *lse, const void *statistics,
                               void *grad_logits, float aux_scale, float z_scale, int64_t tokens, int experts, int k,
                               int shared, int dtype, bool round_grad_scores, hipStream_t stream) {
    FM_DISPATCH_DTYPE(dtype, T, {
        FM_DISPATCH_ROUTER_SHAPE(experts, kGroup, kPerLane, {
            constexpr int64_t kTokens = RouterShape<kGroup, kPerLane>::kTokens * (kRoutingThreads / 64);
            router_backward_kernel<T, kGroup, kPerLane><<<(tokens + kTokens - 1) / kTokens, kRoutingThreads, 0, stream>>>(
                static_cast<const float *>(grad_scores), static_cast<const float *>(scores),
                static_cast<const int64_t *>(top_experts), static_cast<const T *>(logits), static_cast<const T *>(noise),
                static_cast<const float *>(lse), static_cast<const float *>(statistics), static_cast<T *>(grad_logits),
                aux_scale, z_scale, tokens, experts, k, shared, round_grad_scores);
        })
    });
    return check_launch(name);
}

}  // namespace fm

extern "C" int fm_topk_routing(const void *logits, void *top_experts, void *scores, int64_t num_tokens,
                               int64_t num_experts, int64_t experts_per_token, int dtype, void *stream) {
    const char *name = "fm_topk_routing";
    if (int status = check_router_shape(name, num_tokens, num_experts, experts_per_token, 0, dtype)) return status;
    if (num_tokens == 0) return FM_OK;
    FM_REQUIRE(logits && top_experts && scores, "%s: null tensor", name);
    FM_DISPATCH_DTYPE(dtype, T, {
        FM_DISPATCH_ROUTER_SHAPE(num_experts, kGroup, kPerLane, {
            if (int status = launch_router_forward<T, kGroup, kPerLane, false>(
                    logits, nullptr, top_experts, scores, nullptr, nullptr, nullptr, num_tokens, static_cast<int>(num_experts),
                    static_cast<int>(experts_per_token), 0, static_cast<hipStream_t>(stream)))
                return status;
        })
    });
    return check_launch(name);
}

extern "C" int fm_topk_routing_backward(const void *grad_scores, const void *scores, const void *top_experts,
                                        void *grad_logits, int64_t num_tokens, int64_t num_experts,
                                        int64_t experts_per_token, int dtype, void *stream) {
    const char *name = "fm_topk_routing_backward";
    if (int status = check_router_shape(name, num_tokens, num_experts, experts_per_token, 0, dtype)) return status;
    if (num_tokens == 0) return FM_OK;
    FM_REQUIRE(grad_scores && scores && top_experts && grad_logits, "%s: null tensor", name);
    return run_router_backward(name, grad_scores, scores, top_experts, nullptr, nullptr, nullptr, nullptr, grad_logits,
                               0.f, 0.f, num_tokens, static_cast<int>(num_experts),
                               static_cast<int>(experts_per_token), 0, dtype, false, static_cast<hipStream_t>(stream));
}

RouterFinish fm::router_finish_of(const void *workspace, void *statistics, void *losses, int64_t num_tokens, int64_t num_experts,
                                  int64_t shared_experts) {
    const size_t sums = router_counts_bytes(num_tokens, num_experts + kMaxTopK);
    return RouterFinish{static_cast<const int32_t *>(workspace),
                        reinterpret_cast<const float *>(static_cast<const char *>(workspace) + sums),
                        static_cast<float *>(statistics),
                        static_cast<float *>(losses),
                        router_blocks(num_tokens),
                        static_cast<int>(num_experts),
                        static_cast<int>(shared_experts),
                        num_tokens};
}

int fm::router_forward(const void *logits, const void *noise, void *top_experts, void *scores, void *lse, void *statistics,
                       void *losses, void *workspace, size_t workspace_size, int64_t num_tokens, int64_t num_experts,
                       int64_t experts_per_token, int64_t shared_experts, int dtype, bool finish, void *stream_) {
    const char *name = "fm_router_forward";
    if (int status = check_router_shape(name, num_tokens, num_experts, experts_per_token, shared_experts, dtype))
        return status;
    FM_REQUIRE(num_tokens > 0, "%s: no tokens", name);
    // The statistics may be left out together: then only the routing and the counts for the sparse map are computed.
    const bool with_statistics = lse != nullptr || statistics != nullptr || losses != nullptr;
    FM_REQUIRE(logits && top_experts && scores && workspace && (!with_statistics || (lse && statistics && losses)),
               "%s: null tensor", name);
    FM_REQUIRE(workspace_size >= fm_router_workspace_size(num_tokens, num_experts), "%s: workspace of %zu bytes, need %zu",
               name, workspace_size, fm_router_workspace_size(num_tokens, num_experts));
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    const int experts = static_cast<int>(num_experts), shared = static_cast<int>(shared_experts);
    int32_t *block_counts = static_cast<int32_t *>(workspace);
    float *block_sums = reinterpret_cast<float *>(static_cast<char *>(workspace) + router_counts_bytes(num_tokens, num_experts + kMaxTopK));
    FM_DISPATCH_DTYPE(dtype, T, {
        FM_DISPATCH_ROUTER_SHAPE(experts, kGroup, kPerLane, {
            auto launch = with_statistics ? launch_router_forward<T, kGroup, kPerLane, true>
                                          : launch_router_forward<T, kGroup, kPerLane, false>;
            if (int status = launch(logits, noise, top_experts, scores, lse, block_counts, block_sums, num_tokens, experts,
                                    static_cast<int>(experts_per_token), shared, stream))
                return status;
        })
    });
    if (with_statistics && finish)
        router_finish_kernel<<<1, kFinishThreads, 0, stream>>>(
            router_finish_of(workspace, statistics, losses, num_tokens, num_experts, shared_experts));
    return check_launch(name);
}

extern "C" int fm_router_forward(const void *logits, const void *noise, void *top_experts, void *scores, void *lse, void *statistics,
                                 void *losses, void *workspace, size_t workspace_size, int64_t num_tokens, int64_t num_experts,
                                 int64_t experts_per_token, int64_t shared_experts, int dtype, void *stream) {
    return router_forward(logits, noise, top_experts, scores, lse, statistics, losses, workspace, workspace_size, num_tokens, num_experts,
                          experts_per_token, shared_experts, dtype, true, stream);
}

int fm::router_backward(const void *grad_scores, const void *scores, const void *top_experts, const void *logits,
                        const void *noise, const void *lse, const void *statistics, void *grad_logits,
                        double auxiliary_loss_grad, double z_loss_grad, int64_t num_tokens, int64_t num_experts,
                        int64_t experts_per_token, int64_t shared_experts, int dtype, bool round_grad_scores,
                        void *stream_) {
    const char *name = "fm_router_backward";
    if (int status = check_router_shape(name, num_tokens, num_experts, experts_per_token, shared_experts, dtype))
        return status;
    if (num_tokens == 0) return FM_OK;
    const bool with_losses = auxiliary_loss_grad != 0.0 || z_loss_grad != 0.0;
    FM_REQUIRE(grad_scores && scores && top_experts && logits && grad_logits && (!with_losses || (lse && statistics)),
               "%s: null tensor", name);
    hipStream_t stream = static_cast<hipStream_t>(stream_);
    const double count = static_cast<double>(num_tokens);
    const float aux_scale = static_cast<float>(auxiliary_loss_grad / count / count);
    const float z_scale = static_cast<float>(2.0 * z_loss_grad / count);
    return run_router_backward(name, grad_scores, scores, top_experts, logits, noise, lse, statistics, grad_logits,
                               aux_scale, z_scale, num_tokens, static_cast<int>(num_experts),
                               static_cast<int>(experts_per_token), static_cast<int>(shared_experts), dtype,
                               round_grad_scores, stream);
}

extern "C" int fm_router_backward(const void *grad_scores, const void *scores, const void *top_experts,
                                  const void *logits, const void *noise, const void *lse, const void *statistics,
                                  void *grad_logits, double auxiliary_loss_grad, double z_loss_grad,
                                  int64_t num_tokens, int64_t num_experts, int64_t experts_per_token,
                                  int64_t shared_experts, int dtype, void *stream) {
    return router_backward(grad_scores, scores, top_experts, logits, noise, lse, statistics, grad_logits,
                           auxiliary_loss_grad, z_loss_grad, num_tokens, num_experts, experts_per_token, shared_experts,
                           dtype, false, stream);
}
