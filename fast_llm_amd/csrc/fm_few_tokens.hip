// Inference of the dropless MoE MLP for few tokens (text generation): every expert that some token selected is read
// from memory for a handful of rows, so the weights' bytes are the bound and nothing else may cost much.
//
//   * No sparse layout: a workgroup finds the slots (token, choice) of its expert by scanning `top_experts`, and reads
//     the dense rows through them. No map, no dispatch copy, no padding rows.
//   * few_tokens_layer_1_kernel: 16 or 32 gate rows and as many up rows of one expert's weight (or 32 or 64 rows without
//     a gate) per workgroup, multiplied with up to 64 tokens at a time; the four wavefronts take every fourth chunk of K
//     and add up in LDS; the activation is applied there.
//   * few_tokens_layer_2_kernel: 128 output columns of one expert per workgroup and a piece of the reduction. The
//     weight lies [K][column] in memory; a lane loads eight K-rows of its eight columns and transposes the 8 x 8 block in
//     registers (one v_perm_b32 per two values), no LDS either. Pieces and slots are written as fp32 sums.
//   * few_tokens_combine_kernel adds the pieces and the scaled slots of a token in a fixed order.
// All three tolerate any number of rows per expert (they walk them 64 at a time and read the weights again for each);
// the caller decides up to where that is the faster way. Deterministic: every sum has a fixed order.
// One token through 2 of 8 experts of 4096 x 14336: 116 us for the 705 MB of weights (6.1 TB/s), 197 on tiles of 256 rows;
// 64 tokens: 471 us (6.0 TB/s), 704 on tiles.
#include <type_traits>

#include "fm_activation_math.h"
#include "fm_gemm_common.h"

namespace fm {

namespace few {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4_t;

// D[m][n] += sum_k A[m][k] B[n][k]: lane l holds row l % 16, k = 8 (l / 16) .. + 7 of both operands, and of D the
// column n = l % 16, rows m = 4 (l / 16) .. + 3.
__device__ __forceinline__ f32x4_t mfma(bf16_t, u32x4_t a, u32x4_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x4_t mfma(f16_t, u32x4_t a, u32x4_t b, f32x4_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

struct Args {
    const void *x;               // [tokens, hidden]
    const int64_t *top_experts;  // [tokens * slots]
    const float *scores;         // [tokens * slots]
    const void *weight_1, *weight_2;
    void *activation;  // [tokens * slots, ffn]
    float *pieces;     // [splits][tokens * slots, hidden]
    void *out;         // [tokens, hidden]
    int tokens, slots, hidden, ffn, experts, activation_type;
    int entries;   // tokens * slots
    int by_entry;  // a workgroup row per entry instead of one per expert
    int splits, split_length;
};

constexpr int kThreads = 256, kWaves = 4;
constexpr uint32_t kOutOfRange = 0xffffffffu;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void *pointer, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(uniform_pointer(static_cast<const char *>(pointer))), 0,
                                             static_cast<int>(bytes), kBufferResourceFlags);
}
// 16 bytes at a lane's own offset; zeros for offsets outside the buffer.
template <int kCachePolicy = 0>
__device__ __forceinline__ u32x4_t load(__amdgpu_buffer_rsrc_t buffer, uint32_t offset) {
    return __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(buffer, static_cast<int>(offset), 0, kCachePolicy));
}
constexpr int kStreaming = 2;  // nt: weights are read once

// The expert of this workgroup and, in LDS, the entries that selected it. Returns their number (0: nothing to do).
__device__ __forceinline__ int find_rows(const Args &args, int which, int *list, int &expert) {
    __shared__ int count;
    if (threadIdx.x == 0) count = 0;
    expert = args.by_entry ? static_cast<int>(args.top_experts[which]) : which;
    if (expert < 0 || expert >= args.experts) return 0;
    __syncthreads();
    bool seen = false;
    for (int i = threadIdx.x; i < args.entries; i += kThreads) {
        if (args.top_experts[i] != expert) continue;
        // With a workgroup row per entry, the first entry of an expert does the work.
        if (args.by_entry && i < which) seen = true;
        list[atomicAdd(&count, 1)] = i;
    }
    const bool taken = __syncthreads_or(seen);
    return taken ? 0 : __builtin_amdgcn_readfirstlane(count);
}

// ---- layer 1 and activation ----------------------------------------------------------------------------
// Sums over K of kSets x 16 weight rows times kGroups x 16 tokens, this wavefront's chunks of 128 only.
// A load instruction takes 256 bytes of each of four rows (lane l: row l / 16, 16 bytes at 16 (l % 16)); the fragments
// want 16 bytes of each of 16 rows, so the chunk passes through the wavefront's own 4 kSets KiB of LDS (XOR-swizzled: reads and
// writes hit all banks; one wavefront's LDS operations execute in order, so no barrier). Loads shaped like the fragments,
// 64 bytes of each of 16 rows, took 326 us for the 1.9 GB of 8 experts of 4096 x 28672 and 8 tokens where these take 242
// (7.8 TB/s).
// The wavefronts' chunks are taken four by four, from trip `first_trip` (below their number) on and then from the first one.
// `row_offset[i]`: byte offset of the lane's 16 bytes in the rows 4 i + l / 16 at k = 0 (kOutOfRange: no such row).
template <typename T, int kSets, int kGroups>
__device__ __forceinline__ void multiply_rows(__amdgpu_buffer_rsrc_t weight, __amdgpu_buffer_rsrc_t x,
                                              const uint32_t (&row_offset)[kSets * 4], const uint32_t (&token_offset)[kGroups],
                                              FM_LDS(char) * lds, int length, int first_trip, int wave, int lane,
                                              f32x4_t (&sums)[kSets][kGroups]) {
    constexpr int kChunk = 128, kSteps = kChunk / 32;
    const int load_k = (lane & 15) * 8, lane_k = (lane >> 4) * 8, load_row = lane >> 4, row = lane & 15;
    u32x4_t raw[kSets * 4], tokens[2][kGroups][kSteps];
    const auto fetch_rows = [&](int k0) {
        const bool exists = k0 + load_k < length;  // a multiple of 8
#pragma unroll
        for (int i = 0; i < kSets * 4; ++i)
            raw[i] = load<kStreaming>(weight, exists && row_offset[i] != kOutOfRange ? row_offset[i] + k0 * 2 : kOutOfRange);
    };
    const auto fetch_tokens = [&](int k0, u32x4_t(&values)[kGroups][kSteps]) {
#pragma unroll
        for (int s = 0; s < kSteps; ++s)
#pragma unroll
            for (int g = 0; g < kGroups; ++g)
                values[g][s] = load(x, k0 + s * 32 + lane_k < length ? token_offset[g] + (k0 + s * 32 + lane_k) * 2 : kOutOfRange);
    };
    const auto chunk = [&](int next_k0, u32x4_t(&now)[kGroups][kSteps], u32x4_t(&next)[kGroups][kSteps]) {
#pragma unroll
        for (int i = 0; i < kSets * 4; ++i) {
            const int r = (4 * i + load_row) & 15;
            *(FM_LDS(u32x4_t) *)(lds + (i / 4) * 4096 + r * 256 + (((lane & 15) ^ r) << 4)) = raw[i];
        }
        // The next chunk is on its way while this one is multiplied; past the end it is zeros and touches no memory.
        fetch_rows(next_k0);
        fetch_tokens(next_k0, next);
        // The lanes read what others wrote: the hardware keeps a wavefront's LDS operations in order, and this the compiler.
        asm volatile("" ::: "memory");
#pragma unroll
        for (int s = 0; s < kSteps; ++s)
#pragma unroll
            for (int r = 0; r < kSets; ++r) {
                const u32x4_t fragment = *(FM_LDS(u32x4_t) *)(lds + r * 4096 + row * 256 + (((4 * s + (lane >> 4)) ^ row) << 4));
#pragma unroll
                for (int g = 0; g < kGroups; ++g) sums[r][g] = mfma(T(), fragment, now[g][s], sums[r][g]);
            }
        asm volatile("" ::: "memory");  // and the next chunk's writes stay behind these reads
    };
    const int trips = (length + kWaves * kChunk - 1) / (kWaves * kChunk);
    int trip = first_trip, left = trips;
    const auto next_chunk = [&]() {  // where this wavefront's next chunk starts; past the end after the last one
        if (left <= 0) return length;
        const int k0 = (trip * kWaves + wave) * kChunk;
        trip = trip + 1 == trips ? 0 : trip + 1;
        --left;
        return k0;
    };
    const int first = next_chunk();
    fetch_rows(first);
    fetch_tokens(first, tokens[0]);
    for (int t = 0; t < trips; t += 2) {
        chunk(next_chunk(), tokens[0], tokens[1]);
        chunk(next_chunk(), tokens[1], tokens[0]);
    }
}

// Weight rows of up to this many elements are read from another place on by every workgroup: the workgroups keep about the same
// pace, and 1 KiB of rows that are 4 KiB or less apart lie in few of the memory's channels. Whole pass in us, from the start / so:
// 96 tokens over 128 experts of 2048 x 768 225.7 / 220.5, 16 over 64 of 2048 x 1408 170.5 / 167, 40 over 32 of 1024 x 2816 113.5 / 112;
// rows of 4096 are better read in one go: one token over 8 experts of 4096 x 14336 127 / 132, 3000 x 4096 250 / 251.
constexpr int kMaxRotatedRow = 2048;

// kSets x 16 weight rows per workgroup: half of them gate rows and the others the up rows that go with them, or (not
// gated) consecutive rows.
template <typename T, bool kGated, int kSets, int kMaxGroups>
__global__ __launch_bounds__(kThreads) void few_tokens_layer_1_kernel(Args args) {
    extern __shared__ __attribute__((aligned(16))) int list[];  // [entries], then the wavefronts' sums
    int expert;
    const int rows = find_rows(args, blockIdx.y, list, expert);
    if (rows == 0) return;
    f32x4_t *partial = reinterpret_cast<f32x4_t *>(list + (args.entries + 3) / 4 * 4);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ffn = args.ffn, hidden = args.hidden;
    constexpr int kOutputSets = kGated ? kSets / 2 : kSets;  // 16 outputs each
    const int first = blockIdx.x * kOutputSets * 16;
    const int64_t block_elements = static_cast<int64_t>(ffn) * (kGated ? 2 : 1) * hidden;
    const __amdgpu_buffer_rsrc_t weight =
        buffer_of(static_cast<const T *>(args.weight_1) + expert * block_elements, static_cast<uint32_t>(block_elements * 2));
    const __amdgpu_buffer_rsrc_t x = buffer_of(args.x, static_cast<uint32_t>(args.tokens) * hidden * 2);
    uint32_t row_offset[kSets * 4];
#pragma unroll
    for (int i = 0; i < kSets * 4; ++i) {
        const int set = i / 4, f = first + set % kOutputSets * 16 + i % 4 * 4 + (lane >> 4);
        row_offset[i] = f < ffn ? static_cast<uint32_t>(((f + set / kOutputSets * ffn) * static_cast<int64_t>(hidden) + (lane & 15) * 8) * 2)
                                : kOutOfRange;
    }
    const int first_trip = hidden <= kMaxRotatedRow ? blockIdx.x % ((hidden + kWaves * 128 - 1) / (kWaves * 128)) : 0;
    const auto activate = [&](float value) {
        float result;
        FM_DISPATCH_ACTIVATION(args.activation_type, kActivation, result = activation_forward<kActivation>(value));
        return result;
    };

    for (int base = 0; base < rows; base += 16 * kMaxGroups) {
        const int groups = min((rows - base + 15) / 16, kMaxGroups);
        const auto run = [&](auto constant) {
            constexpr int kGroups = decltype(constant)::value;
            uint32_t token_offset[kGroups];
#pragma unroll
            for (int g = 0; g < kGroups; ++g) {
                const int entry = list[min(base + g * 16 + (lane & 15), rows - 1)];
                token_offset[g] = static_cast<uint32_t>(entry / args.slots) * hidden * 2;
            }
            f32x4_t sums[kSets][kGroups];
#pragma unroll
            for (int r = 0; r < kSets; ++r)
#pragma unroll
                for (int g = 0; g < kGroups; ++g) sums[r][g] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            FM_LDS(char) *chunks = (FM_LDS(char) *)reinterpret_cast<char *>(partial) + wave * kSets * 4096;
            multiply_rows<T, kSets, kGroups>(weight, x, row_offset, token_offset, chunks, hidden, first_trip, wave, lane, sums);
            __syncthreads();


            // Token group by token group, [wavefront][set][lane]; wavefront w finishes the output sets w, w + 4, ...
#pragma unroll
            for (int g = 0; g < kGroups; ++g) {
#pragma unroll
                for (int r = 0; r < kSets; ++r) partial[(wave * kSets + r) * 64 + lane] = sums[r][g];
                __syncthreads();
                const int row = base + g * 16 + (lane & 15);
                for (int set = wave; set < kOutputSets; set += kWaves) {
                    const auto total = [&](int r) {
                        f32x4_t sum = partial[r * 64 + lane];
#pragma unroll
                        for (int w = 1; w < kWaves; ++w) sum += partial[(w * kSets + r) * 64 + lane];
                        return sum;
                    };
                    const int f = first + set * 16 + (lane >> 4) * 4;
                    if (row >= rows || f >= ffn) continue;
                    struct alignas(8) Four {
                        T v[4];
                    } result;
                    // Rounded first, like the layer-1 output that the separate kernels store.
                    const f32x4_t gate = total(set);
                    if constexpr (kGated) {
                        const f32x4_t up = total(set + kOutputSets);
#pragma unroll
                        for (int c = 0; c < 4; ++c)
                            result.v[c] = from_float<T>(activate(to_float(from_float<T>(gate[c]))) * to_float(from_float<T>(up[c])));
                    } else {
#pragma unroll
                        for (int c = 0; c < 4; ++c) result.v[c] = from_float<T>(activate(to_float(from_float<T>(gate[c]))));
                    }
                    *reinterpret_cast<Four *>(static_cast<T *>(args.activation) + static_cast<int64_t>(list[row]) * ffn + f) = result;
                }
                __syncthreads();
            }
        };
        if (kMaxGroups == 1 || groups == 1) run(std::integral_constant<int, 1>{});
        else if (kMaxGroups == 2 || groups == 2) run(std::integral_constant<int, (kMaxGroups < 2 ? kMaxGroups : 2)>{});
        else run(std::integral_constant<int, kMaxGroups>{});
    }
}

// ---- layer 2 -------------------------------------------------------------------------------------------
// Sums over f in [begin, end) of 128 weight columns times kGroups x 16 rows, this wavefront's chunks of 32 only.
// sums[i][g]: columns 8 m + i, m = 0 .. 15.
template <typename T, int kGroups>
__device__ __forceinline__ void multiply_columns(__amdgpu_buffer_rsrc_t weight, __amdgpu_buffer_rsrc_t rows, uint32_t column_offset,
                                                 const uint32_t (&row_offset)[kGroups], int stride, int begin, int end, int wave,
                                                 int lane, f32x4_t (&sums)[8][kGroups]) {
    struct Operands {
        u32x4_t columns[8], rows[kGroups];
    };
    const int lane_k = (lane >> 4) * 8;
    const auto fetch = [&](int f0, Operands &operands) {
        const int f = f0 + lane_k;
        const bool exists = f < end;  // a multiple of 8
        const uint32_t offset = exists && column_offset != kOutOfRange ? column_offset + static_cast<uint32_t>(f) * stride : kOutOfRange;
#pragma unroll
        for (int j = 0; j < 8; ++j) operands.columns[j] = load<kStreaming>(weight, offset == kOutOfRange ? kOutOfRange : offset + j * stride);
#pragma unroll
        for (int g = 0; g < kGroups; ++g) operands.rows[g] = load(rows, exists ? row_offset[g] + f * 2 : kOutOfRange);
    };
    const auto multiply = [&](const Operands &operands) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            // Column i of the lane's eight, f = 0 .. 7: the low or high halves of dword i / 2 of the eight loads.
            u32x4_t column;
#pragma unroll
            for (int p = 0; p < 4; ++p)
                column[p] = __builtin_amdgcn_perm(operands.columns[2 * p + 1][i / 2], operands.columns[2 * p][i / 2],
                                                  i % 2 ? 0x07060302u : 0x05040100u);
#pragma unroll
            for (int g = 0; g < kGroups; ++g) sums[i][g] = mfma(T(), column, operands.rows[g], sums[i][g]);
        }
    };
    Operands even, odd;
    fetch(begin + wave * 32, even);
    for (int f0 = begin + wave * 32; f0 < end; f0 += 2 * kWaves * 32) {
        fetch(f0 + kWaves * 32, odd);
        multiply(even);
        fetch(f0 + 2 * kWaves * 32, even);
        multiply(odd);
    }
}

template <typename T, int kMaxGroups>
__global__ __launch_bounds__(kThreads) void few_tokens_layer_2_kernel(Args args) {
    extern __shared__ __attribute__((aligned(16))) int list[];
    int expert;
    const int rows = find_rows(args, blockIdx.y, list, expert);
    if (rows == 0) return;
    float *partial = reinterpret_cast<float *>(list + (args.entries + 3) / 4 * 4);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ffn = args.ffn, hidden = args.hidden;
    const int split = blockIdx.x % args.splits, first = blockIdx.x / args.splits * 128;
    const int begin = split * args.split_length, end = min(begin + args.split_length, ffn);
    const int64_t block_elements = static_cast<int64_t>(ffn) * hidden;
    const __amdgpu_buffer_rsrc_t weight =
        buffer_of(static_cast<const T *>(args.weight_2) + expert * block_elements, static_cast<uint32_t>(block_elements * 2));
    const __amdgpu_buffer_rsrc_t activation =
        buffer_of(args.activation, static_cast<uint32_t>(static_cast<int64_t>(args.entries) * ffn * 2));
    const int column = first + (lane & 15) * 8;
    const uint32_t column_offset = column < hidden ? column * 2 : kOutOfRange;
    float *pieces = args.pieces + static_cast<int64_t>(split) * args.entries * hidden;

    for (int base = 0; base < rows; base += 16 * kMaxGroups) {
        const int groups = min((rows - base + 15) / 16, kMaxGroups);
        const auto run = [&](auto constant) {
            constexpr int kGroups = decltype(constant)::value;
            uint32_t row_offset[kGroups];
#pragma unroll
            for (int g = 0; g < kGroups; ++g)
                row_offset[g] = static_cast<uint32_t>(list[min(base + g * 16 + (lane & 15), rows - 1)]) * ffn * 2;
            f32x4_t sums[8][kGroups];
#pragma unroll
            for (int i = 0; i < 8; ++i)
#pragma unroll
                for (int g = 0; g < kGroups; ++g) sums[i][g] = f32x4_t{0.f, 0.f, 0.f, 0.f};
            multiply_columns<T, kGroups>(weight, activation, column_offset, row_offset, hidden * 2, begin, end, wave, lane, sums);

            // Token group by token group, [wavefront][i][lane]; wavefront w finishes register v = w of every sum: the
            // lane's columns 8 (4 (l / 16) + w) .. + 7.
            f32x4_t *slots = reinterpret_cast<f32x4_t *>(partial);
#pragma unroll
            for (int g = 0; g < kGroups; ++g) {
#pragma unroll
                for (int i = 0; i < 8; ++i) slots[(wave * 8 + i) * 64 + lane] = sums[i][g];
                __syncthreads();
                float total[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    total[i] = partial[(i * 64 + lane) * 4 + wave];
#pragma unroll
                    for (int w = 1; w < kWaves; ++w) total[i] += partial[((w * 8 + i) * 64 + lane) * 4 + wave];
                }
                const int row = base + g * 16 + (lane & 15), h = first + 8 * (4 * (lane >> 4) + wave);
                if (row < rows && h < hidden) {
                    f32x4_t *target = reinterpret_cast<f32x4_t *>(pieces + static_cast<int64_t>(list[row]) * hidden + h);
                    target[0] = f32x4_t{total[0], total[1], total[2], total[3]};
                    target[1] = f32x4_t{total[4], total[5], total[6], total[7]};
                }
                __syncthreads();
            }
        };
        if (kMaxGroups == 1 || groups == 1) run(std::integral_constant<int, 1>{});
        else if (kMaxGroups == 2 || groups == 2) run(std::integral_constant<int, (kMaxGroups < 2 ? kMaxGroups : 2)>{});
        else run(std::integral_constant<int, kMaxGroups>{});
    }
}

// ---- combine -------------------------------------------------------------------------------------------
// out[t, :] = sum over the slots j of scores[t, j] * (sum over the pieces), four columns per thread. The time is that of the
// loads that wait for one another: a token's experts and scores come at once, a lane each, while the pieces of all its slots are
// on their way, 16 at a time. (Slot by slot, the pieces after the slot's expert, eight columns per thread: 7.2 us for 96 tokens
// of 8 slots, 4.7 here; 5.7 and 4.8 for one token, 2 slots of 16 pieces.)
template <typename T>
__global__ __launch_bounds__(kThreads) void few_tokens_combine_kernel(Args args) {
    const int token = blockIdx.y, column = (blockIdx.x * kThreads + threadIdx.x) * 4, lane = threadIdx.x & 63;
    const bool exists = column < args.hidden;
    const int64_t piece_stride = static_cast<int64_t>(args.entries) * args.hidden;
    f32x4_t sum = {0.f, 0.f, 0.f, 0.f};
    for (int first = 0; first < args.slots; first += 64) {
        const int slots = min(args.slots - first, 64), entry = token * args.slots + first;
        const int64_t expert = lane < slots ? args.top_experts[entry + lane] : -1;
        const float lane_score = lane < slots ? args.scores[entry + lane] : 0.f;
        const float *pieces = args.pieces + static_cast<int64_t>(entry) * args.hidden + column;
        constexpr int kBatch = 16;
        f32x4_t value = {0.f, 0.f, 0.f, 0.f};
        int load_slot = 0, load_piece = 0, slot = 0, piece = 0;
        while (slot < slots) {
            f32x4_t loaded[kBatch];
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                loaded[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
                if (load_slot < slots && exists)
                    loaded[i] = *reinterpret_cast<const f32x4_t *>(pieces + load_piece * piece_stride + static_cast<int64_t>(load_slot) * args.hidden);
                if (++load_piece == args.splits) load_piece = 0, ++load_slot;
            }
            const uint64_t taken = __ballot(expert >= 0 && expert < args.experts);  // of the others nothing was written
#pragma unroll
            for (int i = 0; i < kBatch; ++i) {
                value += loaded[i];
                if (++piece == args.splits) {  // wave-uniform; past the last slot nothing is added
                    const float score = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, lane_score), slot & 63));
                    if (slot < slots && (taken >> slot & 1)) sum += score * value;
                    value = f32x4_t{0.f, 0.f, 0.f, 0.f};
                    piece = 0, ++slot;
                }
            }
        }
    }
    if (!exists) return;
    struct alignas(8) Four {
        T v[4];
    } result;
#pragma unroll
    for (int c = 0; c < 4; ++c) result.v[c] = from_float<T>(sum[c]);
    *reinterpret_cast<Four *>(static_cast<T *>(args.out) + static_cast<int64_t>(token) * args.hidden + column) = result;
}

// Workgroup rows: one per expert, or one per entry where there are fewer entries than experts.
static int workgroup_rows(const Args &args) { return args.by_entry ? args.entries : args.experts; }

// Pieces of layer 2's reduction: enough workgroups for four per CU, pieces of at least two chunks per wavefront.
static void plan_splits(Args &args) {
    const int workgroups = min(args.entries, args.experts) * ((args.hidden + 127) / 128);
    const int wanted = (4 * 256 + workgroups - 1) / workgroups, most = max(args.ffn / (2 * kWaves * 32), 1);
    const int splits = max(1, min(wanted, most));
    args.split_length = (args.ffn + splits * kWaves * 32 - 1) / (splits * kWaves * 32) * (kWaves * 32);
    args.splits = (args.ffn + args.split_length - 1) / args.split_length;
}

static size_t activation_bytes(const Args &args) { return (static_cast<size_t>(args.entries) * args.ffn * 2 + 255) / 256 * 256; }

template <typename T, bool kGated, int kSets, int kMaxGroups>
static void launch_layer_1(const Args &args, int list_bytes, hipStream_t stream) {
    constexpr int kOutputs = (kGated ? kSets / 2 : kSets) * 16;
    few_tokens_layer_1_kernel<T, kGated, kSets, kMaxGroups>
        <<<dim3((args.ffn + kOutputs - 1) / kOutputs, workgroup_rows(args)), kThreads, list_bytes + kWaves * kSets * 4096, stream>>>(args);
}

template <typename T, int kSets, int kMaxGroups>
static void launch(const Args &args, bool gated, hipStream_t stream) {
    const int list_bytes = (args.entries + 3) / 4 * 16;
    if (gated) launch_layer_1<T, true, kSets, kMaxGroups>(args, list_bytes, stream);
    else launch_layer_1<T, false, kSets, kMaxGroups>(args, list_bytes, stream);
    const dim3 grid_2((args.hidden + 127) / 128 * args.splits, workgroup_rows(args));
    few_tokens_layer_2_kernel<T, kMaxGroups><<<grid_2, kThreads, list_bytes + kWaves * 8 * 64 * 16, stream>>>(args);
    const dim3 grid_3((args.hidden / 4 + kThreads - 1) / kThreads, args.tokens);
    few_tokens_combine_kernel<T><<<grid_3, kThreads, 0, stream>>>(args);
}

// More token groups at a time read the weights fewer times for experts with many rows and cost registers, i.e. loads in
// flight, for those with few; the line is drawn by the mean number of rows per expert, which is all the host knows.
// Whole pass in us, groups 1 / 2 / 4: 8 of 128 experts, 2048 x 768: 6 rows 213 / 231 / 245, 12 rows 257 / 256 / 263, 24
// rows 430 / 319 / 321; 2 of 8 experts, 4096 x 14336: 8 rows 434 / 434 / 472, 16 rows 674 / 471 / 492, 24 rows 901 / 533
// / 538, 32 rows 1187 / 829 / 621. Weight rows per workgroup, 32 / 64: with long rows (4096) and one group 380 / 402 us
// at 2 rows, with rows of 2048 228 / 213 at 6 rows; four groups 823 / 709 at 48 rows.
template <typename T>
static void launch_groups(const Args &args, bool gated, hipStream_t stream) {
    const int mean_rows = (args.entries + args.experts - 1) / args.experts;
    if (mean_rows <= 10) {
        if (args.hidden > 2048) launch<T, 2, 1>(args, gated, stream);
        else launch<T, 4, 1>(args, gated, stream);
    } else if (mean_rows <= 24) {
        launch<T, 2, 2>(args, gated, stream);
    } else {
        launch<T, 4, 4>(args, gated, stream);
    }
}

constexpr int64_t kMaxEntries = 4096;  // the list in LDS, and the scan of every workgroup

static bool make_args(Args &args, int64_t tokens, int64_t slots, int64_t hidden, int64_t ffn, int64_t experts, bool gated) {
    if (tokens <= 0 || slots <= 0 || hidden <= 0 || ffn <= 0 || experts <= 0) return false;
    if (tokens > kMaxEntries || slots > kMaxEntries || tokens * slots > kMaxEntries || experts > 65535) return false;
    if (hidden % 8 != 0 || ffn % 8 != 0 || hidden > (1 << 20) || ffn > (1 << 20)) return false;
    // 32-bit byte offsets inside an expert's weights and inside the rows.
    if (ffn * (gated ? 2 : 1) * hidden * 2 >= (int64_t(1) << 32) - 256 || tokens * slots * max(hidden, ffn) * 2 >= (int64_t(1) << 32) - 256)
        return false;
    args.tokens = static_cast<int>(tokens), args.slots = static_cast<int>(slots), args.hidden = static_cast<int>(hidden);
    args.ffn = static_cast<int>(ffn), args.experts = static_cast<int>(experts);
    args.entries = args.tokens * args.slots;
    args.by_entry = args.entries < args.experts;
    plan_splits(args);
    return true;
}

}  // namespace few

}  // namespace fm

using namespace fm;

extern "C" size_t fm_few_tokens_workspace_size(int64_t num_tokens, int64_t slots_per_token, int64_t hidden, int64_t ffn,
                                               int64_t num_experts, int gated, int dtype) {
    few::Args args{};
    if ((dtype != FM_DTYPE_BF16 && dtype != FM_DTYPE_F16) ||
        !few::make_args(args, num_tokens, slots_per_token, hidden, ffn, num_experts, gated != 0))
        return 0;
    return few::activation_bytes(args) + sizeof(float) * static_cast<size_t>(args.splits) * args.entries * args.hidden;
}

extern "C" int fm_few_tokens_forward(const void *input, const void *top_experts, const void *scores, const void *weight_1,
                                     const void *weight_2, void *output, int64_t num_tokens, int64_t slots_per_token,
                                     int64_t hidden, int64_t ffn, int64_t num_experts, int gated, int activation,
                                     int dtype, void *workspace, size_t workspace_size, void *stream) {
    const char *name = "fm_few_tokens_forward";
    FM_REQUIRE(activation >= FM_ACT_GELU && activation <= FM_ACT_IDENTITY, "%s: bad activation %d", name, activation);
    const size_t needed = fm_few_tokens_workspace_size(num_tokens, slots_per_token, hidden, ffn, num_experts, gated, dtype);
    if (needed == 0)
        return fail(FM_ERR_UNSUPPORTED, "%s: needs bf16/fp16, hidden and ffn sizes that are multiples of 8 and at most %lld "
                    "(token, slot) pairs", name, static_cast<long long>(few::kMaxEntries));
    FM_REQUIRE(input && top_experts && scores && weight_1 && weight_2 && output, "%s: null tensor", name);
    FM_REQUIRE(aligned16(input) && aligned16(weight_1) && aligned16(weight_2) && aligned16(output), "%s: misaligned tensor", name);
    FM_REQUIRE(workspace && aligned16(workspace) && workspace_size >= needed, "%s: workspace of %zu bytes (16-byte aligned) needed, "
               "got %zu", name, needed, workspace_size);
    few::Args args{};
    few::make_args(args, num_tokens, slots_per_token, hidden, ffn, num_experts, gated != 0);
    args.x = input;
    args.top_experts = static_cast<const int64_t *>(top_experts);
    args.scores = static_cast<const float *>(scores);
    args.weight_1 = weight_1;
    args.weight_2 = weight_2;
    args.activation = workspace;
    args.pieces = reinterpret_cast<float *>(static_cast<char *>(workspace) + few::activation_bytes(args));
    args.out = output;
    args.activation_type = activation;
    if (dtype == FM_DTYPE_BF16) few::launch_groups<bf16_t>(args, gated != 0, static_cast<hipStream_t>(stream));
    else few::launch_groups<f16_t>(args, gated != 0, static_cast<hipStream_t>(stream));
    return check_launch(name);
}
