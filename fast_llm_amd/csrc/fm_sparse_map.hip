// Routing: build the sparse map (expert histogram -> padded expert offsets -> stable row of every
// (token, slot) pair) with integer arithmetic only, so the result is bit-exact and run-to-run identical.
//
// Two small launches over the flattened `top_experts` (M = tokens * experts_per_token entries):
//   1. sparse_map_histogram_kernel: one workgroup per 1024 entries (at most 256 workgroups). Each wavefront finds,
//      with ceil(log2 E) ballots, the set of lanes that hold the same expert ("match-any"); the lowest lane of each
//      set adds the set size to an LDS histogram. The workgroup writes its E counts to the workspace.
//   2. sparse_map_rows_kernel: same partition. Every workgroup adds up all counts and those before its own, and an LDS
//      scan of the padded totals gives expert_ends, expert_pad_begins and the first row of every expert. Rank inside
//      the wavefront = popcount of the match set below the lane; rank inside the workgroup adds an LDS prefix over the
//      16 wavefronts; the global stable rank adds the counts before. row = begin[e] + rank.
// Ranks follow the flattened index order, i.e. the order of a stable sort by expert
// (reference: fast_llm/functional/triton/sparse_copy.py:249-254).
#include "fm_common.h"
#include "fm_router_layout.h"

#include <mutex>

namespace fm {

constexpr int kMapBlock = 1024;  // entries (= threads) per workgroup
constexpr int kMapWaves = kMapBlock / 64;
constexpr int kMapMaxExperts = 1024;
constexpr int kMapMaxBlocks = 256;   // workgroups: every one of them reads the counts of all
constexpr int kMapCountBatch = 16;   // counts a thread requests at a time

__device__ __forceinline__ int log2_ceil(int value) {
    int bits = 0;
    while ((1 << bits) < value) ++bits;
    return bits;
}

// Lanes of this wavefront whose (valid) expert equals this lane's. Undefined for invalid lanes.
__device__ __forceinline__ uint64_t match_expert(int expert, bool valid, int num_bits) {
    uint64_t same = __ballot(valid);
    for (int bit = 0; bit < num_bits; ++bit) {
        const bool set = (expert >> bit) & 1;
        const uint64_t with_bit = __ballot(valid && set);
        same &= set ? with_bit : ~with_bit;
    }
    return same;
}

__global__ __launch_bounds__(kMapBlock) void sparse_map_histogram_kernel(const int64_t *__restrict__ top_experts,
                                                                         int64_t num_entries, int64_t entries_per_block,
                                                                         int num_experts,
                                                                         int32_t *__restrict__ block_counts) {
    extern __shared__ int32_t lds_counts[];  // [num_experts]
    for (int e = threadIdx.x; e < num_experts; e += kMapBlock) lds_counts[e] = 0;
    __syncthreads();

    const int64_t first = static_cast<int64_t>(blockIdx.x) * entries_per_block;
    const int64_t last = min(first + entries_per_block, num_entries);
    const int lane = threadIdx.x & 63;
    for (int64_t chunk = first; chunk < last; chunk += kMapBlock) {
        const int64_t entry = chunk + threadIdx.x;
        const int64_t expert64 = entry < last ? top_experts[entry] : -1;
        const bool valid = expert64 >= 0 && expert64 < num_experts;
        const int expert = valid ? static_cast<int>(expert64) : 0;
        const uint64_t same = match_expert(expert, valid, log2_ceil(num_experts));
        if (valid && (same & ((1ull << lane) - 1)) == 0) atomicAdd(&lds_counts[expert], __popcll(same));
    }
    __syncthreads();

    int32_t *out = block_counts + static_cast<int64_t>(blockIdx.x) * num_experts;
    for (int e = threadIdx.x; e < num_experts; e += kMapBlock) out[e] = lds_counts[e];
}

// Workgroup b ranks the entries [b * entries_per_block, (b + 1) * entries_per_block) of the flattened `top_experts`,
// 1024 at a time, given how many entries of every expert each workgroup's range has (`block_counts[workgroup][expert]`).
// Every workgroup adds up the counts of all workgroups by itself, all of them and those of the workgroups before it,
// and scans the padded totals over the experts: 128 KiB from L2 at 256 workgroups and 128 experts, requested 16 loads
// at a time by all threads. A kernel of one workgroup in between, one thread per expert walking down the workgroups,
// was a serial chain of memory latencies: with 1024 workgroups, 16384 tokens and 8 of 128 experts it took 221 us, and
// this kernel 8; both now take 12.
// kFinish: the first workgroup makes the router's sums instead (`finish_router`), which nothing here waits for: as a launch of their
// own they took 5 (8 experts) to 17 us (128).
template <bool kFinish>
__global__ __launch_bounds__(kMapBlock) void sparse_map_rows_kernel(
    const int64_t *__restrict__ top_experts, int64_t num_entries, int64_t entries_per_block, int num_experts,
    const int32_t *__restrict__ block_counts, int64_t pad_to_multiple, int index_dtype, void *__restrict__ sparse_rows,
    void *__restrict__ expert_ends, void *__restrict__ expert_pad_begins, RouterFinish finish) {
    static_assert(kMapMaxExperts <= kMapBlock, "thread e keeps the running count of expert e in a register");
    // [kMapWaves][num_experts] counts per wavefront: 64 KiB at 1024 experts. Before the first of them, in the same place:
    // partial sums [2][kMapBlock], sums [2][num_experts] and the scan's wavefront totals.
    extern __shared__ __attribute__((aligned(16))) int32_t lds_wave_counts[];
    if constexpr (kFinish) {
        static_assert(kFinishThreads == kMapBlock, "one workgroup of either kind");
        if (blockIdx.x == 0) return finish_router(finish, *reinterpret_cast<FinishLds *>(lds_wave_counts));
    }
    const int block = static_cast<int>(blockIdx.x) - (kFinish ? 1 : 0), num_blocks = static_cast<int>(gridDim.x) - (kFinish ? 1 : 0);
    int32_t *lds_parts = lds_wave_counts, *lds_totals = lds_parts + 2 * kMapBlock;
    int64_t *lds_wave_totals = reinterpret_cast<int64_t *>(lds_totals + 2 * num_experts);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int num_bits = log2_ceil(num_experts);

    // Counts of all workgroups and of those before this one, all experts at once: the threads of a column share the
    // workgroups, eight or more each. (64 experts at a time, two barriers each: one token of 1024 experts 35 us, now
    // 17; 16384 tokens of 16 of them 45, now 37; 8 of 512 25, now 17.)
    const int columns = 1 << max(num_bits, 3);
    const int column = threadIdx.x & (columns - 1), part = threadIdx.x / columns;
    const int per_part = max((num_blocks * columns + kMapBlock - 1) / kMapBlock, 8);
    const int parts = (num_blocks + per_part - 1) / per_part;
    int32_t all = 0, before = 0;
    for (int i0 = 0; i0 < per_part; i0 += kMapCountBatch) {
        int32_t here[kMapCountBatch];
#pragma unroll
        for (int i = 0; i < kMapCountBatch; ++i) {
            const int b = part * per_part + i0 + i;
            here[i] = i0 + i < per_part && b < num_blocks && column < num_experts
                          ? block_counts[static_cast<int64_t>(b) * num_experts + column] : 0;
        }
#pragma unroll
        for (int i = 0; i < kMapCountBatch; ++i) {
            all += here[i];
            if (part * per_part + i0 + i < block) before += here[i];
        }
    }
    lds_parts[threadIdx.x] = all;
    lds_parts[kMapBlock + threadIdx.x] = before;
    __syncthreads();
    for (int i = threadIdx.x; i < 2 * columns; i += kMapBlock) {
        const int which = i / columns, e = i & (columns - 1);
        int32_t total = 0;
        for (int p = 0; p < parts; ++p) total += lds_parts[which * kMapBlock + p * columns + e];
        if (e < num_experts) lds_totals[which * num_experts + e] = total;
    }
    __syncthreads();

    // Inclusive scan of the padded counts over the experts: wavefront scan, then the wavefront totals.
    const int own_expert = threadIdx.x;
    const int64_t count = own_expert < num_experts ? lds_totals[own_expert] : 0;
    const int32_t earlier = own_expert < num_experts ? lds_totals[num_experts + own_expert] : 0;
    const int64_t padded = (count + pad_to_multiple - 1) / pad_to_multiple * pad_to_multiple;
    int64_t inclusive = padded;
#pragma unroll
    for (int offset = 1; offset < 64; offset <<= 1) {
        const int64_t other = __shfl_up(inclusive, offset, 64);
        if (lane >= offset) inclusive += other;
    }
    if (lane == 63) lds_wave_totals[wave] = inclusive;
    __syncthreads();
    for (int w = 0; w < wave; ++w) inclusive += lds_wave_totals[w];
    __syncthreads();  // the chunks' counts take the place of the sums
    // Rows handed out so far to expert threadIdx.x (there are at most as many experts as threads).
    int32_t running = 0;
    if (own_expert < num_experts) {
        const int64_t expert_begin = inclusive - padded;
        running = static_cast<int32_t>(expert_begin) + earlier;
        if (block == 0) {
            store_index(expert_ends, index_dtype, own_expert, inclusive);
            store_index(expert_pad_begins, index_dtype, own_expert, expert_begin + count);
        }
    }

    const int64_t first = static_cast<int64_t>(block) * entries_per_block;
    const int64_t last = min(first + entries_per_block, num_entries);
    for (int64_t chunk = first; chunk < last; chunk += kMapBlock) {
        for (int i = threadIdx.x; i < kMapWaves * num_experts; i += kMapBlock) lds_wave_counts[i] = 0;
        __syncthreads();

        const int64_t entry = chunk + threadIdx.x;
        int64_t expert64 = entry < last ? top_experts[entry] : -1;
        const bool valid = expert64 >= 0 && expert64 < num_experts;
        const int expert = valid ? static_cast<int>(expert64) : 0;
        const uint64_t same = match_expert(expert, valid, num_bits);
        const int rank_in_wave = __popcll(same & ((1ull << lane) - 1));
        if (valid && rank_in_wave == 0) lds_wave_counts[wave * num_experts + expert] = __popcll(same);
        __syncthreads();

        // Exclusive prefix over the wavefronts of the workgroup, per expert, in place, on top of the running count.
        if (own_expert < num_experts) {
#pragma unroll
            for (int w = 0; w < kMapWaves; ++w) {
                const int32_t here = lds_wave_counts[w * num_experts + own_expert];
                lds_wave_counts[w * num_experts + own_expert] = running;
                running += here;
            }
        }
        __syncthreads();

        if (entry < last) {
            int64_t row = -1;
            if (valid) row = static_cast<int64_t>(lds_wave_counts[wave * num_experts + expert]) + rank_in_wave;
            store_index(sparse_rows, index_dtype, entry, row);
        }
        __syncthreads();
    }
}

// Dynamic LDS of the kernel above: the per-wavefront counts, and before them the sums.
static inline size_t map_rows_lds_bytes(int num_experts) {
    const size_t counts = static_cast<size_t>(kMapWaves) * num_experts;
    const size_t sums = 2 * kMapBlock + 2 * static_cast<size_t>(num_experts) + 2 * kMapWaves;
    return sizeof(int32_t) * (counts > sums ? counts : sums);
}

// Entries per workgroup: whole 1024s, few enough workgroups that each can read all the others' counts.
static inline int64_t map_entries_per_block(int64_t num_entries) {
    const int64_t chunks = (num_entries + kMapBlock - 1) / kMapBlock;
    return (chunks + kMapMaxBlocks - 1) / kMapMaxBlocks * kMapBlock;
}
static inline int64_t map_num_blocks(int64_t num_entries) {
    const int64_t per_block = map_entries_per_block(num_entries);
    return per_block > 0 ? (num_entries + per_block - 1) / per_block : 0;
}

}  // namespace fm

extern "C" size_t fm_sparse_map_workspace_size(int64_t num_rows_dense, int64_t num_experts_per_token,
                                               int64_t num_experts) {
    if (num_rows_dense < 0 || num_experts_per_token < 0 || num_experts < 0) return 0;
    const int64_t blocks = fm::map_num_blocks(num_rows_dense * num_experts_per_token);
    const size_t bytes = static_cast<size_t>((blocks + 1) * num_experts) * sizeof(int32_t);
    return (bytes + 255) / 256 * 256 + 256;
}

namespace fm {

// The two launches; `workspace` holds fm_sparse_map_workspace_size(...) bytes.
static int run_sparse_map(const char *name, const int64_t *top_experts, int64_t num_rows_dense,
                          int64_t num_experts_per_token, int64_t num_experts, int64_t pad_to_multiple, int index_dtype,
                          void *sparse_rows, void *expert_ends, void *expert_pad_begins, void *workspace,
                          hipStream_t stream) {
    const int64_t num_entries = num_rows_dense * num_experts_per_token;
    // At least one workgroup: without entries it still lays out the (empty) experts.
    const int blocks = static_cast<int>(max(map_num_blocks(num_entries), int64_t(1)));
    const int64_t entries_per_block = map_entries_per_block(num_entries);
    const int experts = static_cast<int>(num_experts);
    int32_t *block_counts = static_cast<int32_t *>(workspace);
    sparse_map_histogram_kernel<<<blocks, kMapBlock, experts * sizeof(int32_t), stream>>>(
        top_experts, num_entries, entries_per_block, experts, block_counts);
    sparse_map_rows_kernel<false><<<blocks, kMapBlock, map_rows_lds_bytes(experts), stream>>>(
        top_experts, num_entries, entries_per_block, experts, block_counts, pad_to_multiple, index_dtype, sparse_rows,
        expert_ends, expert_pad_begins, RouterFinish());
    return check_launch(name);
}

static int check_sparse_map_arguments(const char *name, const int64_t *top_experts, int64_t num_rows_dense,
                                      int64_t num_experts_per_token, int64_t num_experts, int64_t pad_to_multiple,
                                      int index_dtype, void *sparse_rows, void *expert_ends, void *expert_pad_begins) {
    FM_REQUIRE(num_rows_dense >= 0 && num_experts_per_token >= 0, "%s: negative shape", name);
    FM_REQUIRE(num_experts >= 1 && num_experts <= kMapMaxExperts, "%s: num_experts=%lld outside [1, %d]", name,
               (long long)num_experts, kMapMaxExperts);
    FM_REQUIRE(pad_to_multiple >= 1, "%s: pad_to_multiple=%lld < 1", name, (long long)pad_to_multiple);
    FM_REQUIRE(valid_index_dtype(index_dtype), "%s: bad index_dtype %d", name, index_dtype);
    const int64_t num_entries = num_rows_dense * num_experts_per_token;
    const int64_t max_rows = num_entries + num_experts * pad_to_multiple;
    FM_REQUIRE(max_rows < (int64_t(1) << 31), "%s: %lld padded rows overflow int32", name, (long long)max_rows);
    FM_REQUIRE(index_dtype != FM_INDEX_I16 || max_rows <= 32767 + pad_to_multiple,
               "%s: %lld padded rows do not fit int16", name, (long long)max_rows);
    FM_REQUIRE(expert_ends && expert_pad_begins, "%s: null output", name);
    FM_REQUIRE(num_entries == 0 || (top_experts && sparse_rows), "%s: null top_experts/sparse_rows", name);
    return FM_OK;
}

}  // namespace fm

extern "C" int fm_sparse_map(const int64_t *top_experts, int64_t num_rows_dense, int64_t num_experts_per_token,
                             int64_t num_experts, int64_t pad_to_multiple, int index_dtype, void *sparse_rows,
                             void *expert_ends, void *expert_pad_begins, void *workspace, size_t workspace_size,
                             void *stream) {
    using namespace fm;
    if (int status = check_sparse_map_arguments("fm_sparse_map", top_experts, num_rows_dense, num_experts_per_token,
                                                num_experts, pad_to_multiple, index_dtype, sparse_rows, expert_ends,
                                                expert_pad_begins))
        return status;
    FM_REQUIRE(workspace, "fm_sparse_map: null workspace");
    FM_REQUIRE(workspace_size >= fm_sparse_map_workspace_size(num_rows_dense, num_experts_per_token, num_experts),
               "fm_sparse_map: workspace of %zu bytes is too small", workspace_size);
    FM_REQUIRE(aligned16(workspace), "fm_sparse_map: workspace must be 16-byte aligned");
    return run_sparse_map("fm_sparse_map", top_experts, num_rows_dense, num_experts_per_token, num_experts,
                          pad_to_multiple, index_dtype, sparse_rows, expert_ends, expert_pad_begins, workspace,
                          static_cast<hipStream_t>(stream));
}

// ---- the map from the router's own counts ------------------------------------------------------------------
extern "C" size_t fm_sparse_map_from_router_workspace_size(int64_t num_tokens, int64_t num_experts) {
    return num_tokens < 0 || num_experts < 0 ? 0 : 256;  // the counts are the router's
}

int fm::sparse_map_from_router(const int64_t *top_experts, const void *router_workspace, size_t router_workspace_size,
                               int64_t num_tokens, int64_t num_experts, int64_t experts_per_token, int64_t shared_experts,
                               int64_t pad_to_multiple, int index_dtype, void *sparse_rows, void *expert_ends,
                               void *expert_pad_begins, void *workspace, size_t workspace_size, const RouterFinish *finish,
                               void *stream_) {
    const char *name = "fm_sparse_map_from_router";
    FM_REQUIRE(shared_experts >= 0 && experts_per_token > 0 && num_experts > shared_experts,
               "%s: %lld experts of which %lld shared, %lld per token", name, (long long)num_experts,
               (long long)shared_experts, (long long)experts_per_token);
    const int64_t slots = shared_experts + experts_per_token;
    if (int status = check_sparse_map_arguments(name, top_experts, num_tokens, slots, num_experts, pad_to_multiple,
                                                index_dtype, sparse_rows, expert_ends, expert_pad_begins))
        return status;
    FM_REQUIRE(num_tokens > 0, "%s: no tokens (the router does not run on none either)", name);
    FM_REQUIRE(router_workspace && router_workspace_size >= router_counts_bytes(num_tokens, num_experts),
               "%s: the router workspace must be the buffer fm_router_forward filled, got %zu bytes", name,
               router_workspace_size);
    FM_REQUIRE(workspace && aligned16(workspace) &&
                   workspace_size >= fm_sparse_map_from_router_workspace_size(num_tokens, num_experts),
               "%s: workspace of %zu bytes is null, misaligned or too small", name, workspace_size);
    const int experts = static_cast<int>(num_experts);
    size_t lds_bytes = map_rows_lds_bytes(experts);
    if (finish != nullptr && lds_bytes < sizeof(FinishLds)) lds_bytes = sizeof(FinishLds);
    const auto kernel = finish != nullptr ? sparse_map_rows_kernel<true> : sparse_map_rows_kernel<false>;
    kernel<<<router_blocks(num_tokens) + (finish != nullptr ? 1 : 0), kMapBlock, lds_bytes, static_cast<hipStream_t>(stream_)>>>(
        top_experts, num_tokens * slots, router_tokens_per_block(num_tokens) * slots, experts,
        static_cast<const int32_t *>(router_workspace), pad_to_multiple, index_dtype, sparse_rows, expert_ends,
        expert_pad_begins, finish != nullptr ? *finish : RouterFinish());
    return check_launch(name);
}

extern "C" int fm_sparse_map_from_router(const int64_t *top_experts, const void *router_workspace,
                                         size_t router_workspace_size, int64_t num_tokens, int64_t num_experts,
                                         int64_t experts_per_token, int64_t shared_experts, int64_t pad_to_multiple,
                                         int index_dtype, void *sparse_rows, void *expert_ends,
                                         void *expert_pad_begins, void *workspace, size_t workspace_size,
                                         void *stream) {
    return fm::sparse_map_from_router(top_experts, router_workspace, router_workspace_size, num_tokens, num_experts, experts_per_token,
                                      shared_experts, pad_to_multiple, index_dtype, sparse_rows, expert_ends, expert_pad_begins,
                                      workspace, workspace_size, nullptr, stream);
}

// ---- the same map without any allocation ----------------------------------------------------------------
// The per-workgroup counts live in a fixed array in device memory that is part of the loaded code object: every GPU
// the library runs on holds its own copy, at its own address, until the process ends.
namespace fm {

constexpr size_t kStaticScratchBytes = FM_SPARSE_MAP_STATIC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

constexpr int kMaxDevices = 64;

// Device address of this device's copy of `scratch`, looked up once per device with that device current. In host
// code the array's name is not a device address; only the pointer returned here may go to kernels.
// `stream` (may be null: the current device's default stream) must belong to the current device: the kernels run where
// the stream lives, and each device has its own copy of the array.
static int static_scratch_of_current_device(hipStream_t stream, void **pointer) {
    static std::mutex mutex;
    static void *addresses[kMaxDevices] = {};
    int device = -1;
    hipError_t error = hipGetDevice(&device);
    if (error != hipSuccess) return fail(FM_ERR_LAUNCH, "fm_sparse_map_static: hipGetDevice: %s", hipGetErrorString(error));
    int stream_device = device;
    if (stream != nullptr && hipStreamGetDevice(stream, &stream_device) == hipSuccess && stream_device != device)
        return fail(FM_ERR_INVALID_ARGUMENT,
                    "fm_sparse_map_static: the stream belongs to device %d but device %d is current; make the stream's "
                    "device current before the call",
                    stream_device, device);
    if (device < 0 || device >= kMaxDevices)
        return fail(FM_ERR_UNSUPPORTED, "fm_sparse_map_static: device %d outside [0, %d)", device, kMaxDevices);
    std::lock_guard<std::mutex> lock(mutex);
    if (addresses[device] == nullptr) {
        void *address = nullptr;
        error = hipGetSymbolAddress(&address, HIP_SYMBOL(scratch));
        if (error != hipSuccess || address == nullptr)
            return fail(FM_ERR_LAUNCH, "fm_sparse_map_static: hipGetSymbolAddress: %s", hipGetErrorString(error));
        addresses[device] = address;
    }
    *pointer = addresses[device];
    return FM_OK;
}

}  // namespace fm

extern "C" size_t fm_sparse_map_static_scratch_size(void) { return fm::kStaticScratchBytes; }

extern "C" int fm_sparse_map_static(const int64_t *top_experts, int64_t num_rows_dense, int64_t num_experts_per_token,
                                    int64_t num_experts, int64_t pad_to_multiple, int index_dtype, void *sparse_rows,
                                    void *expert_ends, void *expert_pad_begins, void *stream) {
    using namespace fm;
    if (int status = check_sparse_map_arguments("fm_sparse_map_static", top_experts, num_rows_dense,
                                                num_experts_per_token, num_experts, pad_to_multiple, index_dtype,
                                                sparse_rows, expert_ends, expert_pad_begins))
        return status;
    const size_t needed = fm_sparse_map_workspace_size(num_rows_dense, num_experts_per_token, num_experts);
    if (needed > kStaticScratchBytes)
        return fail(FM_ERR_UNSUPPORTED,
                    "fm_sparse_map_static: %lld x %lld entries over %lld experts need %zu bytes of scratch, the fixed "
                    "array holds %zu; use fm_sparse_map with a workspace",
                    (long long)num_rows_dense, (long long)num_experts_per_token, (long long)num_experts, needed,
                    kStaticScratchBytes);
    void *workspace = nullptr;
    if (int status = static_scratch_of_current_device(static_cast<hipStream_t>(stream), &workspace)) return status;
    // Nothing to clear: the histogram kernel writes every count that the other kernel reads.
    return run_sparse_map("fm_sparse_map_static", top_experts, num_rows_dense, num_experts_per_token, num_experts,
                          pad_to_multiple, index_dtype, sparse_rows, expert_ends, expert_pad_begins, workspace,
                          static_cast<hipStream_t>(stream));
}
