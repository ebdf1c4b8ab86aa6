// Weight gradients of experts of few rows on the gfx950 matrix cores (row-sparse product, bf16 / fp16 operands and results, fp32
// accumulation): out_e [M_s, N] (+)= lhs[rows of e, M_s]^T x rhs[rows of e, N], in tiles of 128 x 256.
//
// With some hundred rows per expert such a product is little but its result: what bounds it is the rate at which that can be written
// (5.5 to 6.2 TB/s for tiles like these). Where a wavefront both loads and stores, its loads wait behind its stores, on the way and in
// `vmcnt`; a tile at a time, the loads, multiplications and stores of a CU follow one another. Here one workgroup per CU has
//   * four wavefronts that only load, straight from memory into LDS, four slices of 32 rows ahead of the multiplications and across
//     the ends of tiles: on their own wavefronts they wait for no store. Four, because one does not issue them fast enough;
//   * eight that multiply 64 x 64 of the tile each and store, and never wait for memory;
//   * the rhs slices of up to five (160 rows) resident in LDS while the workgroup goes down the rows of the result: a tile then loads
//     its lhs slices only, a third of the bytes. With more rows both operands pass through the slots.
// 128 experts of 2048 x 768, 111 rows each: 269 and 137 us for the two gradients in tiles of 128 x 256, two workgroups per CU, 200 and 101
// here: 4 TB/s of results.
// What `out` holds, where the results are added to it, is asked for before a tile is multiplied, two of its four parts ahead: 125 rows of
// 128 experts of 2048 x 768 562 -> 529 us for both gradients, of 8 of 4096 x 14336 1271 -> 1195 (preferred experts 615 -> 609 and 1366 ->
// 1306); from 16 to 180 rows of six shapes 0.99 to 1.08 times as fast as with one part ahead, asked for after the multiplications.
// A workgroup takes items of about the same time (`Items`), so that experts of many rows are spread over the device.
// The order of a sum is that of a tile of 256 x 256: the results are the same bits.
#include <atomic>
#include <type_traits>
#include "fm_gemm_common.h"
#include "fm_partition.h"

namespace fm {

namespace row_panel {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4_t;
typedef __attribute__((__vector_size__(2 * sizeof(uint32_t)))) uint32_t u32x2_t;
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short i16x4_t;

constexpr int kTileM = 128, kTileN = 256, kBK = 32;
constexpr int kBlocks = 2;  // a wavefront multiplies 64 x 64, in 32 x 32 accumulators
constexpr int kMultiplying = 8, kLoading = 4, kThreads = 64 * (kMultiplying + kLoading);  // wavefronts: 2 x 4 multiply a tile
constexpr int kMaxExperts = 256, kExpertRegisters = kMaxExperts / 64;
constexpr int kResident = 256;  // workgroups on the device at one time

__device__ __forceinline__ f32x16_t mfma(bf16_t, u32x4_t a, u32x4_t b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x16_t mfma(f16_t, u32x4_t a, u32x4_t b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// One operand's slice in LDS, [kBK rows][kColumns], and the loads that fill it, a quarter of the rows per loading wavefront.
template <int kColumns>
struct Operand {
    static constexpr int kBytes = kColumns * kBK * 2, kChunks = kColumns / 8;  // 16-byte chunks per row
    static constexpr int kRowsPerLoad = 64 / kChunks, kLoads = kBK / kLoading / kRowsPerLoad;
    static constexpr int kOffsets = 4 / kRowsPerLoad;  // the swizzle repeats after four rows
    static constexpr uint32_t kOutOfRange = 0x80000000u, kRange = 0x7fffffffu;

    // Where chunk `c` of row `k` sits among the row's chunks: the four rows x 32 bytes that a transpose read takes from one
    // column of chunks then lie in different banks.
    static __device__ __forceinline__ int swizzled(int k, int c) { return c ^ ((k & 3) << 2); }

    const char *base;           // wave-uniform: element (first row of the reduction, first column of the tile)
    uint32_t stride;            // bytes between rows
    uint32_t offset[kOffsets];  // per lane, bytes from the slice's first element; out of range where there is no such column
    int row;                    // of the lane's first load
    int target;                 // of the wavefront's first load in a slot

    // `valid`: columns that exist, a multiple of 8. `part`: which of the loading wavefronts.
    __device__ __forceinline__ void setup(const char *first, int64_t stride_, int valid, int part, int lane) {
        base = first;
        stride = static_cast<uint32_t>(stride_);
        row = part * (kBK / kLoading) + lane / kChunks;
        target = part * kLoads * 1024;
#pragma unroll
        for (int j = 0; j < kOffsets; ++j) {
            const int k = row + j * kRowsPerLoad, chunk = swizzled(k, lane % kChunks);
            offset[j] = chunk * 8 < valid ? static_cast<uint32_t>(k * stride_ + chunk * 16) : kOutOfRange;
        }
    }

    // Slice `slice` -> the LDS slot at byte address `slot`; rows from `rows_left` on come as zeros.
    __device__ __forceinline__ void fetch(int slot, int slice, int rows_left) const {
        const __amdgpu_buffer_rsrc_t resource = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<char *>(uniform_pointer(base + static_cast<int64_t>(slice) * kBK * stride)), 0, static_cast<int>(kRange),
            kBufferResourceFlags);
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const uint32_t lane_offset =
                row + j * kRowsPerLoad < rows_left ? offset[j % kOffsets] + j / kOffsets * 4 * stride : kOutOfRange;
            const int at = __builtin_amdgcn_readfirstlane(slot + target + j * 1024);
            asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                         :
                         : "s"(at), "v"(lane_offset), "s"(resource)
                         : "memory");
        }
    }

    // Per lane, the byte addresses (from a slot's) of the fragments of the wavefront's blocks of 32 columns from `first` on;
    // 16 rows further on is a constant. Lane s of a group of 16 supplies the address of four columns (column + 4 (s % 4) ..)
    // of row k + s / 4 and receives rows k .. k + 3 of column + s.
    static __device__ __forceinline__ void fragment_addresses(int first, int lane, int (&addresses)[kBlocks]) {
        const int s = lane & 15, group = lane >> 4, k = ((group >> 1) << 3) + (s >> 2);
#pragma unroll
        for (int i = 0; i < kBlocks; ++i) {
            const int column = first + i * 32 + ((group & 1) << 4) + ((s & 3) << 2);
            addresses[i] = k * kColumns * 2 + swizzled(k, column >> 3) * 16 + (column & 7) * 2;
        }
    }
    // Eight consecutive rows (16 step + 8 (lane / 32) ..) of the lane's column.
    static __device__ __forceinline__ u32x4_t fragment(int address, int step) {
        const uintptr_t at = static_cast<uintptr_t>(address + step * 16 * kColumns * 2);
        const i16x4_t low = __builtin_amdgcn_ds_read_tr16_b64_v4i16((FM_LDS(i16x4_t) *)at);
        const i16x4_t high = __builtin_amdgcn_ds_read_tr16_b64_v4i16((FM_LDS(i16x4_t) *)(at + 4 * kColumns * 2));
        const u32x2_t low_words = __builtin_bit_cast(u32x2_t, low), high_words = __builtin_bit_cast(u32x2_t, high);
        return u32x4_t{low_words[0], low_words[1], high_words[0], high_words[1]};
    }
};

template <int kNewest>
__device__ __forceinline__ void wait_for_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kNewest) : "memory");
}

// A lane holds, of each 32 x 32 accumulator, one row and four groups of four consecutive columns. A wavefront passes 32 rows x 128
// bytes at a time through its own LDS region and stores whole lines (half lines of 16-bit results that are added to what `out` holds:
// those stay in 32 bits until then).
constexpr int kRowBytes = 128 + 16, kStagingBytes = 32 * kRowBytes;

template <typename T, bool kAccumulate>
struct TileStore {
    typedef std::conditional_t<kAccumulate, float, T> StageT;
    typedef __attribute__((__vector_size__(4 * sizeof(StageT)))) uint32_t Group;
    static constexpr int kColumns = 128 / sizeof(StageT), kWide = kColumns / 32, kElements = 16 / sizeof(StageT);  // kWide accumulators side by side
    typedef __attribute__((__vector_size__(kElements * sizeof(T)))) uint32_t Chunk;
    static constexpr int kRounds = kBlocks * kBlocks / kWide;

    __amdgpu_buffer_rsrc_t resource;
    int64_t stride;
    int rows_valid, cols_valid, wave_m, wave_n, lane;
    Chunk previous[2][4];

    // Rows and columns that do not exist are sent out of the buffer's range.
    __device__ __forceinline__ int offset_of(int i, int first, int t) const {
        const int row = wave_m * 64 + i * 32 + t * 8 + (lane >> 3), column = (wave_n * kBlocks + first) * 32 + (lane & 7) * kElements;
        return row < rows_valid && column < cols_valid ? static_cast<int>((row * stride + column) * sizeof(T)) : static_cast<int>(0x80000000u);
    }
    __device__ __forceinline__ void request(int round) {
        const int i = round / (kBlocks / kWide), first = round % (kBlocks / kWide) * kWide;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            if constexpr (sizeof(Chunk) == 16) previous[round & 1][t] = __builtin_amdgcn_raw_buffer_load_b128(resource, offset_of(i, first, t), 0, 0);
            else previous[round & 1][t] = __builtin_amdgcn_raw_buffer_load_b64(resource, offset_of(i, first, t), 0, 0);
        }
    }
    // Asks for the first two rounds of what `out` holds: it comes while the tile is multiplied.
    __device__ __forceinline__ void begin(const char *out, int64_t stride_, int rows_valid_, int cols_valid_, int wave_m_, int wave_n_, int lane_) {
        resource = __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(uniform_pointer(out)), 0, 0x7fffffff, kBufferResourceFlags);
        stride = stride_, rows_valid = rows_valid_, cols_valid = cols_valid_, wave_m = wave_m_, wave_n = wave_n_, lane = lane_;
        if constexpr (kAccumulate) {
            request(0);
            request(1);
        }
    }
    __device__ __forceinline__ void finish(const f32x16_t (&acc)[kBlocks][kBlocks], int staging, bool streaming) {
        const int write_base = staging + (lane & 31) * kRowBytes + (lane >> 5) * 4 * sizeof(StageT);
        const int read_base = staging + (lane >> 3) * kRowBytes + (lane & 7) * 16;
#pragma unroll
        for (int round = 0; round < kRounds; ++round) {
            const int i = round / (kBlocks / kWide), first = round % (kBlocks / kWide) * kWide;
#pragma unroll
            for (int j = 0; j < kWide; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    struct {
                        StageT v[4];
                    } group;
#pragma unroll
                    for (int c = 0; c < 4; ++c) group.v[c] = from_float<StageT>(acc[i][first + j][4 * g + c]);
                    *(FM_LDS(Group) *)static_cast<uintptr_t>(write_base + (j * 32 + 8 * g) * sizeof(StageT)) = __builtin_bit_cast(Group, group);
                }
            asm volatile("" ::: "memory");  // a wavefront's own LDS accesses are carried out in order
            u32x4_t staged[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) staged[t] = *(FM_LDS(u32x4_t) *)static_cast<uintptr_t>(read_base + t * 8 * kRowBytes);
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                Chunk values;
                if constexpr (kAccumulate) {
                    struct {
                        T v[4];
                    } sums = __builtin_bit_cast(decltype(sums), previous[round & 1][t]);
                    const f32x4_t added = __builtin_bit_cast(f32x4_t, staged[t]);
#pragma unroll
                    for (int c = 0; c < 4; ++c) sums.v[c] = from_float<T>(added[c] + to_float(sums.v[c]));
                    values = __builtin_bit_cast(Chunk, sums);
                } else {
                    values = __builtin_bit_cast(Chunk, staged[t]);
                }
                const int offset = offset_of(i, first, t);
                if constexpr (sizeof(Chunk) == 16) {
                    if (streaming) __builtin_amdgcn_raw_buffer_store_b128(values, resource, offset, 0, 2);
                    else __builtin_amdgcn_raw_buffer_store_b128(values, resource, offset, 0, 0);
                } else {
                    __builtin_amdgcn_raw_buffer_store_b64(values, resource, offset, 0, 0);
                }
            }
            if constexpr (kAccumulate)
                if (round + 2 < kRounds) request(round + 2);
            asm volatile("" ::: "memory");
        }
    }
};

// LDS: slots for the slices of each operand, a staging region per wavefront.
typedef Operand<kTileM> Lhs;
typedef Operand<kTileN> Rhs;
constexpr int kSlots = 5, kRhsAt = kSlots * Lhs::kBytes, kStagingAt = kRhsAt + kSlots * Rhs::kBytes;
constexpr int kLdsBytes = kStagingAt + kMultiplying * kStagingBytes;
static_assert(kLdsBytes <= 160 * 1024, "LDS of a CU");

// A workgroup's work at one time: the rows [row, row + rows) x 256 columns of an expert's gradient.
struct Item {
    int expert, begin, count, row, rows, column;
    __device__ __forceinline__ int slices() const { return max((count + kBK - 1) / kBK, 1); }  // no rows: a slice of zeros
    __device__ __forceinline__ bool resident() const { return count <= kSlots * kBK; }  // the rhs slices stay for all tiles
};

// The work of a launch, in items of about the same time: as many for an expert as its tiles take. The time of a tile is taken to be that
// of its slices and kTileCost more. Items of whole columns are 20 % slower where one expert has a tenth of the rows (128 experts of 2048 x
// 768, 120 rows on average: 208 and 291 us, 143 and 238 so); 12 items per workgroup gain 5 % there and cost as much elsewhere.
struct Items {
    static constexpr int kTileCost = 4, kItemsPerWorkgroup = 6, kLeastItem = 24;
    int begin[kExpertRegisters], count[kExpertRegisters], items_to[kExpertRegisters];  // of an expert per lane and register
    int panels, tiles, target, next;

    // Tiles of an item of an expert with `rows` rows.
    __device__ __forceinline__ int tiles_per_item(int rows) const {
        return min(max(target / ((rows + kBK - 1) / kBK + kTileCost), 1), tiles);
    }

    __device__ __forceinline__ void load(const GemmArgs &args, int lane) {
        panels = args.tiles_n;
        tiles = static_cast<int>((args.sparse_size + kTileM - 1) / kTileM);
        int64_t cost = 0;
#pragma unroll
        for (int i = 0; i < kExpertRegisters; ++i) {
            const int e = i * 64 + lane;
            int64_t first = 0, end = 0;
            if (e < args.num_experts) {
                first = e > 0 ? max(load_index(args.expert_ends, args.index_dtype, e - 1), static_cast<int64_t>(0)) : 0;
                end = min(load_index(args.expert_pad_begins, args.index_dtype, e), args.inner);
                cost += max((end - first + kBK - 1) / kBK, static_cast<int64_t>(0)) + kTileCost;
            }
            begin[i] = static_cast<int>(first);
            count[i] = static_cast<int>(max(end - first, static_cast<int64_t>(0)));
        }
#pragma unroll
        for (int offset = 32; offset > 0; offset >>= 1) cost += __shfl_xor(cost, offset, 64);
        target = __builtin_amdgcn_readfirstlane(static_cast<int>(max(cost * tiles * panels / (kResident * kItemsPerWorkgroup), static_cast<int64_t>(kLeastItem))));
        int total = 0;
#pragma unroll
        for (int i = 0; i < kExpertRegisters; ++i) {
            const int per_item = tiles_per_item(count[i]);
            // Nothing is added where there are no rows.
            const bool wanted = i * 64 + lane < args.num_experts && (count[i] > 0 || !args.accumulate);
            int inclusive = wanted ? panels * ((tiles + per_item - 1) / per_item) : 0;
#pragma unroll
            for (int offset = 1; offset < 64; offset <<= 1) {
                const int other = __shfl_up(inclusive, offset, 64);
                if (lane >= offset) inclusive += other;
            }
            items_to[i] = total + inclusive;
            total = __builtin_amdgcn_readlane(items_to[i], 63);
        }
        // Consecutive workgroup ids go to the 8 XCDs in turn; the 32 workgroups of an XCD take consecutive items.
        next = blockIdx.x % 8 * 32 + blockIdx.x / 8;
    }

    // The next item of this workgroup. Wave-uniform.
    __device__ __forceinline__ bool take(const GemmArgs &args, Item &item) {
        const int logical = next;
        next += kResident;
        bool found = false;
#pragma unroll
        for (int i = 0; i < kExpertRegisters; ++i) {
            if (found) continue;
            const uint64_t later = __ballot(items_to[i] > logical);
            if (later == 0) continue;
            found = true;
            const int owner = __ffsll(static_cast<unsigned long long>(later)) - 1;
            item.expert = i * 64 + owner;
            item.begin = __builtin_amdgcn_readlane(begin[i], owner);
            item.count = __builtin_amdgcn_readlane(count[i], owner);
            const int per_item = tiles_per_item(item.count), parts = (tiles + per_item - 1) / per_item;
            const int in_expert = logical - (__builtin_amdgcn_readlane(items_to[i], owner) - panels * parts), part = in_expert / panels;
            const int first = part_begin(part, tiles, parts), last = part_begin(part + 1, tiles, parts);
            item.row = first * kTileM;
            item.rows = static_cast<int>(min(static_cast<int64_t>(last) * kTileM, args.sparse_size) - item.row);
            item.column = (in_expert - part * panels) * kTileN;
        }
        return found;
    }
};

// Of 16 rows of the reduction.
struct Fragments {
    u32x4_t a[kBlocks], b[kBlocks];
    __device__ __forceinline__ void read(const int (&lhs_addresses)[kBlocks], int lhs, const int (&rhs_addresses)[kBlocks], int rhs, int step) {
#pragma unroll
        for (int i = 0; i < kBlocks; ++i) a[i] = Lhs::fragment(lhs + lhs_addresses[i], step);
#pragma unroll
        for (int j = 0; j < kBlocks; ++j) b[j] = Rhs::fragment(rhs + rhs_addresses[j], step);
    }
    // Operands swapped: a lane holds one row of the tile and groups of four consecutive columns.
    template <typename T>
    __device__ __forceinline__ void multiply(f32x16_t (&acc)[kBlocks][kBlocks]) const {
#pragma unroll
        for (int i = 0; i < kBlocks; ++i)
#pragma unroll
            for (int j = 0; j < kBlocks; ++j) acc[i][j] = mfma(T(), b[j], a[i], acc[i][j]);
    }
};

__device__ __forceinline__ void clear(f32x16_t (&acc)[kBlocks][kBlocks]) {
#pragma unroll
    for (int i = 0; i < kBlocks; ++i)
#pragma unroll
        for (int j = 0; j < kBlocks; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
}

template <typename T, bool kAccumulate>
__global__ __launch_bounds__(kThreads, 1) void grouped_gemm_row_panel_kernel(GemmArgs args) {
    extern __shared__ __attribute__((aligned(1024))) char lds_generic[];
    const int lds = static_cast<int>(reinterpret_cast<uintptr_t>((FM_LDS(char) *)lds_generic));
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    Items items;
    items.load(args, lane);
    Item item;

    // The slices of an item's tiles, one tile after the other, pass through the slots: slice s sits in slot s % kSlots (a resident rhs
    // slice in that of its place in the reduction). The barrier in front of its multiplications makes it visible (the loading
    // wavefronts have waited for their loads of it) and ends the reads of slice s - 1, whose slot the loads of slice s + kSlots - 1
    // then fill.
    if (wave >= kMultiplying) {
        const int part = wave - kMultiplying;
        const int64_t lhs_stride = args.lhs_stride_inner * 2, rhs_stride = args.rhs_stride_inner * 2;
        while (items.take(args, item)) {
            const int slices = item.slices(), tiles = (item.rows + kTileM - 1) / kTileM, total = tiles * slices;
            const bool resident = item.resident();
            const char *lhs_first = static_cast<const char *>(args.lhs) + item.begin * lhs_stride + item.row * 2;
            Lhs lhs;
            Rhs rhs;
            rhs.setup(static_cast<const char *>(args.rhs) + item.begin * rhs_stride + item.column * 2, rhs_stride,
                      static_cast<int>(min(static_cast<int64_t>(kTileN), args.cols - item.column)), part, lane);
            int slot = 0, slice = 0, tile = 0;
            const auto fetch = [&]() {
                if (slice == 0) lhs.setup(lhs_first + tile * kTileM * 2, lhs_stride, item.rows - tile * kTileM, part, lane);
                const int rows_left = tile < tiles ? item.count - slice * kBK : 0;
                lhs.fetch(lds + slot * Lhs::kBytes, slice, rows_left);
                if (!resident) rhs.fetch(lds + kRhsAt + slot * Rhs::kBytes, slice, rows_left);
                slot = slot == kSlots - 1 ? 0 : slot + 1;
                if (++slice == slices) slice = 0, ++tile;
            };
            if (resident)
                for (int s = 0; s < slices; ++s) rhs.fetch(lds + kRhsAt + s * Rhs::kBytes, s, item.count - s * kBK);
#pragma unroll 1
            for (int s = 0; s < kSlots - 1; ++s) fetch();
            for (int s = 0; s < total; ++s) {
                if (resident) wait_for_loads<(kSlots - 2) * Lhs::kLoads>();
                else wait_for_loads<(kSlots - 2) * (Lhs::kLoads + Rhs::kLoads)>();
                __syncthreads();
                fetch();
            }
            wait_for_loads<0>();  // zeros on their way to the slots
            __syncthreads();      // the last slice has been multiplied: the next item's may replace it
        }
        return;
    }

    const int wave_m = wave / 4, wave_n = wave % 4;
    int lhs_addresses[kBlocks], rhs_addresses[kBlocks];
    Lhs::fragment_addresses(wave_m * 64, lane, lhs_addresses);
    Rhs::fragment_addresses(wave_n * 64, lane, rhs_addresses);
    const int64_t row_bytes = args.out_stride_row * sizeof(T);
    const bool streaming = (reinterpret_cast<uintptr_t>(args.out) | row_bytes) % 128 == 0;
    while (items.take(args, item)) {
        const int slices = item.slices(), tiles = (item.rows + kTileM - 1) / kTileM;
        const int cols_valid = static_cast<int>(min(static_cast<int64_t>(kTileN), args.cols - item.column));
        const char *out = static_cast<const char *>(args.out) + (item.expert * args.sparse_size + item.row) * row_bytes + item.column * sizeof(T);
        int lhs = lds, rhs = lds + kRhsAt;
        const int last_rhs = lds + kRhsAt + (item.resident() ? slices - 1 : kSlots - 1) * Rhs::kBytes;
        Fragments first, second;
        __syncthreads();
        first.read(lhs_addresses, lhs, rhs_addresses, rhs, 0);
#pragma unroll 1
        for (int tile = 0; tile < tiles; ++tile) {
            TileStore<T, kAccumulate> store;
            store.begin(out, args.out_stride_row, item.rows - tile * kTileM, cols_valid, wave_m, wave_n, opaque(lane));
            f32x16_t acc[kBlocks][kBlocks];
            clear(acc);
#pragma unroll 1
            for (int s = 0; s < slices; ++s) {
                second.read(lhs_addresses, lhs, rhs_addresses, rhs, 1);
                first.template multiply<T>(acc);
                lhs = lhs == lds + (kSlots - 1) * Lhs::kBytes ? lds : lhs + Lhs::kBytes;
                rhs = rhs == last_rhs ? lds + kRhsAt : rhs + Rhs::kBytes;
                __syncthreads();
                // (After the last slice of an item what lies there is read, and not multiplied.)
                first.read(lhs_addresses, lhs, rhs_addresses, rhs, 0);
                second.template multiply<T>(acc);
            }
            store.finish(acc, lds + kStagingAt + wave * kStagingBytes, streaming);
            out += kTileM * row_bytes;
        }
    }
}

template <typename T, bool kAccumulate>
static int launch(const GemmArgs &args, hipStream_t stream) {
    const auto kernel = grouped_gemm_row_panel_kernel<T, kAccumulate>;
    static std::atomic<uint64_t> configured{0};
    if (int status = allow_lds(reinterpret_cast<const void *>(kernel), kLdsBytes, configured)) return status;
    kernel<<<kResident, kThreads, kLdsBytes, stream>>>(args);
    return FM_OK;
}

template <typename T>
static int launch(GemmArgs args, hipStream_t stream) {
    args.tiles_n = static_cast<int>((args.cols + kTileN - 1) / kTileN);
    return args.accumulate ? launch<T, true>(args, stream) : launch<T, false>(args, stream);
}

}  // namespace row_panel

// Where the lines lie, as times of the kernels that such products ran on before (fm_gemm_row_sparse.hip; added to `out`:
// fm_gemm_mfma.hip) over those here, both gradients of a layer:
//   rows per expert            16    40    80    120   180   260   400
//   128 of 2048 x 768         1.08  1.16  1.38  1.29  1.06  0.99  0.99
//    some experts preferred   1.01  1.01  1.10  1.10  1.16  1.08  0.99
//   64 of 2048 x 1408         1.06  1.18  1.33  1.26  1.06  1.05  0.95
//    some experts preferred   1.00  1.00  1.08  1.07  1.01  1.02  0.94
//   8 of 4096 x 14336         1.15  1.15  1.25  1.19  1.04  1.04  0.95
//   32 of 1536 x 2048         0.98  1.09  1.10  1.08  0.94  0.94  0.97
//    some experts preferred   0.97  0.92  0.95  0.95  0.95  1.04  1.03
//   16 of 1280 x 3416         1.05  1.07  1.06  0.85  0.91  0.95  1.02
//   added, 128 of 2048 x 768  1.32  1.21  1.16  1.12  1.20  0.96  0.97
//    some experts preferred   1.60  1.46  1.37  1.22  1.13  0.99  1.00
//   added, 8 of 4096 x 14336  1.14  1.07  1.09  1.04  1.06  1.05  1.02
//   added, 16 of 1280 x 3416  1.11  1.06  1.11  1.05  1.04  0.99  1.00
// The rows are those that the operands have, with up to 128 of padding per expert. Products that are not added are taken from 22 tiles per
// workgroup on (of the 32 experts the larger gradient has 24, the smaller one 12; neither of the 16): in a trace of 420 drawn training steps
// and layers (rows up to 320) 22 to 31 tiles are 1.14 times as fast as before (0.98 at worst, 47 gradients), 32 to 63 1.12 (0.97, 55),
// more 1.05 (0.91, 13), added ones 1.33 (1.01, 56). Results in 32 bits are no faster: 0.89 to 1.18, added 0.94 to 1.09 (at 5 TB/s of values
// read and written either way).
constexpr int64_t kMaxRowsPerExpert = 320, kLeastTiles = 22 * row_panel::kResident;

// `args` as `mfma_gemm_eligible` takes them.
bool row_panel_gemm_chosen(const GemmArgs &args, int dtype) {
    using namespace row_panel;
    if (args.mode != kInputRowSparse || args.expert_ends == nullptr || args.out_dtype != dtype || args.lhs_stride_row != 1 ||
        args.rhs_stride_col != 1 || args.out_stride_row >= (int64_t(1) << 21) || args.num_experts > kMaxExperts || args.inner > kMaxRowsPerExpert * args.num_experts)
        return false;
    const int64_t tiles = (args.sparse_size + kTileM - 1) / kTileM * ((args.cols + kTileN - 1) / kTileN) * args.num_experts;
    return args.sparse_size < (int64_t(1) << 30) && tiles < (int64_t(1) << 30) && (args.accumulate || tiles >= kLeastTiles);
}

int row_panel_gemm_launch(const GemmArgs &args, int dtype, hipStream_t stream) {
    return dtype == FM_DTYPE_BF16 ? row_panel::launch<bf16_t>(args, stream) : row_panel::launch<f16_t>(args, stream);
}

}  // namespace fm
