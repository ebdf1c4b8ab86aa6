// Products with expert weights that are bound by the rate at which those come from memory (some hundred rows per expert), or that have
// few tiles, in half precision: 128 rows x 256, 192 or 128 columns (with the gated activation half of them gates, half ups).
//
// In the kernels where each wavefront loads, multiplies and stores, nothing is on its way while a tile is set up and written out, and a
// launch of 1.1 rounds of tiles takes two. Here one workgroup per CU walks its tiles with
//   * four wavefronts that only load, straight from memory into LDS, up to two slices of 64 along K ahead of the multiplications and
//     on into the next tile: what is asked for does not depend on where a tile ends;
//   * eight that multiply 64 x 64 of the tile each and store, and never wait for memory;
//   * the width of the tiles chosen on the device, from the rows that the experts have, so that the last round is full (`Tiles`);
//   * tiles found from row counts in registers, without a table that a kernel in front has to write (5 to 9 us).
// One GPU, us before and now: layer 1's product with 40 rows for each of 8 experts of 4096 x 14336 418 -> 384 (1.88 GB: 4.9 TB/s,
// 5.3 without what a launch takes to start and end), of 16 of 4096 x 4096 201 -> 189 (5.7 TB/s); layer 2's for 80 rows of 16 of
// 1280 x 3416 64 -> 55. What is on its way (64 KB of weights per CU) limits it: wider or taller tiles leave LDS for fewer slices.
// Sums in fp32, in the order of the large tiles' kernel (fm_gemm_mfma.hip): the same bits.
#include "fm_activation_math.h"
#include "fm_gemm_slices.h"

namespace fm {

namespace weight_stream {

using namespace slices;

constexpr int kTileM = 128, kTileN = 256, kBlocks = 2;  // a wavefront multiplies 64 x 64, in 32 x 32 accumulators
constexpr int kMultiplying = 8, kThreads = 64 * kMultiplying + kLoadingThreads;
constexpr int kMaxExperts = 256, kExpertRegisters = kMaxExperts / 64;
constexpr int kResident = 256;  // workgroups on the device at one time

// LDS: slots for slices of both operands, a staging region per multiplying wavefront.
constexpr int kSlots = 3, kSlotBytes = (kTileM + kTileN) * kBK * 2, kStagingAt = kSlots * kSlotBytes, kStagingBytes = 2048;
constexpr int kLdsBytes = kStagingAt + kMultiplying * kStagingBytes;
static_assert(kLdsBytes <= 160 * 1024, "LDS of a CU");

struct Tile {
    int expert, row, rows_valid, tile_n;
};

// The tiles of a workgroup. The experts' row counts stay in registers: a tile is found without waiting for memory.
// The columns of a tile are those with which the launch is shortest, if a round takes as long as its columns and kWidthCost more (the
// rows of the other operand, and what a tile takes besides): layer 2's input gradient of 40 rows of 128 experts of 2048 x 768 is 384
// tiles of 256 columns, 1.5 rounds, or 512 of 192: 101.5 -> 95.9 us; layer 1's input gradient of 8 experts of 4096 x 14336 is 128 of
// 256 or 256 of 128: 520 -> 370.
struct Tiles {
    static constexpr int kLeastWidth = 128, kWidthCost = 64;
    int begin[kExpertRegisters], rows[kExpertRegisters], row_tiles_to[kExpertRegisters];  // of an expert per lane and register
    int width, tiles_n, total, next;  // columns of a tile, tiles next to one another

    // `columns`: of the weights of one expert.
    __device__ __forceinline__ void load(const GemmArgs &args, int columns, int lane) {
        int row_tiles = 0;
#pragma unroll
        for (int i = 0; i < kExpertRegisters; ++i) {
            const int e = i * 64 + lane;
            int64_t first = 0, end = 0;
            if (args.expert_ends == nullptr) end = e == 0 ? args.rows : 0;
            else if (e < args.num_experts) rows_of_expert(args, e, first, end);
            begin[i] = static_cast<int>(first);
            rows[i] = static_cast<int>(max(end - first, static_cast<int64_t>(0)));
            int inclusive = (rows[i] + kTileM - 1) / kTileM;
#pragma unroll
            for (int offset = 1; offset < 64; offset <<= 1) {
                const int other = __shfl_up(inclusive, offset, 64);
                if (lane >= offset) inclusive += other;
            }
            row_tiles_to[i] = row_tiles + inclusive;
            row_tiles = __builtin_amdgcn_readlane(row_tiles_to[i], 63);
        }
        int least = 0x7fffffff;
        width = kTileN;
#pragma unroll
        for (int w = kTileN; w >= kLeastWidth; w -= 64) {
            const int rounds = (row_tiles * ((columns + w - 1) / w) + kResident - 1) / kResident, cost = rounds * (w + kWidthCost);
            if (cost < least) least = cost, width = w;
        }
        tiles_n = (columns + width - 1) / width;
        total = row_tiles * tiles_n;
        // Consecutive workgroup ids go to the 8 XCDs in turn; the 32 workgroups of an XCD take consecutive tiles.
        next = blockIdx.x % 8 * 32 + blockIdx.x / 8;
    }

    __device__ __forceinline__ int left() const { return next < total ? (total - next + kResident - 1) / kResident : 0; }

    // The next tile of this workgroup, where one is left. Wave-uniform.
    __device__ __forceinline__ Tile take() {
        const int logical = next, row_tile = logical / tiles_n;
        next += kResident;
        Tile tile{};
        bool found = false;
#pragma unroll
        for (int i = 0; i < kExpertRegisters; ++i) {
            if (found) continue;
            const uint64_t later = __ballot(row_tiles_to[i] > row_tile);
            if (later == 0) continue;
            found = true;
            const int owner = __ffsll(static_cast<unsigned long long>(later)) - 1;
            const int expert_rows = __builtin_amdgcn_readlane(rows[i], owner), count = (expert_rows + kTileM - 1) / kTileM;
            const int first = __builtin_amdgcn_readlane(row_tiles_to[i], owner) - count;
            int in_expert;
            place_in_expert(logical - first * tiles_n, count, tiles_n, in_expert, tile.tile_n);
            tile.expert = i * 64 + owner;
            tile.row = __builtin_amdgcn_readlane(begin[i], owner) + in_expert * kTileM;
            tile.rows_valid = min(kTileM, expert_rows - in_expert * kTileM);
        }
        return tile;
    }
};

// value(i, j, v), of 32 x 32 accumulators -> rows of `out`, as many at a time as the wavefront's part of LDS takes: 16 bytes per lane and
// store. The tile's rows are the MFMA's columns: a lane's four accumulators are consecutive columns of one row.
template <typename T, int kColumnBlocks, typename Value>
__device__ __forceinline__ void store_tile(Value &&value, int staging, T *out, int64_t stride, int rows_valid, int cols_valid, int wave_m,
                                           int wave_n, int lane) {
    constexpr int kWaveCols = kColumnBlocks * 32, kRowBytes = kWaveCols * 2, kChunks = kWaveCols / 8;  // 16-byte chunks per row
    constexpr int kPassRows = kStagingBytes / kRowBytes, kRowsPerRead = 64 / kChunks, kReads = kPassRows / kRowsPerRead;
    // Where a chunk sits in its row: a column of chunks lies in different banks.
    const auto address = [&](int row, int chunk) {
        return staging + row * kRowBytes + (chunk ^ ((row / (16 / kChunks)) & (kChunks - 1))) * 16;
    };
    const int read_row = lane / kChunks, read_chunk = lane % kChunks, column = wave_n * kWaveCols + read_chunk * 8;
#pragma unroll
    for (int i = 0; i < kBlocks; ++i) {
        u32x2_t groups[kChunks];
#pragma unroll
        for (int chunk = 0; chunk < kChunks; ++chunk) {
            struct {
                T v[4];
            } group;
#pragma unroll
            for (int c = 0; c < 4; ++c) group.v[c] = from_float<T>(value(i, chunk / 4, chunk % 4 * 4 + c));
            groups[chunk] = __builtin_bit_cast(u32x2_t, group);
        }
#pragma unroll
        for (int pass = 0; pass < 32 / kPassRows; ++pass) {
            const int write_row = (lane & 31) - pass * kPassRows;
            if (write_row >= 0 && write_row < kPassRows) {
#pragma unroll
                for (int chunk = 0; chunk < kChunks; ++chunk)
                    *(FM_LDS(u32x2_t) *)static_cast<uintptr_t>(address(write_row, chunk) + (lane >> 5) * 8) = groups[chunk];
            }
            asm volatile("" ::: "memory");  // a wavefront's own LDS accesses are carried out in order
            u32x4_t staged[kReads];
#pragma unroll
            for (int t = 0; t < kReads; ++t)
                staged[t] = *(FM_LDS(u32x4_t) *)static_cast<uintptr_t>(address(read_row + t * kRowsPerRead, read_chunk));
#pragma unroll
            for (int t = 0; t < kReads; ++t) {
                const int row = (wave_m * kBlocks + i) * 32 + pass * kPassRows + t * kRowsPerRead + read_row;
                if (row < rows_valid && column < cols_valid)
                    __builtin_nontemporal_store(staged[t], reinterpret_cast<u32x4_t *>(out + row * stride + column));
            }
            asm volatile("" ::: "memory");
        }
    }
}

template <typename T, bool kRhsK, bool kGated>
__global__ __launch_bounds__(kThreads, 1) void grouped_gemm_weight_stream_kernel(GemmArgs args) {
    typedef Operand<kTileM, true, kBlocks> Lhs;
    typedef Operand<kTileN, kRhsK, kBlocks> Rhs;
    constexpr int kLoads = Lhs::kLoads + Rhs::kLoads;
      static_assert(Lhs::kBytes + Rhs::kBytes == kSlotBytes, "a slot");
    extern __shared__ __attribute__((aligned(1024))) char lds_generic[];
    const int lds = static_cast<int>(reinterpret_cast<uintptr_t>((FM_LDS(char) *)lds_generic));
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    Tiles tiles;
    tiles.load(args, static_cast<int>(kGated ? 2 * args.half : args.cols), lane);
    const int k_count = static_cast<int>(args.inner), num_slices = (k_count + kBK - 1) / kBK;
    const int num_tiles = tiles.left();
    if (num_tiles == 0) return;
    const int columns = kGated ? tiles.width / 2 : tiles.width;  // of the result
    const auto cols_valid = [&](const Tile &tile) {
        return static_cast<int>(min(static_cast<int64_t>(columns), (kGated ? args.half : args.cols) - static_cast<int64_t>(tile.tile_n) * columns));
    };

    // The slices of the workgroup's tiles pass through the slots one after the other, number s through slot s % kSlots. Barrier s makes
    // slice s visible (the loading wavefronts have waited for their loads of it) and ends the reads of slice s - 1, whose slot
    // slice s + kSlots - 1 then fills.
    if (wave >= kMultiplying) {
        const int part = wave - kMultiplying, total = num_tiles * num_slices;
        Lhs lhs;
        Rhs rhs;
        int slot = lds, tiles_left = num_tiles, slices_left = 0;
        // As soon as a tile's last slice has been asked for, long before the next tile's first one is.
        const auto next_tile = [&]() {
            const Tile tile = tiles.take();
            const int64_t col0 = static_cast<int64_t>(tile.tile_n) * columns;
            const int64_t rhs_offset = args.mode == kOutputSparse
                                           ? (static_cast<int64_t>(tile.expert) * args.sparse_size + col0) * args.rhs_stride_col
                                           : static_cast<int64_t>(tile.expert) * args.sparse_size * args.rhs_stride_inner + col0 * args.rhs_stride_col;
            const int first_slice = __builtin_amdgcn_readfirstlane(first_slice_of(args, tile.expert));
            lhs.template setup<false>(reinterpret_cast<const char *>(static_cast<const T *>(args.lhs) + tile.row * args.lhs_stride_row),
                                      args.lhs_stride_row * 2, tile.rows_valid, k_count, first_slice, part, lane, 0);
            rhs.template setup<kGated>(reinterpret_cast<const char *>(static_cast<const T *>(args.rhs) + rhs_offset),
                                       (kRhsK ? args.rhs_stride_col : args.rhs_stride_inner) * 2, cols_valid(tile), k_count, first_slice,
                                       part, lane, args.half);
            --tiles_left;
            slices_left = num_slices;
        };
        const auto fetch = [&]() {
            // (After the last slice of the last tile: zeros.)
            rhs.fetch(slot + Lhs::kBytes, part);
            lhs.fetch(slot, part);
            slot = slot == lds + (kSlots - 1) * kSlotBytes ? lds : slot + kSlotBytes;
            if (--slices_left == 0 && tiles_left > 0) next_tile();
        };
        next_tile();
#pragma unroll 1
        for (int s = 0; s < kSlots - 1; ++s) fetch();
#pragma unroll 1
        for (int s = 0; s <= total; ++s) {
            wait_for_loads<(kSlots - 2) * kLoads>();
            __syncthreads();
            fetch();
        }
        wait_for_loads<0>();
        return;
    }

    const int wave_m = wave / 4, wave_n = wave % 4;
    int lhs_addresses[Lhs::kAddresses], rhs_addresses[Rhs::kAddresses];
    Lhs::fragment_addresses(wave_m * kBlocks * 32, lane, lhs_addresses);
    Rhs::fragment_addresses(wave_n * kBlocks * 32, lane, rhs_addresses);
    u32x4_t a[2][kBlocks], b[2][kBlocks];
    const auto read = [&](int buffer, int slot, int step) {
#pragma unroll
        for (int i = 0; i < kBlocks; ++i) a[buffer][i] = Lhs::fragment(lhs_addresses, slot, i, step);
#pragma unroll
        for (int j = 0; j < kBlocks; ++j) b[buffer][j] = Rhs::fragment(rhs_addresses, slot + Lhs::kBytes, j, step);
    };
    int slot = lds;
    const auto following = [&]() { return slot == lds + (kSlots - 1) * kSlotBytes ? lds : slot + kSlotBytes; };
    static_assert(kSteps % 2 == 0, "fragment buffers alternate");
    __syncthreads();
    read(0, slot, 0);
#pragma unroll 1
    for (int n = 0; n < num_tiles; ++n) {
        const Tile tile = tiles.take();
        if (wave_m * kBlocks * 32 >= tile.rows_valid || wave_n * kBlocks * 32 >= tiles.width) {  // nothing of the wavefront's exists
#pragma unroll 1
            for (int t = 0; t < num_slices; ++t) {
                __syncthreads();
                slot = following();
            }
            read(0, slot, 0);
            continue;
        }
        f32x16_t acc[kBlocks][kBlocks];
#pragma unroll
        for (int i = 0; i < kBlocks; ++i)
#pragma unroll
            for (int j = 0; j < kBlocks; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
#pragma unroll 1
        for (int t = 0; t < num_slices; ++t) {
            const int next_slot = following();
#pragma unroll
            for (int step = 0; step < kSteps; ++step) {
                const bool last = step + 1 == kSteps;
                if (last) __syncthreads();
                // (After the last slice of the last tile zeros are read, and not multiplied.)
                read((step + 1) & 1, last ? next_slot : slot, last ? 0 : step + 1);
#pragma unroll
                for (int i = 0; i < kBlocks; ++i)
#pragma unroll
                    for (int j = 0; j < kBlocks; ++j) acc[i][j] = mfma(T(), b[step & 1][j], a[step & 1][i], acc[i][j]);
            }
            slot = next_slot;
        }
        const int staging = lds + kStagingAt + wave * kStagingBytes, valid = cols_valid(tile);
        const int64_t col0 = static_cast<int64_t>(tile.tile_n) * columns;
        if constexpr (kGated) {
            // From the rounded values, as the activation's own kernel computes: the same bits.
            T *out = static_cast<T *>(args.fused_out) + tile.row * args.fused_stride + col0;
            const auto store = [&](auto activate) {
                store_tile<T, 1>(
                    [&](int i, int, int v) {
                        return activate(to_float(from_float<T>(acc[i][0][v]))) * to_float(from_float<T>(acc[i][1][v]));
                    },
                    staging, out, args.fused_stride, tile.rows_valid, valid, wave_m, wave_n, opaque(lane));
            };
            FM_DISPATCH_ACTIVATION(args.activation, kActivation, store([](float x) { return activation_forward<kActivation>(x); }));
        } else {
            T *out = static_cast<T *>(args.out) + tile.row * args.out_stride_row + col0;
            store_tile<T, 2>([&](int i, int j, int v) { return acc[i][j][v]; }, staging, out, args.out_stride_row, tile.rows_valid, valid,
                             wave_m, wave_n, opaque(lane));
        }
    }
}

template <typename T, bool kRhsK, bool kGated>
static int launch(const GemmArgs &args, hipStream_t stream) {
    const auto kernel = grouped_gemm_weight_stream_kernel<T, kRhsK, kGated>;
    static std::atomic<uint64_t> configured{0};
    if (int status = allow_lds(reinterpret_cast<const void *>(kernel), kLdsBytes, configured)) return status;
    kernel<<<kResident, kThreads, kLdsBytes, stream>>>(args);
    return FM_OK;
}

template <typename T>
static int launch(const GemmArgs &args, hipStream_t stream) {
    if (args.fusion == kFusionGatedForward) return launch<T, true, true>(args, stream);
    return args.rhs_stride_inner == 1 ? launch<T, true, false>(args, stream) : launch<T, false, false>(args, stream);
}

}  // namespace weight_stream

// Where the lines lie: 300 layers in inference (24 to 800 rows per expert, experts equally and unequally liked; layer 1 with the gated
// activation), the time with large tiles (up to 256 tiles: of fm_gemm_few_tiles.hip) over the time with one of the two products here,
// geometric means (and the worst), by the bound of the 128 x 256 tiles that the host knows and by the mean rows per expert:
//    layer 1, rows       97 ..       257 ..       401 ..       601 ..       1001 ..      more
//     24 .. 59        0.99 (.88)   1.05 (.99)   1.14 (.99)   1.06 (.98)   1.04 (1.00)  1.09 (1.00)
//     60 .. 99        0.97 (.93)   1.02 (.90)   1.14 (1.11)  1.09 (1.04)  1.03 (.97)   1.09 (1.07)
//    100 .. 139       1.05 (.98)   1.01 (.91)   1.10 (1.05)  1.06 (1.03)  1.04 (.97)   1.04 (.97)
//    140 .. 199       0.93                      0.97 (.95)   1.05 (.97)   1.02 (.98)   1.01 (.97)
//    200 .. 269       1.00 (.97)   1.08 (1.00)  0.94         0.98 (.93)   1.01 (.92)   1.00 (.90)
//    more             1.07         0.93 (.89)   0.92 (.85)   1.03 (.93)   1.00 (.90)   0.99 (.90)
//    layer 2, rows
//     24 .. 59        1.02 (.90)   1.03 (.99)   1.06 (1.03)  1.02 (.98)   1.01 (.98)   1.03 (1.01)
//     60 .. 99        1.04 (.88)   1.02 (.99)   1.03 (1.00)  1.00 (.96)   1.01 (.99)   1.00 (.96)
//    100 .. 139       1.03 (.90)   0.99 (.94)   1.02 (1.00)  1.01 (.99)   1.04 (.98)   1.00 (.98)
//    140 .. 199       1.03 (.84)   1.04 (.98)   1.05         1.00 (.95)   0.98 (.95)   0.98 (.97)
//    200 .. 269       1.01 (.81)   1.02 (.98)   0.97 (.83)   1.00 (1.00)  0.97 (.93)   0.97 (.95)
//    more             1.06 (1.00)  1.03 (.99)   0.92 (.77)   0.99 (.93)   1.00 (.96)   0.97 (.95)
// (those below 1 up to 256 tiles with the other product on large tiles instead of few). With both here, which also saves the launch that
// writes the tables, the whole layer is 1.07 to 1.27 times as fast below 100 rows, 1.0 to 1.2 from 100 to 199. Whole training steps of
// 64 rows: 1.01 (128 experts of 2048 x 768) to 1.14 (16 of 1280 x 3416). The host knows rows with up to 128 of padding per expert.
// With more rows than the first of the rules below allows, those whose expected tiles (half of the padding taken off) are one round:
// 1.04 (.95) to 1.17 with 200 to 256 tiles; 0.96 (.80) with 257 to 400.
// Reductions that the large tiles' kernel splits into pieces (`splits`): 0.87 to 0.91 with 260 rows for each of 8 experts of 4096 x
// 14336, 0.99 (1.25 with some experts preferred) with 180.
// `args` as `mfma_gemm_eligible` (or, with the activation, `mfma_gemm_fusion_eligible`) takes them.
bool weight_stream_gemm_chosen(const GemmArgs &args, int dtype, bool splits) {
    using namespace weight_stream;
    if (args.mode == kInputRowSparse || args.num_experts > kMaxExperts || args.accumulate || args.out_dtype != dtype ||
        args.lhs_stride_inner != 1 || args.rows >= (int64_t(1) << 30))
        return false;
    // With the gated activation where layer 1's own output is not wanted; the ups are addressed with 32 bits from the gates.
    if (args.fusion == kFusionGatedForward && (args.out != nullptr || (args.half + 128) * args.rhs_stride_col * 2 >= (int64_t(1) << 31)))
        return false;
    if (args.fusion == kFusionGatedBackward) return false;
    const int64_t row_tiles = (args.rows + kTileM - 1) / kTileM, tiles_n = (args.cols + kTileN - 1) / kTileN, tiles = row_tiles * tiles_n;
    const int64_t experts = args.num_experts;
    if ((row_tiles + experts) * ((args.cols + Tiles::kLeastWidth - 1) / Tiles::kLeastWidth) >= (int64_t(1) << 30)) return false;
    if (tiles <= 96 || (splits && args.rows > 320 * experts)) return false;
    const bool contiguous = args.rhs_stride_inner == 1;
    if (args.rows <= (contiguous || tiles <= 1000 ? 228 : 180) * experts) return true;
    if ((args.rows - 64 * experts) * tiles_n <= kResident * kTileM) return true;
    return contiguous && tiles <= 1000 && args.rows <= 300 * experts;
}

int weight_stream_gemm_launch(const GemmArgs &args, int dtype, hipStream_t stream) {
    return dtype == FM_DTYPE_BF16 ? weight_stream::launch<bf16_t>(args, stream) : weight_stream::launch<f16_t>(args, stream);
}

}  // namespace fm
