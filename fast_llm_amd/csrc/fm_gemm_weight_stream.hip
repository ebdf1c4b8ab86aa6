// Products with expert weights that are bound by the rate at which those come from memory (some hundred rows per expert), or that have
// few tiles, in half precision: 128 or 192 rows x 256, 192 or 128 columns (with the gated activation half of them gates, half ups).
//
// In the kernels where each wavefront loads, multiplies and stores, nothing is on its way while a tile is set up and written out, and a
// launch of 1.1 rounds of tiles takes two. Here one workgroup per CU walks its tiles with
//   * four wavefronts that only load, straight from memory into LDS, up to two slices of 64 along K ahead of the multiplications and
//     on into the next tile: what is asked for does not depend on where a tile ends;
//   * eight that multiply 64 x 64 or 96 x 64 of the tile each and store, and never wait for memory;
//   * the tiles' width and height chosen on the device, from the rows that the experts have, so that the last round is full (`Tiles`);
//   * tiles found from row counts in registers, without a table that a kernel in front has to write (5 to 9 us).
// One GPU, us before and now: layer 1's product with 40 rows for each of 8 experts of 4096 x 14336 418 -> 384 (1.88 GB: 4.9 TB/s,
// 5.3 without what a launch takes to start and end), of 16 of 4096 x 4096 201 -> 189 (5.7 TB/s); layer 2's for 80 rows of 16 of
// 1280 x 3416 64 -> 55. What is on its way (64 KB of weights per CU) limits it. These are its best shapes: tall tiles of 125 rows for each of
// 128 experts of 2048 x 768 (150 us a launch, 2048 columns on average) read weights at 4.0 TB/s, 4.9 with activations and results.
// Tall tiles are for experts of 100 rows and more, whose rows would be two tiles of 128, the second nearly empty, or one large one:
// inference of 125 and 150 rows for each of 32 experts of 3000 x 1000 258 -> 210 and 271 -> 222 us, 250 390 -> 307; of 125 of 16 of 4096 x
// 4096 382 -> 358; a training step of 375 of 16 of 1280 x 3416 842 -> 802. They leave LDS for two slices of the lhs, which mostly comes
// from L2, and are 2 to 10 % slower where 128 rows would do.
// Sums in fp32, in the order of the large tiles' kernel (fm_gemm_mfma.hip) where that does not cut its reductions into pieces: those bits.
// Reductions that it would cut are one chain of additions here.
#include <cmath>
#include <type_traits>
#include "fm_activation_math.h"
#include "fm_gemm_slices.h"
#include "fm_partition.h"

namespace fm {

namespace weight_stream {

using namespace slices;

// Tiles have up to 128 rows, or (tall ones) up to 192. A wavefront multiplies half of the rows x 64, in 32 x 32 accumulators.
template <bool kTall>
constexpr int kTileM = kTall ? 192 : 128;
template <bool kTall>
constexpr int kBlocksM = kTileM<kTall> / 64;
constexpr int kTileN = 256, kLeastWidth = 128, kBlocksN = 2;
constexpr int kMultiplying = 8, kThreads = 64 * kMultiplying + kLoadingThreads;
constexpr int kMaxExperts = 256, kExpertRegisters = kMaxExperts / 64;
constexpr int kResident = 256;  // workgroups on the device at one time

// LDS: slots for slices of both operands, a staging region per multiplying wavefront.
template <bool kTall>
constexpr int kLhsSlots = kTall ? 2 : 3;
template <bool kTall>
constexpr int kLhsBytes = kTileM<kTall> * kBK * 2;
constexpr int kRhsSlots = 3, kRhsBytes = kTileN * kBK * 2, kRhsAt = kLhsSlots<true> * kLhsBytes<true>;
static_assert(kRhsAt == kLhsSlots<false> * kLhsBytes<false>, "the same LDS for both heights");
constexpr int kStagingAt = kRhsAt + kRhsSlots * kRhsBytes, kStagingBytes = 2048;
constexpr int kLdsBytes = kStagingAt + kMultiplying * kStagingBytes;
static_assert(kLdsBytes <= 160 * 1024, "LDS of a CU");

struct Tile {
    int expert, row, rows_valid, tile_n;
};

// The tiles of a workgroup. The experts' row counts stay in registers: a tile is found without waiting for memory.
// The columns and most rows of a tile are those with which the launch is shortest, if a round takes as long as its columns, half of its
// mean rows (from L2, where the weights come from memory) and 16 more: layer 2's input gradient of 40 rows of 128 experts of 2048 x 768 is
// 384 tiles of 256 columns, 1.5 rounds, or 512 of 192: 101.5 -> 95.9 us; layer 1's input gradient of 8 experts of 4096 x 14336 is 128 of
// 256 or 256 of 128: 520 -> 370.
template <bool kTall>
struct Tiles {
    static constexpr int kLeastHeight = 128, kHeight = kTileM<kTall>;
    int begin[kExpertRegisters], rows[kExpertRegisters], row_tiles_to[kExpertRegisters];  // of an expert per lane and register
    int height, width, tiles_n, total, next;  // most rows of a tile, its columns, tiles next to one another

    // `columns`: of the weights of one expert.
    __device__ __forceinline__ void load(const GemmArgs &args, int columns, int lane) {
        int all_rows = 0, low = 0, high = 0;  // row tiles of the least height, and of the most
#pragma unroll
        for (int i = 0; i < kExpertRegisters; ++i) {
            const int e = i * 64 + lane;
            int64_t first = 0, end = 0;
            if (args.expert_ends == nullptr) end = e == 0 ? args.rows : 0;
            else if (e < args.num_experts) rows_of_expert(args, e, first, end);
            begin[i] = static_cast<int>(first);
            rows[i] = static_cast<int>(max(end - first, static_cast<int64_t>(0)));
            all_rows += rows[i];
            low += (rows[i] + kLeastHeight - 1) / kLeastHeight;
            high += (rows[i] + kHeight - 1) / kHeight;
        }
#pragma unroll
        for (int offset = 32; offset > 0; offset >>= 1) {
            all_rows += __shfl_xor(all_rows, offset, 64);
            low += __shfl_xor(low, offset, 64);
            high += __shfl_xor(high, offset, 64);
        }
        all_rows = __builtin_amdgcn_readfirstlane(all_rows);
        int least = 0x7fffffff;
        height = kLeastHeight;
        width = kTileN;
#pragma unroll
        for (int h = kLeastHeight; h <= kHeight; h += 64) {
            const int row_tiles = __builtin_amdgcn_readfirstlane(h == kLeastHeight ? low : high);
            const int row_cost = (kTall ? all_rows / max(row_tiles, 1) : 96) / 2 + 16;
#pragma unroll
            for (int w = kTileN; w >= kLeastWidth; w -= 64) {
                const int rounds = (row_tiles * ((columns + w - 1) / w) + kResident - 1) / kResident, cost = rounds * (w + row_cost);
                if (cost < least) least = cost, height = h, width = w;
            }
        }
        int row_tiles = 0;
#pragma unroll
        for (int i = 0; i < kExpertRegisters; ++i) {
            int inclusive = (rows[i] + height - 1) / height;
#pragma unroll
            for (int offset = 1; offset < 64; offset <<= 1) {
                const int other = __shfl_up(inclusive, offset, 64);
                if (lane >= offset) inclusive += other;
            }
            row_tiles_to[i] = row_tiles + inclusive;
            row_tiles = __builtin_amdgcn_readlane(row_tiles_to[i], 63);
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
            const int expert_rows = __builtin_amdgcn_readlane(rows[i], owner), count = (expert_rows + height - 1) / height;
            const int first = __builtin_amdgcn_readlane(row_tiles_to[i], owner) - count;
            int in_expert;
            place_in_expert(logical - first * tiles_n, count, tiles_n, in_expert, tile.tile_n);
            tile.expert = i * 64 + owner;
            TileRows of_tile{in_expert * kHeight, min((in_expert + 1) * kHeight, expert_rows)};
            if constexpr (kTall) of_tile = rows_of_tile(in_expert, expert_rows, count);
            tile.row = __builtin_amdgcn_readlane(begin[i], owner) + of_tile.first;
            tile.rows_valid = of_tile.last - of_tile.first;
        }
        return tile;
    }
};

// value(i, j, v), of 32 x 32 accumulators -> rows of `out`, as many at a time as the wavefront's part of LDS takes: 16 bytes per lane and
// store. The tile's rows are the MFMA's columns: a lane's four accumulators are consecutive columns of one row.
template <typename T, int kRowBlocks, int kColumnBlocks, typename Value>
__device__ __forceinline__ void store_tile(Value &&value, int staging, T *out, int64_t stride, int rows_valid, int cols_valid, int first_row,
                                           int blocks, int wave_n, int lane) {
    constexpr int kWaveCols = kColumnBlocks * 32, kRowBytes = kWaveCols * 2, kChunks = kWaveCols / 8;  // 16-byte chunks per row
    constexpr int kPassRows = kStagingBytes / kRowBytes, kRowsPerRead = 64 / kChunks, kReads = kPassRows / kRowsPerRead;
    // Where a chunk sits in its row: a column of chunks lies in different banks.
    const auto address = [&](int row, int chunk) {
        return staging + row * kRowBytes + (chunk ^ ((row / (16 / kChunks)) & (kChunks - 1))) * 16;
    };
    const int read_row = lane / kChunks, read_chunk = lane % kChunks, column = wave_n * kWaveCols + read_chunk * 8;
#pragma unroll
    for (int i = 0; i < kRowBlocks; ++i) {
        if (i >= blocks) continue;
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
                const int row = first_row + i * 32 + pass * kPassRows + t * kRowsPerRead + read_row;
                if (row < rows_valid && column < cols_valid)
                    __builtin_nontemporal_store(staged[t], reinterpret_cast<u32x4_t *>(out + row * stride + column));
            }
            asm volatile("" ::: "memory");
        }
    }
}

template <typename T, bool kRhsK, bool kGated, bool kTall>
__global__ __launch_bounds__(kThreads, 1) void grouped_gemm_weight_stream_kernel(GemmArgs args) {
    constexpr int kBlocksM = weight_stream::kBlocksM<kTall>, kLhsSlots = weight_stream::kLhsSlots<kTall>, kLhsBytes = weight_stream::kLhsBytes<kTall>;
    typedef Operand<kTileM<kTall>, true, kBlocksM> Lhs;
    typedef Operand<kTileN, kRhsK, kBlocksN> Rhs;
    static_assert(Lhs::kBytes == kLhsBytes && Rhs::kBytes == kRhsBytes, "slots");
    extern __shared__ __attribute__((aligned(1024))) char lds_generic[];
    const int lds = static_cast<int>(reinterpret_cast<uintptr_t>((FM_LDS(char) *)lds_generic));
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    Tiles<kTall> tiles;
    tiles.load(args, static_cast<int>(kGated ? 2 * args.half : args.cols), lane);
    const int k_count = static_cast<int>(args.inner), num_slices = (k_count + kBK - 1) / kBK;
    const int num_tiles = tiles.left();
    if (num_tiles == 0) return;
    const int columns = kGated ? tiles.width / 2 : tiles.width;  // of the result
    const auto cols_valid = [&](const Tile &tile) {
        return static_cast<int>(min(static_cast<int64_t>(columns), (kGated ? args.half : args.cols) - static_cast<int64_t>(tile.tile_n) * columns));
    };
    const auto next_slot = [&](int slot, int first, int bytes, int count) { return slot == first + (count - 1) * bytes ? first : slot + bytes; };

    // The slices of the workgroup's tiles pass through the slots one after the other, number s through slots s % kLhsSlots and s %
    // kRhsSlots. Barrier s makes slice s visible (the loading wavefronts have waited for their loads of it) and ends the reads of slice
    // s - 1, whose slots slices s + kLhsSlots - 1 of the lhs, which mostly comes from L2, and s + kRhsSlots - 1 of the weights then fill.
    if (wave >= kMultiplying) {
        const int part = wave - kMultiplying, total = num_tiles * num_slices;
        constexpr bool kApart = kLhsSlots < kRhsSlots;  // the weights are a slice ahead of the lhs, and at most a tile
        static_assert(kLhsSlots == kRhsSlots - kApart, "slices ahead");
        Lhs lhs;
        Rhs rhs;
        int lhs_slot = lds, rhs_slot = lds + kRhsAt, lhs_tiles = num_tiles, rhs_tiles = num_tiles, lhs_slices = 0, rhs_slices = 0;
        Tile tile{};  // of the weights
        const auto next_weights = [&]() {
            tile = tiles.take();
            const int64_t col0 = static_cast<int64_t>(tile.tile_n) * columns;
            const int64_t rhs_offset = args.mode == kOutputSparse
                                           ? (static_cast<int64_t>(tile.expert) * args.sparse_size + col0) * args.rhs_stride_col
                                           : static_cast<int64_t>(tile.expert) * args.sparse_size * args.rhs_stride_inner + col0 * args.rhs_stride_col;
            rhs.template setup<kGated>(reinterpret_cast<const char *>(static_cast<const T *>(args.rhs) + rhs_offset),
                                       (kRhsK ? args.rhs_stride_col : args.rhs_stride_inner) * 2, cols_valid(tile), k_count,
                                       __builtin_amdgcn_readfirstlane(first_slice_of(args, tile.expert)), part, lane, args.half);
            --rhs_tiles;
            rhs_slices = num_slices;
        };
        const auto next_lhs = [&]() {
            lhs.template setup<false>(reinterpret_cast<const char *>(static_cast<const T *>(args.lhs) + tile.row * args.lhs_stride_row),
                                      args.lhs_stride_row * 2, tile.rows_valid, k_count,
                                      __builtin_amdgcn_readfirstlane(first_slice_of(args, tile.expert)), part, lane, 0);
            --lhs_tiles;
            lhs_slices = num_slices;
        };
        // (After the last slice of the last tile: zeros.)
        const auto fetch_lhs = [&]() {
            lhs.fetch(lhs_slot, part);
            lhs_slot = next_slot(lhs_slot, lds, kLhsBytes, kLhsSlots);
            --lhs_slices;
        };
        const auto fetch_weights = [&]() {
            rhs.fetch(rhs_slot, part);
            rhs_slot = next_slot(rhs_slot, lds + kRhsAt, kRhsBytes, kRhsSlots);
            --rhs_slices;
        };
        // The next tile as soon as the last slice of one has been asked for, long before its own first one is. The tile that the lhs goes on
        // to is the one of the weights, which are ahead of it or go on with it. (One loop, the first slices too: what is executed once
        // comes from memory, and a launch of 60 us gets 4 us longer with this set-up inlined three times.)
#pragma unroll 1
        for (int s = 1 - kRhsSlots; s <= total; ++s) {
            const bool lhs_too = !kApart || s > 1 - kRhsSlots;
            if (kApart && lhs_too && lhs_slices == 0 && lhs_tiles > 0) next_lhs();
            if (rhs_slices == 0 && rhs_tiles > 0) next_weights();
            if (!kApart && lhs_slices == 0 && lhs_tiles > 0) next_lhs();
            if (s >= 0) {
                wait_for_loads<Rhs::kLoads + (kApart ? 0 : Lhs::kLoads)>();
                __syncthreads();
            }
            if (lhs_too) fetch_lhs();
            fetch_weights();
        }
        wait_for_loads<0>();
        return;
    }

    // The lower wavefronts have the first 64 rows, half of the blocks of 32 where there are more than 128, the upper ones the rest.
    const int wave_m = wave / 4, wave_n = wave % 4;
    int lhs_addresses[Lhs::kAddresses], rhs_addresses[Rhs::kAddresses];
    Lhs::fragment_addresses(0, lane, lhs_addresses);
    Rhs::fragment_addresses(wave_n * kBlocksN * 32, lane, rhs_addresses);
    const auto blocks_of = [&](const Tile &tile) { return kTall ? max((tile.rows_valid + 63) / 64, 2) : 2; };
    u32x4_t a[2][kBlocksM], b[2][kBlocksN];
    int lhs_slot = lds, rhs_slot = lds + kRhsAt, lhs_row = 0;  // lhs_row: the wavefront's first, in bytes
    const auto read = [&](auto blocks, int buffer, int step) {
#pragma unroll
        for (int i = 0; i < blocks; ++i) a[buffer][i] = Lhs::fragment(lhs_addresses, lhs_slot + lhs_row, i, step);
#pragma unroll
        for (int j = 0; j < kBlocksN; ++j) b[buffer][j] = Rhs::fragment(rhs_addresses, rhs_slot, j, step);
    };
    const auto advance = [&]() {
        lhs_slot = next_slot(lhs_slot, lds, kLhsBytes, kLhsSlots);
        rhs_slot = next_slot(rhs_slot, lds + kRhsAt, kRhsBytes, kRhsSlots);
    };
    static_assert(kSteps % 2 == 0, "fragment buffers alternate");
    constexpr std::integral_constant<int, kBlocksM> all{};
    Tile tile, upcoming = tiles.take();
    const auto start_row = [&](const Tile &of) { return wave_m * blocks_of(of) * 32 * kBK * 2; };
    lhs_row = start_row(upcoming);
    __syncthreads();
    read(all, 0, 0);
#pragma unroll 1
    for (int n = 0; n < num_tiles; ++n) {
        tile = upcoming;
        if (n + 1 < num_tiles) upcoming = tiles.take();
        const int tile_blocks = blocks_of(tile);
        f32x16_t acc[kBlocksM][kBlocksN];
#pragma unroll
        for (int i = 0; i < kBlocksM; ++i)
#pragma unroll
            for (int j = 0; j < kBlocksN; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
        const auto multiply_tile = [&](auto blocks) {
#pragma unroll 1
            for (int t = 0; t < num_slices; ++t) {
#pragma unroll
                for (int step = 0; step < kSteps; ++step) {
                    const bool last = step + 1 == kSteps;
                    if (last) {
                        __syncthreads();
                        advance();
                        if (t + 1 == num_slices) lhs_row = start_row(upcoming);
                        // (After the last slice of the last tile zeros are read, and not multiplied.)
                        read(all, (step + 1) & 1, 0);
                    } else {
                        read(blocks, (step + 1) & 1, step + 1);
                    }
#pragma unroll
                    for (int i = 0; i < blocks; ++i)
#pragma unroll
                        for (int j = 0; j < kBlocksN; ++j) acc[i][j] = mfma(T(), b[step & 1][j], a[step & 1][i], acc[i][j]);
                }
            }
        };
        if (wave_m * tile_blocks * 32 >= tile.rows_valid || wave_n * kBlocksN * 32 >= tiles.width) {  // nothing of the wavefront's exists
#pragma unroll 1
            for (int t = 0; t < num_slices; ++t) {
                __syncthreads();
                advance();
            }
            lhs_row = start_row(upcoming);
            read(all, 0, 0);
            continue;
        }
        if (!kTall || tile_blocks == 2) multiply_tile(std::integral_constant<int, 2>{});
        else multiply_tile(all);
        const int staging = lds + kStagingAt + wave * kStagingBytes, valid = cols_valid(tile), first_row = wave_m * tile_blocks * 32;
        const int64_t col0 = static_cast<int64_t>(tile.tile_n) * columns;
        if constexpr (kGated) {
            // From the rounded values, as the activation's own kernel computes: the same bits.
            T *out = static_cast<T *>(args.fused_out) + tile.row * args.fused_stride + col0;
            const auto store = [&](auto activate) {
                store_tile<T, kBlocksM, 1>(
                    [&](int i, int, int v) {
                        return activate(to_float(from_float<T>(acc[i][0][v]))) * to_float(from_float<T>(acc[i][1][v]));
                    },
                    staging, out, args.fused_stride, tile.rows_valid, valid, first_row, tile_blocks, wave_n, opaque(lane));
            };
            FM_DISPATCH_ACTIVATION(args.activation, kActivation, store([](float x) { return activation_forward<kActivation>(x); }));
        } else {
            T *out = static_cast<T *>(args.out) + tile.row * args.out_stride_row + col0;
            store_tile<T, kBlocksM, 2>([&](int i, int j, int v) { return acc[i][j][v]; }, staging, out, args.out_stride_row, tile.rows_valid, valid,
                             first_row, tile_blocks, wave_n, opaque(lane));
        }
    }
}

template <typename T, bool kRhsK, bool kGated, bool kTall>
static int launch(const GemmArgs &args, hipStream_t stream) {
    const auto kernel = grouped_gemm_weight_stream_kernel<T, kRhsK, kGated, kTall>;
    static std::atomic<uint64_t> configured{0};
    if (int status = allow_lds(reinterpret_cast<const void *>(kernel), kLdsBytes, configured)) return status;
    kernel<<<kResident, kThreads, kLdsBytes, stream>>>(args);
    return FM_OK;
}

template <typename T, bool kTall>
static int launch(const GemmArgs &args, hipStream_t stream) {
    if (args.fusion == kFusionGatedForward) return launch<T, true, true, kTall>(args, stream);
    return args.rhs_stride_inner == 1 ? launch<T, true, false, kTall>(args, stream) : launch<T, false, false, kTall>(args, stream);
}

// Tiles of 128 rows where most experts have no more (the host knows rows with up to 128 of padding per expert), and where the expected
// ones, half of the padding taken off, are one round.
static bool low_tiles(const GemmArgs &args) {
    constexpr int64_t kMostRowsOfLowTiles = 228;
    const int64_t experts = args.num_experts;
    return args.rows <= kMostRowsOfLowTiles * experts || (args.rows - 64 * experts) * ((args.cols + kTileN - 1) / kTileN) <= kResident * 128;
}

template <typename T>
static int launch(const GemmArgs &args, hipStream_t stream) {
    return low_tiles(args) ? launch<T, false>(args, stream) : launch<T, true>(args, stream);
}

}  // namespace weight_stream

// Where the lines lie. 420 drawn layers (inference of 9 to 900 rows per expert, training steps up to 900; all shapes, preferences and
// recompute levels), kernel by kernel in a trace: the time with large tiles over the time here, geometric mean (worst, products), by the
// cost (`Tiles`) of the tiles that the host expects here per round of 256 x 256 ones:
//   weights along K, low tiles      up to 220  .. 250  .. 280  .. 300  .. 320  more
//                                   1.45       1.18    1.17    1.10    1.07    1.06
//                                   (1.10, 22) (.85, 72) (.92, 46) (.87, 82) (.83, 44) (1.00, 13)
//   weights along K, tall tiles     up to 300  .. 340  .. 380  .. 400  .. 420  .. 440  more
//                                   1.10       1.04    1.03    1.09    1.02    0.98    0.99
//                                   (.71, 31)  (.87, 42) (.84, 99) (.98, 12) (.86, 26) (.83, 36) (.90, 9)
//   weights along rows, low tiles   up to 220  .. 250  .. 280  .. 300  more
//    inner size of whole slices     1.17       1.12    1.08    0.97    0.96
//                                   (.84, 55)  (.87, 43) (.90, 27) (.82, 82) (.81, 20)
//    of no whole slices             1.44 (1.21, 4), .. 260 1.36 (1.16, 7), .. 300 1.29 (.98, 8), more 1.33 (1)
//   weights along rows, tall tiles  whole slices .. 300 0.96 (.76, 9), .. 320 1.07 (1), .. 345 1.02 (1); no whole slices .. 360 1.20 (1.07, 11)
// Weights along rows of some 30 rows per expert, as many rounds of tiles here as there, run at 4.9 TB/s here and at 5.7 there (64 experts of
// 2048 x 1408: 75 and 65 us), but there a launch in front writes the table of tiles, 5 to 10 us: whole layers with those products on large
// tiles are 0.95 to 0.97 times as fast in inference, level in training. The same for tall tiles from 280 to 320: 0.93 to 0.96 (four
// layers in inference), 1.04 (two training steps of preferred experts). The masked last slice of a reduction of no whole slices costs the
// large tiles more. With weights along K whole layers from 420 to 440 are 1.02 times as fast on large tiles (0.99 to 1.05).
// Tall tiles lose where some experts are preferred and the host's count of tiles is off: 0.71 to 0.88 are such (and 128 experts of 2048
// x 768 at 150 to 160 rows, exactly 3 rounds of large tiles: 0.87 to 0.92); 2 rounds gain 1.09 on average, 1 and more than 2 1.02.
// More than 1000 low tiles of weights along rows: 0.96 to 1.04, 1.00 on average from 60 rows per expert on, which leaves them to the large.
// 97 to 256 tiles are all taken: 0.80 (12 us) to 1.34, 1.04 on average, against the kernel for few tiles with 128 and 256 columns.
// The host knows rows with up to 128 of padding per expert. Low tiles from 229 rows on are those whose expected tiles (half of the padding
// taken off) are one round: 1.04 (.95) to 1.17 with 200 to 256 tiles; 0.96 (.80) with 257 to 400. A map of the rows in use has some 64 of
// padding: its experts are taken to have 64 rows fewer than they do.
// Reductions that the large tiles' kernel splits into pieces (`splits`) are in these figures (tall 1.01, low 1.04 to 1.24); with 260 rows
// for each of 8 experts of 4096 x 14336 0.87 to 0.91; with 140 to 200 1.05 to 1.3 where some experts are preferred, 0.87 to 1.1 where none is.
namespace weight_stream {

// Row tiles of `height` rows, in fifths (whole numbers: a launch of exactly one round is not to be taken for two), if tokens choose experts
// independently, all alike: a fifth of the experts each has rows of that many standard deviations from the mean.
static int64_t expected_row_tiles(const GemmArgs &args, int height) {
    const float rows = fmaxf(static_cast<float>(args.rows) / args.num_experts - (args.expert_ends != nullptr ? 128.f : 0.f), 1.f);
    int64_t tiles = 0;
    for (const float deviations : {-1.4f, -0.53f, 0.f, 0.53f, 1.4f})
        tiles += static_cast<int64_t>(ceilf(fmaxf(rows + (args.num_experts > 1 ? deviations * sqrtf(rows) : 0.f), 1.f) / height));
    return args.num_experts * tiles;
}

// Rounds of as many tiles next to one another. `row_tiles` in fifths.
static int64_t rounds_of(int64_t row_tiles, int64_t tiles_n) { return (row_tiles * tiles_n + 5 * kResident - 1) / (5 * kResident); }

// What `Tiles` makes of them.
static float expected_cost(const GemmArgs &args) {
    const float rows = fmaxf(static_cast<float>(args.rows - (args.expert_ends != nullptr ? 128 * args.num_experts : 0)), 1.f);
    float least = INFINITY;
    for (int height = 128; height <= kTileM<true>; height += 64) {
        const int64_t row_tiles = expected_row_tiles(args, height);
        const float row_cost = 5 * rows / (2 * row_tiles) + 16;
        for (int width = kTileN; width >= kLeastWidth; width -= 64)
            least = fminf(least, rounds_of(row_tiles, (args.cols + width - 1) / width) * (width + row_cost));
    }
    return least;
}

static int64_t expected_large_rounds(const GemmArgs &args) { return rounds_of(expected_row_tiles(args, 256), (args.cols + 255) / 256); }

}  // namespace weight_stream

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
    const int64_t row_tiles = (args.rows + 127) / 128, tiles_n = (args.cols + kTileN - 1) / kTileN, tiles = row_tiles * tiles_n;
    const int64_t experts = args.num_experts;
    if ((row_tiles + experts) * ((args.cols + kLeastWidth - 1) / kLeastWidth) >= (int64_t(1) << 30)) return false;
    if (tiles <= 96 || (splits && args.rows > 320 * experts)) return false;
    const bool contiguous = args.rhs_stride_inner == 1;
    if (low_tiles(args)) return contiguous || tiles <= 1000 || args.rows <= 180 * experts;
    const int most = contiguous ? 420 : args.inner % kBK == 0 ? 320 : 360;
    return expected_cost(args) <= most * expected_large_rounds(args);
}

int weight_stream_gemm_launch(const GemmArgs &args, int dtype, hipStream_t stream) {
    return dtype == FM_DTYPE_BF16 ? weight_stream::launch<bf16_t>(args, stream) : weight_stream::launch<f16_t>(args, stream);
}

}  // namespace fm
