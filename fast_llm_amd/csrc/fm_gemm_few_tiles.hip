// Grouped products of few output tiles, in half precision: 128 rows x 64 columns (128 or 256 with more than 256 experts).
//
// A launch of a third of a 256 x 256 tile per CU lasts as long as one tile does, on whatever part of the chip, and most of a tile's rows are
// padding where experts have some 100 tokens. With tiles of an eighth of that size more CUs share the same work; two per CU overlap
// one's loads with the other's MFMAs. A CU then reads more operand bytes per multiplication, which is why launches of more tiles
// go elsewhere (fm_gemm_weight_stream.hip; the line, and what was measured on both sides of it, are at few_tiles_gemm_chosen).
//
// Slices of 64 along K (whole 128-byte lines of K-contiguous rows; with 32 the same tiles take 10 to 20 % longer), two or three in LDS,
// filled straight from memory; the fragments of the next 16 are read while the MFMAs of this 16 run. Sums in fp32, in the order of
// the large tiles' kernel.
#include "fm_activation_math.h"
#include "fm_gemm_slices.h"

namespace fm {

namespace few_tiles {

using namespace slices;

constexpr int kTileM = 128, kThreads = kLoadingThreads;
// 2 x 2 wavefronts, 32 x 32 accumulators. With the gated activation the columns are 32 gates and 32 ups, which one wavefront has to have
// both of: 4 x 1.
template <bool kGated>
constexpr int kWavesN = kGated ? 1 : 2;
template <bool kGated>
constexpr int kBlocksM = kTileM / 32 * kWavesN<kGated> / 4;
template <int kTileN, bool kGated>
constexpr int kBlocksN = kTileN / 32 / kWavesN<kGated>;

// value(i, j, v), of 32 x 32 accumulators -> rows of `out`, 32 rows of the wavefront's columns at a time through its own part of LDS: 16
// bytes per lane and store. The tile's rows are the MFMA's columns: a lane's four accumulators are consecutive columns of one row.
template <typename T, int kRowBlocks, int kColumnBlocks, typename Value>
__device__ __forceinline__ void store_tile(Value &&value, int staging, T *out, int64_t stride, int rows_valid, int cols_valid, int wave_m,
                                           int wave_n, int lane) {
    constexpr int kWaveCols = kColumnBlocks * 32, kRowBytes = kWaveCols * 2 + 16;
    constexpr int kLanesPerRow = kWaveCols / 8, kRowsPerRead = 64 / kLanesPerRow, kReads = 32 / kRowsPerRead;
    const int write_base = staging + (lane & 31) * kRowBytes + (lane >> 5) * 8;
    const int read_row = lane / kLanesPerRow, read_column = lane % kLanesPerRow * 8;
    const int read_base = staging + read_row * kRowBytes + read_column * 2;
    const int column = wave_n * kWaveCols + read_column, first_row = wave_m * kRowBlocks * 32 + read_row;
#pragma unroll
    for (int i = 0; i < kRowBlocks; ++i) {
#pragma unroll
        for (int j = 0; j < kColumnBlocks; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                struct {
                    T v[4];
                } group;
#pragma unroll
                for (int c = 0; c < 4; ++c) group.v[c] = from_float<T>(value(i, j, 4 * g + c));
                *(FM_LDS(u32x2_t) *)static_cast<uintptr_t>(write_base + (j * 32 + 8 * g) * 2) = __builtin_bit_cast(u32x2_t, group);
            }
        asm volatile("" ::: "memory");  // a wavefront's own LDS accesses are carried out in order
        u32x4_t staged[kReads];
#pragma unroll
        for (int t = 0; t < kReads; ++t)
            staged[t] = *(FM_LDS(u32x4_t) *)static_cast<uintptr_t>(read_base + t * kRowsPerRead * kRowBytes);
#pragma unroll
        for (int t = 0; t < kReads; ++t) {
            const int row = first_row + i * 32 + t * kRowsPerRead;
            if (row < rows_valid && column < cols_valid)
                __builtin_nontemporal_store(staged[t], reinterpret_cast<u32x4_t *>(out + row * stride + column));
        }
        asm volatile("" ::: "memory");
    }
}

template <int kTileN>
constexpr int kStages = kTileN == 128 ? 2 : 3;  // slices in LDS
template <int kTileN>
constexpr int kWorkgroups = kTileN == 256 ? 1 : 2;  // per CU
template <int kTileN>
constexpr int kLdsBytes = kStages<kTileN> * (kTileM + kTileN) * kBK * 2;

template <typename T, int kTileN, bool kRhsK, bool kGated>
__global__ __launch_bounds__(kThreads, kWorkgroups<kTileN>) void grouped_gemm_few_tiles_kernel(GemmArgs args) {
    constexpr int kBlocksM = few_tiles::kBlocksM<kGated>, kBlocksN = few_tiles::kBlocksN<kTileN, kGated>;
    constexpr int kStages = few_tiles::kStages<kTileN>, kLdsBytes = few_tiles::kLdsBytes<kTileN>;
    typedef Operand<kTileM, true, kBlocksM> Lhs;
    typedef Operand<kTileN, kRhsK, kBlocksN> Rhs;
    constexpr int kSlotBytes = Lhs::kBytes + Rhs::kBytes, kLoads = Lhs::kLoads + Rhs::kLoads;
    constexpr int kColumns = kGated ? kTileN / 2 : kTileN;  // of the result
    static_assert(kLdsBytes * kWorkgroups<kTileN> <= 160 * 1024 && kLdsBytes >= 4 * 32 * (kTileN + 16), "LDS of a CU");
    extern __shared__ __attribute__((aligned(1024))) char lds_generic[];
    const int lds = static_cast<int>(reinterpret_cast<uintptr_t>((FM_LDS(char) *)lds_generic));

    // Consecutive workgroup ids go to the 8 XCDs in turn; an XCD gets runs of `chunk_tiles` consecutive logical tiles.
    const int pid = blockIdx.x, local = pid / 8;
    const int logical = (local / args.chunk_tiles * 8 + pid % 8) * args.chunk_tiles + local % args.chunk_tiles;
    RowTile tile;
    if (!locate_tile<kTileM>(args, logical, tile)) return;
    const int64_t col0 = static_cast<int64_t>(tile.tile_n) * kColumns;
    const int rows_valid = __builtin_amdgcn_readfirstlane(tile.rows_valid);
    const int cols_valid = __builtin_amdgcn_readfirstlane(
        static_cast<int>(min(static_cast<int64_t>(kColumns), (kGated ? args.half : args.cols) - col0)));
    const int64_t rhs_offset = args.mode == kOutputSparse
                                   ? (static_cast<int64_t>(tile.expert) * args.sparse_size + col0) * args.rhs_stride_col
                                   : static_cast<int64_t>(tile.expert) * args.sparse_size * args.rhs_stride_inner + col0 * args.rhs_stride_col;
    const int k_count = static_cast<int>(args.inner), num_slices = (k_count + kBK - 1) / kBK;
    const int first_slice = __builtin_amdgcn_readfirstlane(first_slice_of(args, tile.expert));

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wave_m = wave / kWavesN<kGated>, wave_n = wave % kWavesN<kGated>;
    Lhs lhs;
    Rhs rhs;
    lhs.template setup<false>(reinterpret_cast<const char *>(static_cast<const T *>(args.lhs) + tile.row0 * args.lhs_stride_row),
                              args.lhs_stride_row * 2, rows_valid, k_count, first_slice, wave, lane, 0);
    rhs.template setup<kGated>(reinterpret_cast<const char *>(static_cast<const T *>(args.rhs) + rhs_offset),
                               (kRhsK ? args.rhs_stride_col : args.rhs_stride_inner) * 2, cols_valid, k_count, first_slice, wave, lane,
                               args.half);
    int lhs_addresses[Lhs::kAddresses], rhs_addresses[Rhs::kAddresses];
    Lhs::fragment_addresses(wave_m * kBlocksM * 32, lane, lhs_addresses);
    Rhs::fragment_addresses(wave_n * kBlocksN * 32, lane, rhs_addresses);
    f32x16_t acc[kBlocksM][kBlocksN];
#pragma unroll
    for (int i = 0; i < kBlocksM; ++i)
#pragma unroll
        for (int j = 0; j < kBlocksN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

    int fetch_slot = 0;
    const auto fetch_slice = [&]() {
        lhs.fetch(lds + fetch_slot, wave);
        rhs.fetch(lds + fetch_slot + Lhs::kBytes, wave);
        fetch_slot = fetch_slot == (kStages - 1) * kSlotBytes ? 0 : fetch_slot + kSlotBytes;
    };
    // The oldest slice under way is there, for all wavefronts, and the slot of the slice before it is filled anew: its last fragments
    // have been read.
    const auto next_slice = [&]() {
        wait_for_loads<(kStages - 2) * kLoads>();
        __syncthreads();
        fetch_slice();
    };
    u32x4_t a[2][kBlocksM], b[2][kBlocksN];
    const auto read = [&](int buffer, int slot, int step) {
#pragma unroll
        for (int i = 0; i < kBlocksM; ++i) a[buffer][i] = Lhs::fragment(lhs_addresses, slot, i, step);
#pragma unroll
        for (int j = 0; j < kBlocksN; ++j) b[buffer][j] = Rhs::fragment(rhs_addresses, slot + Lhs::kBytes, j, step);
    };
#pragma unroll
    for (int s = 0; s < kStages - 1; ++s) fetch_slice();
    next_slice();
    int slot = lds;
    read(0, slot, 0);
    static_assert(kSteps % 2 == 0, "fragment buffers alternate");
    for (int t = 0; t < num_slices; ++t) {
        const int next_slot = slot == lds + (kStages - 1) * kSlotBytes ? lds : slot + kSlotBytes;
#pragma unroll
        for (int step = 0; step < kSteps; ++step) {
            const bool last = step + 1 == kSteps;
            if (last) next_slice();
            read((step + 1) & 1, last ? next_slot : slot, last ? 0 : step + 1);
#pragma unroll
            for (int i = 0; i < kBlocksM; ++i)
#pragma unroll
                for (int j = 0; j < kBlocksN; ++j) acc[i][j] = mfma(T(), b[step & 1][j], a[step & 1][i], acc[i][j]);
            // The reads between the MFMAs, not all in front of them.
#pragma unroll
            for (int n = 0; n < kBlocksM * kBlocksN; ++n) {
                __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, kRhsK ? 1 : 2, 0);
            }
        }
        slot = next_slot;
    }
    wait_for_loads<0>();  // zeros on their way to the slots
    __syncthreads();
    const int staging = lds + wave * 32 * (kTileN + 16);
    if constexpr (kGated) {
        // From the rounded values, as the activation's own kernel computes: the same bits.
        T *out = static_cast<T *>(args.fused_out) + tile.row0 * args.fused_stride + col0;
        const auto store = [&](auto activate) {
            store_tile<T, kBlocksM, kBlocksN / 2>(
                [&](int i, int j, int v) {
                    return activate(to_float(from_float<T>(acc[i][2 * j][v]))) * to_float(from_float<T>(acc[i][2 * j + 1][v]));
                },
                staging, out, args.fused_stride, rows_valid, cols_valid, wave_m, wave_n, lane);
        };
        FM_DISPATCH_ACTIVATION(args.activation, kActivation, store([](float x) { return activation_forward<kActivation>(x); }));
    } else {
        T *out = static_cast<T *>(args.out) + tile.row0 * args.out_stride_row + col0;
        store_tile<T, kBlocksM, kBlocksN>([&](int i, int j, int v) { return acc[i][j][v]; }, staging, out, args.out_stride_row, rows_valid,
                                          cols_valid, wave_m, wave_n, lane);
    }
}

// Tiles of 128 x 256, by the upper bound that the host knows of their row tiles (a static map has one tile of padding per expert).
static int64_t most_tiles(const GemmArgs &args) { return (args.rows + kTileM - 1) / kTileM * ((args.cols + 255) / 256); }

template <typename T, int kTileN, bool kRhsK, bool kGated = false>
static int launch(const GemmArgs &args, hipStream_t stream) {
    const auto kernel = grouped_gemm_few_tiles_kernel<T, kTileN, kRhsK, kGated>;
    static std::atomic<uint64_t> configured{0};
    if (int status = allow_lds(reinterpret_cast<const void *>(kernel), kLdsBytes<kTileN>, configured)) return status;
    const int64_t tiles = static_cast<int64_t>(args.tiles_m) * args.tiles_n, round = 8 * static_cast<int64_t>(args.chunk_tiles);
    kernel<<<static_cast<uint32_t>((tiles + round - 1) / round * round), kThreads, kLdsBytes<kTileN>, stream>>>(args);
    return FM_OK;
}

template <typename T, int kTileN>
static int launch(GemmArgs args, hipStream_t stream) {
    args.tiles_m = static_cast<int>((args.rows + kTileM - 1) / kTileM + (args.num_experts > 1 ? args.num_experts : 0));
    args.tiles_n = static_cast<int>((args.cols + kTileN - 1) / kTileN);
    const int64_t tiles = static_cast<int64_t>(args.tiles_m) * args.tiles_n;
    if (tiles >= (int64_t(1) << 30)) return fail(FM_ERR_UNSUPPORTED, "grouped gemm: too many tiles");
    // Runs of 16 tiles per XCD; 8 and 32 are up to 3 and 5 % slower (128 columns).
    args.chunk_tiles = static_cast<int>(min(int64_t(16), (tiles + 7) / 8));
    if constexpr (kTileN == 64)
        if (args.fusion == kFusionGatedForward) return launch<T, kTileN, true, true>(args, stream);
    return args.rhs_stride_inner == 1 ? launch<T, kTileN, true>(args, stream) : launch<T, kTileN, false>(args, stream);
}

template <typename T>
static int launch(const GemmArgs &args, hipStream_t stream) {
    const int64_t tiles = most_tiles(args);
    return tiles <= 96 ? launch<T, 64>(args, stream) : tiles <= 160 ? launch<T, 128>(args, stream) : launch<T, 256>(args, stream);
}

}  // namespace few_tiles

// Where the lines lie. Over 240 layers of random shapes (4 to 1100 rows per expert, experts equally and unequally liked, sizes that are
// whole slices and that are not), weights in memory and activations in cache, the time of 256 x 256 tiles divided by that of 64, 128 and
// 256 columns, geometric means (and the worst), by most_tiles:
//       up to 64       2.00 (1.85), 1.46, 1.27
//       65 .. 96       1.74 (1.10), 1.44 (1.19), 1.20
//       97 .. 160      1.28 (0.95), 1.40 (1.10), 1.23 (0.99)
//       161 .. 192     1.08, 1.16 (0.99), 1.16 (1.01)
//       193 .. 256     0.98, 1.09 (0.96), 1.16 (1.00)
//       257 .. 320     0.95, 1.08 (0.71), 1.13 (0.73): two rounds where 256 x 256 tiles take one
// Above 96 the kernel that streams weights takes all of up to 256 experts, 1.0 to 1.2 times as fast as 128 or 256 columns here (inference
// of 40 to 200 rows for each of 8 experts of 1024 x 2816 1.24 to 1.34, of 4096 x 1536 1.10 to 1.14); up to 96 it is no faster, with 64
// columns either (0.98 to 1.02). More experts with so few tiles are those of which most have no rows: 100 to 250 of 300 and 512 with 60 rows,
// 256 columns 20 to 67 us here, 26 to 75 with 64 columns, 32 to 68 on 256 x 256 tiles.
// Reductions that the large tiles' kernel splits into pieces for all CUs: 1.33 (0.87) up to 96, and no better with more: they stay there.
// With the gated activation against fused tiles of 256 x 256, layer 1 of 800 tokens of 8 experts of 1536 x 512 (6 each) 45 -> 31 us.
bool few_tiles_gemm_chosen(const GemmArgs &args, int dtype, bool splits) {
    if (dtype == FM_DTYPE_F32 || args.mode == kInputRowSparse || args.accumulate || args.out_dtype != dtype || args.lhs_stride_inner != 1 ||
        splits)
        return false;
    // With the gated activation where layer 1's own output is not wanted; the ups are addressed with 32 bits from the gates.
    if (args.fusion == kFusionGatedForward && (args.out != nullptr || (args.half + 128) * args.rhs_stride_col * 2 >= (int64_t(1) << 31)))
        return false;
    if (args.fusion == kFusionGatedBackward) return false;
    return few_tiles::most_tiles(args) <= (args.fusion == kFusionNone ? 256 : 96);
}

int few_tiles_gemm_launch(const GemmArgs &args, int dtype, hipStream_t stream) {
    return dtype == FM_DTYPE_BF16 ? few_tiles::launch<bf16_t>(args, stream) : few_tiles::launch<f16_t>(args, stream);
}

}  // namespace fm
