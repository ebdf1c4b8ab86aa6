// Grouped matrix products of fp32 operands on the gfx950 matrix cores (v_mfma_f32_32x32x2_f32: true fp32
// multiply-adds, which is what the 1e-5 fp32 parity bound needs).
//
// An MFMA of this kind keeps the matrix pipe busy for 64 cycles and needs two 256-byte operand fragments, so neither
// LDS nor address arithmetic is near a limit; what has to be hidden is memory latency, and many small workgroups per CU
// hide it better than deep pipelines: eight of them (16 KiB of LDS, at most 64 registers per lane), each one slice
// ahead. Tiles of 128 x 128 with two or three workgroups per CU and two to four slots were slower at every size tried,
// and so were fewer workgroups with more slots. Forward and backward products of 4096 rows over 8 experts, 1024 x 2816
// (5632): 5350 us for the six on tiles of 128 x 128 x 16 fetched element by element through registers, 2120 here (88 to
// 116 TFLOP/s of rows that exist; padding is another 12 %; the device's library reaches 153 on a dense product).
//   * Operand slices (kBK reduction indices) go straight from global memory into LDS (`buffer_load ... lds`, 16 bytes
//     per lane), one slice ahead of the multiplications, one barrier per slice. Lanes that have nothing to fetch (rows past the tile's last one, indices past the reduction range) are sent out of the buffer's range and
//     bring zeros.
//   * An operand may be contiguous along K (activations, `weight.t()`): stored [row][K], fragments are 128-bit reads of
//     four K values of one row; or along its other axis (`weight`, `activations.t()`): stored [K][row] as in memory,
//     fragments are four 32-bit reads. A group of eight K values is split over the wavefront's halves as 0..3 and 4..7;
//     both layouts agree on that, and the order of a sum is free. Chunks are XOR-swizzled on the global side so that
//     fragment reads hit all banks.
//   * Tiles never straddle experts (they are enumerated per expert from `expert_ends`), so any padding multiple works.
// Two tiles, by how many there are (see `f32_gemm_launch`):
//   64 x 64, 4 wavefronts of 32 x 32;
//   32 x 32, the 4 wavefronts take a quarter of every slice each and add up in LDS: four times the workgroups, for
//   launches whose outputs are too few to fill the CUs otherwise.
#include "fm_gemm_common.h"

namespace fm {

namespace f32 {

typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;

constexpr int kThreads = 256;

// One operand's slice in LDS and the loads that fill it.
template <int kTile, int kBK, bool kContiguousK>
struct Operand {
    static constexpr int kBytes = kTile * kBK * 4;
    static constexpr int kLoads = kBytes / 16 / kThreads;              // 16-byte loads per lane and slice
    static constexpr int kChunks = (kContiguousK ? kBK : kTile) / 4;   // 16-byte chunks along the contiguous axis
    static_assert(kLoads * kThreads * 16 == kBytes, "whole loads");

    // Where chunk `c` of line `line` (a row, or a K-row) sits among the line's chunks.
    static __device__ __forceinline__ int swizzled(int line, int c) {
        if constexpr (kContiguousK) {
            constexpr int kLinesPer256 = kBK >= 64 ? 1 : 64 / kBK;
            return c ^ ((line / kLinesPer256) & (kChunks < 16 ? kChunks - 1 : 15));
        } else {
            return c ^ (kChunks > 8 ? ((line >> 2) & 1) << 3 : 0);
        }
    }

    const char *base;          // wave-uniform: element (first row of the tile, first k of the next slice to fetch)
    int64_t step;              // bytes from one slice to the next
    uint32_t offset[kLoads];   // per lane, bytes from `base`; out of range where there is nothing to fetch
    int k_local[kLoads];       // first reduction index of the chunk within the slice
    int k_left;                // reduction indices from `base` on
    static constexpr uint32_t kOutOfRange = 0x80000000u, kRange = 0x7fffffffu;

    // `stride`: bytes between lines. `valid`: rows that exist.
    __device__ __forceinline__ void setup(const char *first, int64_t stride, int valid, int k_count, int wave, int lane) {
        base = uniform_pointer(first);
        step = kContiguousK ? kBK * 4 : kBK * stride;
        k_left = k_count;
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const int slot = (wave * kLoads + j) * 64 + lane;
            const int line = slot / kChunks, chunk = swizzled(line, slot % kChunks);
            const bool exists = kContiguousK ? line < valid : chunk * 4 < valid;
            offset[j] = exists ? static_cast<uint32_t>(line * stride + chunk * 16) : kOutOfRange;
            k_local[j] = kContiguousK ? chunk * 4 : line;
        }
    }

    // Fetches the next slice into the LDS slot at byte address `slot`.
    __device__ __forceinline__ void fetch(int slot, int wave) {
        const __amdgpu_buffer_rsrc_t resource = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<char *>(uniform_pointer(base)), 0, static_cast<int>(kRange), kBufferResourceFlags);
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const uint32_t lane_offset = k_local[j] < k_left ? offset[j] : kOutOfRange;
            const int target = __builtin_amdgcn_readfirstlane(slot + (wave * kLoads + j) * 1024);
            asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                         :
                         : "s"(target), "v"(lane_offset), "s"(resource)
                         : "memory");
        }
        base += step;
        k_left -= kBK;
    }

    // The lane's four K values (8 q + 4 half + 0 .. 3) of row `row`, from the slot at byte address `slot`.
    static __device__ __forceinline__ void fragment(int slot, int row, int q, int half, float (&values)[4]) {
        if constexpr (kContiguousK) {
            const int address = slot + (row * kChunks + swizzled(row, 2 * q + half)) * 16;
            const f32x4_t vector = *(FM_LDS(f32x4_t) *)static_cast<uintptr_t>(address);
#pragma unroll
            for (int i = 0; i < 4; ++i) values[i] = vector[i];
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int k = 8 * q + 4 * half + i;
                const int address = slot + k * kTile * 4 + swizzled(k, row >> 2) * 16 + (row & 3) * 4;
                values[i] = *(FM_LDS(float) *)static_cast<uintptr_t>(address);
            }
        }
    }
};

template <int kNewest>
__device__ __forceinline__ void wait_for_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kNewest) : "memory");
}

template <int kTile, int kBK, int kStages, bool kLhsK, bool kRhsK>
__global__ __launch_bounds__(kThreads, 8) void grouped_gemm_f32_kernel(GemmArgs args) {
    constexpr int kWavesK = kTile == 32 ? 4 : 1, kWavesN = kTile == 32 ? 1 : 2;
    constexpr int kWaveTile = kTile / kWavesN, kBlocks = kWaveTile / 32;
    typedef Operand<kTile, kBK, kLhsK> Lhs;
    typedef Operand<kTile, kBK, kRhsK> Rhs;
    constexpr int kSlotBytes = Lhs::kBytes + Rhs::kBytes, kLoads = Lhs::kLoads + Rhs::kLoads;
    constexpr int kSteps = kBK / 8 / kWavesK;  // groups of eight K values per wavefront and slice
    extern __shared__ __attribute__((aligned(1024))) char lds_generic[];
    const int lds = static_cast<int>(reinterpret_cast<uintptr_t>((FM_LDS(char) *)lds_generic));

    // Consecutive workgroup ids go to the 8 XCDs in turn; an XCD gets runs of `chunk_tiles` consecutive logical tiles.
    const int pid = blockIdx.x, local = pid / 8;
    const int logical = (local / args.chunk_tiles * 8 + pid % 8) * args.chunk_tiles + local % args.chunk_tiles;
    int64_t lhs_offset, rhs_offset, out_offset, k_lo = 0, k_hi = args.inner;
    int rows_valid, cols_valid;
    if (args.mode == kInputRowSparse) {
        if (logical >= args.tiles_m * args.tiles_n) return;
        int tile_m, tile_n;
        tile_coordinates(logical, args.tiles_m, args.tiles_n, tile_m, tile_n);
        const int tiles_per_expert = static_cast<int>((args.sparse_size + kTile - 1) / kTile);
        const int expert = tile_m / tiles_per_expert;
        const int64_t row = static_cast<int64_t>(tile_m - expert * tiles_per_expert) * kTile;
        const int64_t col0 = static_cast<int64_t>(tile_n) * kTile;
        rows_valid = static_cast<int>(min(static_cast<int64_t>(kTile), args.sparse_size - row));
        cols_valid = static_cast<int>(min(static_cast<int64_t>(kTile), args.cols - col0));
        if (args.expert_ends != nullptr) {
            k_lo = expert > 0 ? load_index(args.expert_ends, args.index_dtype, expert - 1) : 0;
            k_hi = load_index(args.expert_pad_begins, args.index_dtype, expert);
            k_lo = max(k_lo, static_cast<int64_t>(0));
            k_hi = min(k_hi, args.inner);
        } else if (args.piece_length > 0) {
            k_lo = expert * args.piece_length;
            k_hi = min(k_lo + args.piece_length, args.inner);
        }
        lhs_offset = row * args.lhs_stride_row + k_lo * args.lhs_stride_inner;
        rhs_offset = col0 * args.rhs_stride_col + k_lo * args.rhs_stride_inner;
        out_offset = (expert * args.sparse_size + row) * args.out_stride_row + col0;
    } else {
        RowTile tile;
        if (!locate_tile<kTile>(args, logical, tile)) return;
        const int64_t col0 = static_cast<int64_t>(tile.tile_n) * kTile;
        rows_valid = tile.rows_valid;
        cols_valid = static_cast<int>(min(static_cast<int64_t>(kTile), args.cols - col0));
        lhs_offset = tile.row0 * args.lhs_stride_row;
        out_offset = tile.row0 * args.out_stride_row + col0;
        rhs_offset = args.mode == kOutputSparse
                         ? (static_cast<int64_t>(tile.expert) * args.sparse_size + col0) * args.rhs_stride_col
                         : static_cast<int64_t>(tile.expert) * args.sparse_size * args.rhs_stride_inner + col0 * args.rhs_stride_col;
    }
    const int k_count = __builtin_amdgcn_readfirstlane(static_cast<int>(max(k_hi - k_lo, static_cast<int64_t>(0))));
    const int num_slices = (k_count + kBK - 1) / kBK;
    rows_valid = __builtin_amdgcn_readfirstlane(rows_valid);
    cols_valid = __builtin_amdgcn_readfirstlane(cols_valid);

    const int lane = threadIdx.x & 63, half = lane >> 5, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wave_m = kWavesK > 1 ? 0 : wave / kWavesN, wave_n = kWavesK > 1 ? 0 : wave % kWavesN;
    const int first_step = kWavesK > 1 ? wave * kSteps : 0;
    const int lhs_row = wave_m * kWaveTile + (lane & 31), rhs_row = wave_n * kWaveTile + (lane & 31);

    Lhs lhs;
    Rhs rhs;
    lhs.setup(reinterpret_cast<const char *>(static_cast<const float *>(args.lhs) + lhs_offset),
              (kLhsK ? args.lhs_stride_row : args.lhs_stride_inner) * 4, rows_valid, k_count, wave, lane);
    rhs.setup(reinterpret_cast<const char *>(static_cast<const float *>(args.rhs) + rhs_offset),
              (kRhsK ? args.rhs_stride_col : args.rhs_stride_inner) * 4, cols_valid, k_count, wave, lane);
    f32x16_t acc[kBlocks][kBlocks];
#pragma unroll
    for (int i = 0; i < kBlocks; ++i)
#pragma unroll
        for (int j = 0; j < kBlocks; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

    // Slice t sits in slot t % kStages. The barrier of iteration t makes slice t visible (every wavefront has waited
    // for its own loads of it first; loads complete in order) and ends the reads of slice t - 1, whose slot the loads
    // of slice t + kStages - 1 then fill. Slices past the last one are fetched as zeros.
    int fetch_slot = 0;
    auto fetch_slice = [&]() {
        lhs.fetch(lds + fetch_slot, wave);
        rhs.fetch(lds + fetch_slot + Lhs::kBytes, wave);
        fetch_slot = fetch_slot == (kStages - 1) * kSlotBytes ? 0 : fetch_slot + kSlotBytes;
    };
#pragma unroll
    for (int s = 0; s < kStages - 1; ++s) fetch_slice();
    int slot = lds;
    for (int t = 0; t < num_slices; ++t) {
        wait_for_loads<(kStages - 2) * kLoads>();
        __syncthreads();
        fetch_slice();
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            const int q = first_step + s;
            float a[kBlocks][4], b[kBlocks][4];
#pragma unroll
            for (int i = 0; i < kBlocks; ++i) {
                Lhs::fragment(slot, lhs_row + i * 32, q, half, a[i]);
                Rhs::fragment(slot + Lhs::kBytes, rhs_row + i * 32, q, half, b[i]);
            }
            // Operands swapped: a lane holds one row of the tile and groups of four consecutive columns.
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int i = 0; i < kBlocks; ++i)
#pragma unroll
                    for (int j = 0; j < kBlocks; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(b[j][k], a[i][k], acc[i][j], 0, 0, 0);
        }
        slot = slot == lds + (kStages - 1) * kSlotBytes ? lds : slot + kSlotBytes;
    }
    wait_for_loads<0>();  // the zero-filling loads past the end still write LDS

    auto store = [&](int row, int column, f32x4_t value) {
        if (row >= rows_valid || column >= cols_valid) return;  // cols_valid is a multiple of 4
        float *target = static_cast<float *>(args.out) + out_offset + row * args.out_stride_row + column;
        if (args.accumulate) value += *reinterpret_cast<const f32x4_t *>(target);
        *reinterpret_cast<f32x4_t *>(target) = value;
    };
    if constexpr (kWavesK == 1) {
#pragma unroll
        for (int i = 0; i < kBlocks; ++i)
#pragma unroll
            for (int j = 0; j < kBlocks; ++j)
#pragma unroll
                for (int g = 0; g < 4; ++g)
                    store(lhs_row + i * 32, wave_n * kWaveTile + j * 32 + 8 * g + 4 * half,
                          f32x4_t{acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]});
    } else {
        // Wavefront w finishes columns 8 w .. 8 w + 7: the four partial sums, in wavefront order.
        __syncthreads();
        const auto part = [&](int from, int g) { return (FM_LDS(f32x4_t) *)static_cast<uintptr_t>(lds + ((from * 4 + g) * 64 + lane) * 16); };
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *part(wave, g) = f32x4_t{acc[0][0][4 * g], acc[0][0][4 * g + 1], acc[0][0][4 * g + 2], acc[0][0][4 * g + 3]};
        __syncthreads();
        f32x4_t sum = *part(0, wave);
#pragma unroll
        for (int w = 1; w < kWavesK; ++w) sum += *part(w, wave);
        store(lane & 31, 8 * wave + 4 * half, sum);
    }
}

}  // namespace f32

bool f32_gemm_eligible(const GemmArgs &args, int dtype) {
    if (dtype != FM_DTYPE_F32 || args.out_dtype != FM_DTYPE_F32 || args.out_stride_col != 1) return false;
    const bool lhs_k = args.lhs_stride_inner == 1, lhs_m = args.lhs_stride_row == 1;
    const bool rhs_k = args.rhs_stride_inner == 1, rhs_n = args.rhs_stride_col == 1;
    if (!(lhs_k || lhs_m) || !(rhs_k || rhs_n)) return false;
    // A ragged reduction range can start at any K-row of row-contiguous operands, at no K of the others.
    if (args.mode == kInputRowSparse && args.expert_ends != nullptr && (lhs_k || rhs_k)) return false;
    const auto vector_ok = [](const void *pointer, int64_t stride) { return aligned16(pointer) && stride % 4 == 0; };
    if (!vector_ok(args.lhs, lhs_k ? args.lhs_stride_row : args.lhs_stride_inner) ||
        !vector_ok(args.rhs, rhs_k ? args.rhs_stride_col : args.rhs_stride_inner) ||
        !vector_ok(args.out, args.out_stride_row))
        return false;
    // 16-byte chunks must not straddle the end of an axis or of an expert's block.
    if (args.inner <= 0 || args.inner % 4 != 0 || args.sparse_size % 4 != 0 || args.cols % 4 != 0) return false;
    // Rows along the contiguous axis: an expert may start at any of them, and the last chunk would then end past the last row.
    if (!lhs_k && args.mode != kInputRowSparse && (args.rows % 4 != 0 || args.expert_ends != nullptr)) return false;
    if (args.inner >= (int64_t(1) << 30)) return false;
    // Per-lane byte offsets inside a slice are below 2^31: at most 64 lines.
    return max(max(args.lhs_stride_row, args.lhs_stride_inner), max(args.rhs_stride_inner, args.rhs_stride_col)) < (int64_t(1) << 21);
}

template <int kTile, int kBK, int kStages>
static int launch_f32_tile(GemmArgs args, int64_t tiles, hipStream_t stream) {
    const bool lhs_k = args.lhs_stride_inner == 1, rhs_k = args.rhs_stride_inner == 1;
    const auto kernel = lhs_k ? (rhs_k ? f32::grouped_gemm_f32_kernel<kTile, kBK, kStages, true, true>
                                       : f32::grouped_gemm_f32_kernel<kTile, kBK, kStages, true, false>)
                              : (rhs_k ? f32::grouped_gemm_f32_kernel<kTile, kBK, kStages, false, true>
                                       : f32::grouped_gemm_f32_kernel<kTile, kBK, kStages, false, false>);
    // Runs of 64 tiles per XCD (8 row tiles x 8 column tiles), shorter if they would not reach all XCDs.
    args.chunk_tiles = static_cast<int>(min(int64_t(64), (tiles + 7) / 8));
    const int64_t round = 8 * static_cast<int64_t>(args.chunk_tiles);
    const int64_t grid = (tiles + round - 1) / round * round;
    if (grid >= (int64_t(1) << 31)) return fail(FM_ERR_UNSUPPORTED, "grouped gemm: too many tiles");
    constexpr int kLds = kStages * 2 * kTile * kBK * 4;
    static_assert(kLds <= 160 * 1024 / 8, "eight workgroups per CU");
    kernel<<<static_cast<uint32_t>(grid), f32::kThreads, kLds, stream>>>(args);
    return FM_OK;
}

// Fewer tiles of 64 x 64 than this (six per CU; an upper bound of the tiles that exist is counted): tiles of 32 x 32.
// us, 64 / 32: 160 tiles 20 / 13, 400 tiles 100 / 47, 560 tiles 55 / 27, 640 tiles 15.5 / 14.3, 1056 tiles 36 / 34, 1120
// tiles 24 / 26, 1408 tiles 295 / 265, 2048 tiles 23 / 29, 3872 tiles 238 / 254.
constexpr int64_t kF32LargeTiles = 1536;

int f32_gemm_launch(GemmArgs args, hipStream_t stream) {
    // Upper bounds of the numbers of tiles (the surplus ids have none).
    const auto count = [&](int tile) {
        if (args.mode == kInputRowSparse)
            args.tiles_m = static_cast<int>((args.sparse_size + tile - 1) / tile) * args.num_experts;
        else
            args.tiles_m = static_cast<int>((args.rows + tile - 1) / tile + (args.num_experts > 1 ? args.num_experts : 0));
        args.tiles_n = static_cast<int>((args.cols + tile - 1) / tile);
        return static_cast<int64_t>(args.tiles_m) * args.tiles_n;
    };
    const int64_t large = count(64);
    if (large >= kF32LargeTiles) return launch_f32_tile<64, 16, 2>(args, large, stream);
    const int64_t small = count(32);
    return launch_f32_tile<32, 32, 2>(args, small, stream);
}

}  // namespace fm
