// Grouped matrix products of fp32 operands on the gfx950 matrix cores, by one of two instructions:
//   * v_mfma_f32_32x32x16_bf16 on operands split into three bf16 parts each (`grouped_gemm_f32_split_kernel`, below): six
//     products of parts instead of one of values at 16 times the rate of fp32 multiply-adds;
//   * v_mfma_f32_32x32x2_f32 (`grouped_gemm_f32_kernel`), for short reductions and few tiles (see `forward_tile`).
// Forward and backward products of 4096 rows over 8 experts, 1024 x 2816 (5632): 1864 us for the six on fp32 multiply-adds, 1345 on
// split operands.
//   * Operand slices (kBK reduction indices) go straight from global memory into LDS (`buffer_load ... lds`, 16 bytes
//     per lane), at least one slice ahead of the multiplications, one barrier per slice. Lanes that have nothing to fetch (rows
//     past the tile's last one, indices past the reduction range) are sent out of the buffer's range and bring zeros.
//   * An operand may be contiguous along K (activations, `weight.t()`): stored [row][K], fragments are 128-bit reads of
//     four K values of one row; or along its other axis (`weight`, `activations.t()`): stored [K][row] as in memory,
//     fragments are 32-bit reads. A group of K values is split over the wavefront's halves, first half and second half;
//     both layouts agree on that, and the order of a sum is free. Chunks are XOR-swizzled on the global side so that
//     fragment reads hit all banks.
//   * Tiles never straddle experts (they are enumerated per expert from `expert_ends`), so any padding multiple works.
#include "fm_gemm_common.h"

namespace fm {

namespace f32 {

typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;
typedef __attribute__((__vector_size__(2 * sizeof(float)))) float f32x2_t;
typedef __attribute__((__vector_size__(8 * sizeof(bf16_t)))) bf16_t bf16x8_t;
typedef __attribute__((__vector_size__(2 * sizeof(bf16_t)))) bf16_t bf16x2_t;

constexpr int kThreads = 256;

// One operand's slice in LDS and the loads that fill it.
// `kGroup`: reduction indices that a wavefront multiplies at a time, the first half of them in its lanes 0..31.
template <int kTile, int kBK, int kGroup, bool kContiguousK>
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
            return c ^ (kChunks > 8 ? (line / (kGroup / 2) & 1) << 3 : 0);
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

    // The lane's K values (kGroup (q + half / 2) + 0, 1, ...) of row `row`, from the slot at byte address `slot`.
    static __device__ __forceinline__ void fragment(int slot, int row, int q, int half, float (&values)[kGroup / 2]) {
        if constexpr (kContiguousK) {
#pragma unroll
            for (int c = 0; c < kGroup / 8; ++c) {
                const int address = slot + (row * kChunks + swizzled(row, (2 * q + half) * (kGroup / 8) + c)) * 16;
                const f32x4_t vector = *(FM_LDS(f32x4_t) *)static_cast<uintptr_t>(address);
#pragma unroll
                for (int i = 0; i < 4; ++i) values[4 * c + i] = vector[i];
            }
        } else if constexpr (kGroup == 8) {
            // An address per value: the multiply-adds' loop then waits for one value after the other. With one address for all of them the
            // reads are all in front of the MFMAs, and launches that are little but stores take longer: weight gradients of 7
            // rows for each of 64 experts, 128 x 8176, 76 -> 86 us.
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int k = 8 * q + 4 * half + i;
                values[i] = *(FM_LDS(float) *)static_cast<uintptr_t>(slot + k * kTile * 4 + swizzled(k, row >> 2) * 16 + (row & 3) * 4);
            }
        } else {
            const int address = slot + (kGroup * q + kGroup / 2 * half) * kTile * 4 + ((row >> 2) ^ (kChunks > 8 ? half << 3 : 0)) * 16 + (row & 3) * 4;
#pragma unroll
            for (int i = 0; i < kGroup / 2; ++i) values[i] = *(FM_LDS(float) *)static_cast<uintptr_t>(address + i * kTile * 4);
        }
    }
};

template <int kNewest>
__device__ __forceinline__ void wait_for_loads() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kNewest) : "memory");
}

// Where a workgroup's tile and its operands lie.
struct TileOperands {
    int64_t lhs_offset, rhs_offset, out_offset;  // elements
    int rows_valid, cols_valid, k_count;
    bool exists;
};

template <int kTileM, int kTileN>
__device__ __forceinline__ TileOperands find_tile(const GemmArgs &args) {
    TileOperands found;
    found.exists = false;
    // Consecutive workgroup ids go to the 8 XCDs in turn; an XCD gets runs of `chunk_tiles` consecutive logical tiles.
    const int pid = blockIdx.x, local = pid / 8;
    const int logical = (local / args.chunk_tiles * 8 + pid % 8) * args.chunk_tiles + local % args.chunk_tiles;
    int64_t k_lo = 0, k_hi = args.inner;
    if (args.mode == kInputRowSparse) {
        if (logical >= args.tiles_m * args.tiles_n) return found;
        int tile_m, tile_n;
        tile_coordinates(logical, args.tiles_m, args.tiles_n, tile_m, tile_n);
        const int tiles_per_expert = static_cast<int>((args.sparse_size + kTileM - 1) / kTileM);
        const int expert = tile_m / tiles_per_expert;
        const int64_t row = static_cast<int64_t>(tile_m - expert * tiles_per_expert) * kTileM;
        const int64_t col0 = static_cast<int64_t>(tile_n) * kTileN;
        found.rows_valid = static_cast<int>(min(static_cast<int64_t>(kTileM), args.sparse_size - row));
        found.cols_valid = static_cast<int>(min(static_cast<int64_t>(kTileN), args.cols - col0));
        if (args.expert_ends != nullptr) {
            k_lo = expert > 0 ? load_index(args.expert_ends, args.index_dtype, expert - 1) : 0;
            k_hi = load_index(args.expert_pad_begins, args.index_dtype, expert);
            k_lo = max(k_lo, static_cast<int64_t>(0));
            k_hi = min(k_hi, args.inner);
        } else if (args.piece_length > 0) {
            k_lo = expert * args.piece_length;
            k_hi = min(k_lo + args.piece_length, args.inner);
        }
        found.lhs_offset = row * args.lhs_stride_row + k_lo * args.lhs_stride_inner;
        found.rhs_offset = col0 * args.rhs_stride_col + k_lo * args.rhs_stride_inner;
        found.out_offset = (expert * args.sparse_size + row) * args.out_stride_row + col0;
    } else {
        RowTile tile;
        if (!locate_tile<kTileM>(args, logical, tile)) return found;
        const int64_t col0 = static_cast<int64_t>(tile.tile_n) * kTileN;
        found.rows_valid = tile.rows_valid;
        found.cols_valid = static_cast<int>(min(static_cast<int64_t>(kTileN), args.cols - col0));
        found.lhs_offset = tile.row0 * args.lhs_stride_row;
        found.out_offset = tile.row0 * args.out_stride_row + col0;
        found.rhs_offset = args.mode == kOutputSparse
                         ? (static_cast<int64_t>(tile.expert) * args.sparse_size + col0) * args.rhs_stride_col
                         : static_cast<int64_t>(tile.expert) * args.sparse_size * args.rhs_stride_inner + col0 * args.rhs_stride_col;
    }
    found.k_count = __builtin_amdgcn_readfirstlane(static_cast<int>(max(k_hi - k_lo, static_cast<int64_t>(0))));
    found.rows_valid = __builtin_amdgcn_readfirstlane(found.rows_valid);
    found.cols_valid = __builtin_amdgcn_readfirstlane(found.cols_valid);
    found.exists = true;
    return found;
}

// fp32 multiply-adds. An MFMA of this kind keeps the matrix pipe busy for 64 cycles and needs two 256-byte operand fragments, so
// neither LDS nor address arithmetic is near a limit; what has to be hidden is memory latency, and many small workgroups per CU
// hide it better than deep pipelines: eight of them (16 KiB of LDS, at most 64 registers per lane), each one slice ahead.
//   64 x 64, 4 wavefronts of 32 x 32;
//   32 x 32, the 4 wavefronts take a quarter of every slice each and add up in LDS: four times the workgroups, for
//   launches whose outputs are too few to fill the CUs otherwise.
template <int kTile, int kBK, int kStages, bool kLhsK, bool kRhsK>
__global__ __launch_bounds__(kThreads, 8) void grouped_gemm_f32_kernel(GemmArgs args) {
    constexpr int kWavesK = kTile == 32 ? 4 : 1, kWavesN = kTile == 32 ? 1 : 2;
    constexpr int kWaveTile = kTile / kWavesN, kBlocks = kWaveTile / 32;
    typedef Operand<kTile, kBK, 8, kLhsK> Lhs;
    typedef Operand<kTile, kBK, 8, kRhsK> Rhs;
    constexpr int kSlotBytes = Lhs::kBytes + Rhs::kBytes, kLoads = Lhs::kLoads + Rhs::kLoads;
    constexpr int kSteps = kBK / 8 / kWavesK;  // groups of eight K values per wavefront and slice
    extern __shared__ __attribute__((aligned(1024))) char lds_generic[];
    const int lds = static_cast<int>(reinterpret_cast<uintptr_t>((FM_LDS(char) *)lds_generic));

    const TileOperands tile = find_tile<kTile, kTile>(args);
    if (!tile.exists) return;
    const int k_count = tile.k_count, rows_valid = tile.rows_valid, cols_valid = tile.cols_valid;
    const int64_t lhs_offset = tile.lhs_offset, rhs_offset = tile.rhs_offset, out_offset = tile.out_offset;
    const int num_slices = (k_count + kBK - 1) / kBK;
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

// ---- operands split into bf16 parts ---------------------------------------------------------------------------------------
// A value is the sum of three bf16 (8 significant bits each): the nearest to it, to the rest, and to the rest of that. Of the nine
// products of two values' parts, the six above 2^-25 of the whole are taken, in fp32 accumulators of their own for the five small
// kinds, so that the large sum is rounded once per 16 reduction indices (every 2 on fp32 multiply-adds) and results are nearer to
// 64 bits than those: relative 1.9e-7 against 5.7e-7 (layer 1, 1024 reduction indices), 1.6e-7 against 4.8e-7 (layer 2, 2816),
// 1.3e-7 against 4.1e-7 (weight gradients, 512), and for all shapes and products measured.
//
// Every value is multiplied by 2^24 first. bf16 has the exponents of fp32 but 8 bits, so the second and third part of a value below
// 2^-110 would lie under bf16's range whatever the value is multiplied with; scaled, the parts of every fp32 value are
// normal bf16 numbers, and the products of parts that the sums (2^48 of the result) cannot hold are below a result's smallest unit.
// What is lost is the other end: operands from 2^103 and sums from 2^80 on become infinite, which their results show. A result that is
// infinite or NaN is taken from fp32 multiply-adds: its tile is computed again, on two workgroups per CU (layer 1 of the above with a
// NaN in one row 304 -> 331 us, with one in every tile 655, where fp32 multiply-adds in the first place take 390). The six products
// take 5 % longer for the scaling; one vector instruction per value is also what it takes to look for values that are too small.
//
// Every wavefront splits the fragments it multiplies: 8.7 vector instructions per MFMA of 32 cycles, interleaved with the MFMAs of
// the fragments before (two wavefronts per SIMD; 6 such instructions cost an MFMA nothing, and the residual as a bf16 dot product,
// half as many instructions, 5 cycles each of the matrix pipe). Splitting once per workgroup instead would move 6 bytes per
// element through LDS both ways, which is as long as the MFMAs take. The device then runs at 1.84 GHz: power.
// A wavefront computes 64 x 64 of the tile; the four of them are
//   128 x 128: 2 x 2 of the tile, slices of 16;
//   128 x 64: 2 of the tile x 2 halves of a slice of 32;
//   64 x 64: 4 quarters of a slice of 64
// (halves and quarters add up in LDS), by how many tiles there are: see `forward_tile` and `gradient_tile`.

constexpr float kOperandScale = 0x1p24f, kResultScale = 0x1p-48f;

__device__ __forceinline__ void split(const float (&values)[8], bf16x8_t (&parts)[3]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float rest_0 = values[2 * i] * kOperandScale, rest_1 = values[2 * i + 1] * kOperandScale;
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            const bf16x2_t pair = __builtin_convertvector((f32x2_t{rest_0, rest_1}), bf16x2_t);
            parts[p][2 * i] = pair[0];
            parts[p][2 * i + 1] = pair[1];
            const uint32_t bits = __builtin_bit_cast(uint32_t, pair);
            rest_0 -= __builtin_bit_cast(float, bits << 16);
            rest_1 -= __builtin_bit_cast(float, bits & 0xffff0000u);
        }
    }
}

// Six times: one MFMA, seven vector instructions.
__device__ __forceinline__ void interleave() {
#pragma unroll
    for (int n = 0; n < 6; ++n) {
        __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x2, 7, 0);
    }
}

template <int kTileM, int kTileN, int kStages, bool kLhsK, bool kRhsK>
__global__ __launch_bounds__(kThreads, 2) void grouped_gemm_f32_split_kernel(GemmArgs args) {
    constexpr int kWavesM = kTileM / 64, kWavesN = kTileN / 64, kWavesK = 4 / (kWavesM * kWavesN), kBK = 16 * kWavesK;
    typedef Operand<kTileM, kBK, 16, kLhsK> Lhs;
    typedef Operand<kTileN, kBK, 16, kRhsK> Rhs;
    constexpr int kSlotBytes = Lhs::kBytes + Rhs::kBytes, kLoads = Lhs::kLoads + Rhs::kLoads;
    extern __shared__ __attribute__((aligned(1024))) char lds_generic[];
    const int lds = static_cast<int>(reinterpret_cast<uintptr_t>((FM_LDS(char) *)lds_generic));
    const TileOperands tile = find_tile<kTileM, kTileN>(args);
    if (!tile.exists) return;
    const int num_slices = (tile.k_count + kBK - 1) / kBK;
    const int lane = threadIdx.x & 63, half = lane >> 5, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wave_k = wave % kWavesK, wave_m = wave / kWavesK / kWavesN, wave_n = wave / kWavesK % kWavesN;
    const int lhs_row = wave_m * 64 + (lane & 31), rhs_row = wave_n * 64 + (lane & 31);

    // Slice t sits in slot t % kStages; slices past the last one are fetched as zeros.
    Lhs lhs;
    Rhs rhs;
    int fetch_slot;
    const auto fetch_slice = [&]() {
        lhs.fetch(lds + fetch_slot, wave);
        rhs.fetch(lds + fetch_slot + Lhs::kBytes, wave);
        fetch_slot = fetch_slot == (kStages - 1) * kSlotBytes ? 0 : fetch_slot + kSlotBytes;
    };
    const auto start = [&]() {
        lhs.setup(reinterpret_cast<const char *>(static_cast<const float *>(args.lhs) + tile.lhs_offset),
                  (kLhsK ? args.lhs_stride_row : args.lhs_stride_inner) * 4, tile.rows_valid, tile.k_count, wave, lane);
        rhs.setup(reinterpret_cast<const char *>(static_cast<const float *>(args.rhs) + tile.rhs_offset),
                  (kRhsK ? args.rhs_stride_col : args.rhs_stride_inner) * 4, tile.cols_valid, tile.k_count, wave, lane);
        fetch_slot = 0;
#pragma unroll
        for (int s = 0; s < kStages - 1; ++s) fetch_slice();
    };
    // Every wavefront has waited for its loads of the slice after those in flight, and has read the slice before it: that
    // slice is visible after the barrier, and the slot of the one before can be filled.
    const auto next_slice = [&]() {
        wait_for_loads<(kStages - 2) * kLoads>();
        __syncthreads();
        fetch_slice();
    };
    float a[2][8], b[2][8];
    const auto read = [&](int slot, int i) {
        Lhs::fragment(lds + slot, lhs_row + i * 32, wave_k, half, a[i]);
        Rhs::fragment(lds + slot + Lhs::kBytes, rhs_row + i * 32, wave_k, half, b[i]);
    };
    // Operands swapped in all MFMAs: a lane holds one row of a block of 32 x 32 and groups of four consecutive columns.
    f32x16_t acc[2][2];
    {
        f32x16_t small[2][2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = small[i][j][v] = 0.f;
        bf16x8_t a_parts[2][3], b_parts[2][3];
        const auto multiply = [&](int i, int j) {
#pragma unroll
            for (int sum = 2; sum >= 0; --sum)
#pragma unroll
                for (int p = 0; p <= sum; ++p) {
                    f32x16_t &target = sum == 0 ? acc[i][j] : small[i][j];
                    target = __builtin_amdgcn_mfma_f32_32x32x16_bf16(b_parts[j][sum - p], a_parts[i][p], target, 0, 0, 0);
                }
        };
        start();
        next_slice();
        read(0, 0);
        read(0, 1);
        split(a[0], a_parts[0]);
        split(b[0], b_parts[0]);
        int next = 0;  // slot of the slice to read
        for (int t = 0; t < num_slices; ++t) {
            // Here the first fragments of slice t are split, the second ones read.
            next = next == (kStages - 1) * kSlotBytes ? 0 : next + kSlotBytes;
            next_slice();
            read(next, 0);
            split(b[1], b_parts[1]);
            multiply(0, 0);
            interleave();
            split(a[1], a_parts[1]);
            multiply(0, 1);
            interleave();
            read(next, 1);
            bf16x8_t a_next[3], b_next[3];
            split(a[0], a_next);
            multiply(1, 0);
            interleave();
            split(b[0], b_next);
            multiply(1, 1);
            interleave();
#pragma unroll
            for (int p = 0; p < 3; ++p) {
                a_parts[0][p] = a_next[p];
                b_parts[0][p] = b_next[p];
            }
        }
        wait_for_loads<0>();  // the zero-filling loads past the end still write LDS
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acc[i][j] += small[i][j];
    }

    // The sums over the wavefronts that share a reduction, in wavefront order; each then holds kHeld of its four blocks.
    constexpr int kHeld = 4 / kWavesK;
    const auto add_shares = [&]() {
        if constexpr (kWavesK > 1) {
            static_assert(kStages * kSlotBytes >= 4 * 4 * 4096 || kWavesK == 1, "space for four wavefronts' blocks");
            const auto share = [&](int from, int g) { return (FM_LDS(f32x4_t) *)static_cast<uintptr_t>(lds + ((from * 16 + g) * 64 + lane) * 16); };
            __syncthreads();
#pragma unroll
            for (int g = 0; g < 16; ++g) {
                const f32x16_t &block = acc[g / 8][g / 4 % 2];
                *share(wave, g) = f32x4_t{block[g % 4 * 4], block[g % 4 * 4 + 1], block[g % 4 * 4 + 2], block[g % 4 * 4 + 3]};
            }
            __syncthreads();
#pragma unroll
            for (int g = 0; g < 4 * kHeld; ++g) {
                f32x4_t sum = *share(wave - wave_k, wave_k * 4 * kHeld + g);
#pragma unroll
                for (int w = 1; w < kWavesK; ++w) sum += *share(wave - wave_k + w, wave_k * 4 * kHeld + g);
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[g / 8][g / 4 % 2][g % 4 * 4 + v] = sum[v];
            }
        }
    };
    add_shares();
    const auto in_doubt = [](float value) { return !__builtin_isfinite(value); };
    bool again = false;
#pragma unroll
    for (int held = 0; held < kHeld; ++held)
#pragma unroll
        for (int v = 0; v < 16; ++v) again |= in_doubt(acc[held / 2][held % 2][v]);
    if (__syncthreads_or(again)) {
        f32x16_t first[2][2];
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                first[i][j] = acc[i][j];
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;
            }
        start();
        int slot = 0;
        for (int t = 0; t < num_slices; ++t) {
            next_slice();
            read(slot, 0);
            read(slot, 1);
#pragma unroll
            for (int k = 0; k < 8; ++k)
#pragma unroll
                for (int i = 0; i < 2; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(b[j][k], a[i][k], acc[i][j], 0, 0, 0);
            slot = slot == (kStages - 1) * kSlotBytes ? 0 : slot + kSlotBytes;
        }
        wait_for_loads<0>();
        add_shares();
        // What was in no doubt stays: the other rows and columns of the tile, padding with whatever it holds, change nobody's result.
#pragma unroll
        for (int held = 0; held < kHeld; ++held)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const float value = first[held / 2][held % 2][v];
                if (!in_doubt(value)) acc[held / 2][held % 2][v] = value * kResultScale;
            }
    } else {
#pragma unroll
        for (int held = 0; held < kHeld; ++held)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[held / 2][held % 2][v] *= kResultScale;
    }
#pragma unroll
    for (int held = 0; held < kHeld; ++held) {
        const int block = wave_k * kHeld + held;
        const int row = wave_m * 64 + block / 2 * 32 + (lane & 31);
        if (row >= tile.rows_valid) continue;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            const int column = wave_n * 64 + block % 2 * 32 + 8 * g + 4 * half;
            if (column >= tile.cols_valid) continue;  // a multiple of 4
            const f32x16_t &from = acc[held / 2][held % 2];
            f32x4_t value = f32x4_t{from[4 * g], from[4 * g + 1], from[4 * g + 2], from[4 * g + 3]};
            float *target = static_cast<float *>(args.out) + tile.out_offset + row * args.out_stride_row + column;
            if (args.accumulate) value += *reinterpret_cast<const f32x4_t *>(target);
            *reinterpret_cast<f32x4_t *>(target) = value;
        }
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
    // Per-lane byte offsets inside a slice are below 2^31: at most 128 lines.
    return max(max(args.lhs_stride_row, args.lhs_stride_inner), max(args.rhs_stride_inner, args.rhs_stride_col)) < (int64_t(1) << 21);
}

template <int kTileM, int kTileN, int kStages>
static int launch_f32_split(GemmArgs args, int64_t tiles, hipStream_t stream) {
    const bool lhs_k = args.lhs_stride_inner == 1, rhs_k = args.rhs_stride_inner == 1;
    const auto kernel = lhs_k ? (rhs_k ? f32::grouped_gemm_f32_split_kernel<kTileM, kTileN, kStages, true, true>
                                       : f32::grouped_gemm_f32_split_kernel<kTileM, kTileN, kStages, true, false>)
                              : (rhs_k ? f32::grouped_gemm_f32_split_kernel<kTileM, kTileN, kStages, false, true>
                                       : f32::grouped_gemm_f32_split_kernel<kTileM, kTileN, kStages, false, false>);
    // Runs of 16 tiles per XCD (8 row tiles x 2 column tiles): with 32 the XCDs end further apart, with 8 the panels are read more often
    // (six products, us: 1490, 1467, 1477).
    args.chunk_tiles = static_cast<int>(min(int64_t(16), (tiles + 7) / 8));
    const int64_t round = 8 * static_cast<int64_t>(args.chunk_tiles);
    const int64_t grid = (tiles + round - 1) / round * round;
    if (grid >= (int64_t(1) << 31)) return fail(FM_ERR_UNSUPPORTED, "grouped gemm: too many tiles");
    constexpr int kBK = 16 * 4 * 64 * 64 / (kTileM * kTileN), kLds = kStages * (kTileM + kTileN) * kBK * 4;
    static_assert(kLds <= 80 * 1024, "two workgroups per CU");
    if constexpr (kLds > 64 * 1024) {
        static std::atomic<uint64_t> configured[4];
        if (int status = allow_lds(reinterpret_cast<const void *>(kernel), kLds, configured[2 * lhs_k + rhs_k])) return status;
    }
    kernel<<<static_cast<uint32_t>(grid), f32::kThreads, kLds, stream>>>(args);
    return FM_OK;
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

// Which kernel and tile, by the 64 x 64 tiles that the rows are expected to fill (half a tile per expert of a map is not; a buffer's own
// rows are mostly padding where experts have few). Short reductions are start and epilogue, and what few tiles there are runs on more CUs
// as tiles of 32 x 32: there eight workgroups of fp32 multiply-adds per CU are faster. Time over that on multiply-adds, operands not in
// L2, geometric means over 8500 grouped products of 2 to 128 experts of 1 to 800 rows, equally and unequally liked, 64 x 64 / 128 x 64 / 128 x
// 128 on split operands; first line of a pair: experts of up to 32 rows, second: of more.
//     tiles          reduction 96 .. 127   192 .. 255          384 .. 511          768 .. 1023         from 2048 on
//     up to 255      1.24 1.38 1.58    1.16 1.31 1.59    1.01 1.16 1.51    0.92 1.08 1.56    0.82 0.98 1.54
//                    1.27 1.46 1.66    1.18 1.35 1.65    1.06 1.26 1.69    0.94 1.14 1.69    0.85 1.06 1.72
//     256 .. 511     1.15 1.03 0.92    1.00 0.91 0.84    0.85 0.80 0.80    0.78 0.74 0.71    0.68 0.67 0.68
//                    1.06 1.01 1.04    1.02 0.95 1.02    0.86 0.84 0.93    0.77 0.78 0.95    0.71 0.72 0.92
//     512 .. 1023    1.32 1.11 0.95    1.14 0.97 0.86    0.94 0.82 0.78    0.77 0.71 0.73    0.66 0.68 0.73
//                    1.11 0.97 0.89    1.02 0.92 0.86    0.86 0.79 0.82    0.79 0.75 0.78    0.70 0.71 0.73
//     1024 .. 2499   1.37 1.10 0.91    1.13 0.91 0.78    0.86 0.73 0.72    0.75 0.68 0.68
//                    1.32 1.11 0.97    1.13 0.95 0.86    0.94 0.81 0.81    0.80 0.74 0.76    0.68 0.69 0.71
//     more           1.56 1.16 0.88    1.22 0.93 0.75
//                    1.48 1.12 0.89    1.19 0.91 0.76    0.93 0.77 0.72    0.79 0.71 0.68
// Experts of few rows (64 by the estimate) are weights read from memory: large tiles, which start over less often, are ahead early. In a
// layer, whose activations are in cache, long reductions and more rows are better off on small ones, and their lines are drawn for that
// (us on 64 x 64 / 128 x 64 / 128 x 128: 16 experts of 37 rows, 1024 columns of 2816 (336 tiles) 53 / 79, of 48 rows, 5632 of 1024 115 / 154 /
// 147; 8 of 37, 2496 of 960 26 / 44; 8 of 266, 2048 of 512 (1184) 45 / - / 51; 8 of 512, 1024 of 2816 (1088) 181 / 194 / 228, 2816 of 1024 (2992)
// 161 / 157 / 158, 5632 of 1024 (5984) 333 / 300 / 298).
// A side of up to 32 leaves half of every split tile empty, up to 16 columns three quarters: 16384 x 32 of 256 7 us on multiply-adds
// against 10, of 2816 66 against 51; 39467 x 8 of 1328 80 against 92. By the rule the grouped products take 0.945 of the time of
// multiply-adds (worst 1.18; the best choice for each 0.913), 3000 dense ones of 1 to 65536 rows 0.95 (0.93).
constexpr int64_t kF32LargeTiles = 1536;  // of fp32 multiply-adds, by their upper bound: 1056 36 (32 x 32: 34), 1120 24 (26), 1408 295
                                          // (265), 2048 23 (29), 3872 238 (254)
enum class F32Tile { kMultiplyAdds, k64x64, k128x64, k128x128 };

static F32Tile forward_tile(int64_t rows, int64_t cols, int64_t reduction, int64_t tiles, bool mapped) {
    if (cols <= 16) return F32Tile::kMultiplyAdds;
    if (mapped && rows <= 64 && cols > 32) {
        const int64_t shortest = tiles < 64 ? 1024 : tiles < 256 ? 768 : tiles < 1024 ? 256 : tiles < 2500 ? 128 : 96;
        if (reduction < shortest) return F32Tile::kMultiplyAdds;
        if (tiles < 2500 && reduction >= 768) return F32Tile::k64x64;
        return tiles < 1024 ? F32Tile::k128x64 : F32Tile::k128x128;
    }
    const int64_t shortest = tiles < 64 ? 1024 : tiles < 400 ? 512 : tiles < 700 ? 384 : tiles < 1536 ? 256 : tiles < 2500 ? 192 : 128;
    const bool narrow = cols <= 32 || (!mapped && rows <= 32);
    if (reduction < (narrow ? max(shortest, int64_t(768)) : shortest)) return F32Tile::kMultiplyAdds;
    return tiles < 1200 ? F32Tile::k64x64 : tiles < 2816 ? F32Tile::k128x64 : F32Tile::k128x128;
}

// Weight gradients, the same over 8100 products of 4 to 3000 rows per expert, those where no edge leaves a large tile empty:
//     tiles          reduction 65 .. 128   129 .. 256          257 .. 512          513 .. 1024         2049 .. 4096
//     64 .. 255      1.20 1.37 1.59    1.10 1.31 1.59    0.98 1.23 1.69    0.86 1.12 1.74    0.78 1.07 1.89
//     256 .. 511     1.11 1.10 1.26    1.04 1.06 1.31    0.92 0.96 1.28    0.86 0.89 1.32    0.76 0.81 1.31
//     512 .. 1023    1.16 1.08 0.98    1.07 1.00 0.98    0.95 0.93 1.01    0.85 0.84 0.92    0.75 0.77 0.86
//     1024 .. 2499   1.22 1.08 0.95    1.04 0.94 0.89    0.90 0.86 0.89    0.77 0.75 0.80    0.69 0.72 0.84
//     more           1.53 1.18 0.93    1.19 0.97 0.81    0.92 0.80 0.75    0.78 0.73 0.72    0.66 0.68 0.74
// With the operands in cache, as after the product before, few tiles gain later (128 tiles of 2048 29 us on multiply-adds, 33 so) and large ones
// are ahead earlier (2048 tiles of 266 34 us on 128 x 128, 41 on 128 x 64). Large tiles whose area is a tenth (128 x 64) or a quarter (128 x
// 128) more than that of the 64 x 64 ones waste it: 64 experts, 64 x 3440, 47 rows 42 -> 51 us, 144 x 360, 186 rows 34 -> 39. By the rule
// 0.972 of the time of multiply-adds; 35 of the 8100 are slower than those by more than a tenth (worst 1.45), all but a few with one expert
// that has several times the rows of the others: a long reduction on few tiles.
static F32Tile gradient_tile(int64_t reduction, int64_t tiles, int64_t tiles_128x64, int64_t tiles_128x128) {
    const int64_t area = 4 * 100 * tiles_128x128 / tiles;  // percent of that of the 64 x 64 tiles
    const int64_t shortest = tiles < 64 ? 4096 : tiles < 256 ? 2048 : tiles < 512 ? 512 : tiles < 1024 ? 256 : area < 115 ? 96 : 192;
    if (reduction < shortest) return F32Tile::kMultiplyAdds;
    if (tiles >= 1024 && area < 125) return F32Tile::k128x128;
    return tiles >= 512 && 2 * 10 * tiles_128x64 < 11 * tiles ? F32Tile::k128x64 : F32Tile::k64x64;
}

// Rows per expert that a map's buffer has on top of the tokens': 128 of a static shape, 64 on average of a dynamic one. From the buffer
// alone, whoever calls: the layer's products and those of its parts then sum in the same order.
constexpr int64_t kPadding = 112;

int f32_gemm_launch(GemmArgs args, hipStream_t stream) {
    // Upper bounds of the numbers of tiles (the surplus ids have none).
    const auto count = [&](int tile_m, int tile_n) {
        if (args.mode == kInputRowSparse)
            args.tiles_m = static_cast<int>((args.sparse_size + tile_m - 1) / tile_m) * args.num_experts;
        else
            args.tiles_m = static_cast<int>((args.rows + tile_m - 1) / tile_m + (args.num_experts > 1 ? args.num_experts : 0));
        args.tiles_n = static_cast<int>((args.cols + tile_n - 1) / tile_n);
        return static_cast<int64_t>(args.tiles_m) * args.tiles_n;
    };
    const bool mapped = args.expert_ends != nullptr;
    F32Tile tile = F32Tile::kMultiplyAdds;
    if (args.mode == kInputRowSparse) {
        const int64_t reduction = mapped ? args.inner / args.num_experts - kPadding : args.piece_length > 0 ? args.piece_length : args.inner;
        if (args.sparse_size >= 64 && args.cols >= 64) tile = gradient_tile(reduction, count(64, 64), count(128, 64), count(128, 128));
    } else {
        const int64_t rows = mapped ? max(args.rows / args.num_experts - kPadding, int64_t(1)) : args.rows;
        const int64_t tiles_m = mapped ? args.num_experts * (rows + 32) / 64 : (rows + 63) / 64;
        tile = forward_tile(rows, args.cols, args.inner, tiles_m * ((args.cols + 63) / 64), mapped);
    }
    switch (tile) {  // `count` sets what the kernel goes by
        case F32Tile::k64x64: {
            const int64_t tiles = count(64, 64);
            return launch_f32_split<64, 64, 2>(args, tiles, stream);
        }
        case F32Tile::k128x64: {
            const int64_t tiles = count(128, 64);
            return launch_f32_split<128, 64, 3>(args, tiles, stream);
        }
        case F32Tile::k128x128: {
            const int64_t tiles = count(128, 128);
            return launch_f32_split<128, 128, 3>(args, tiles, stream);
        }
        case F32Tile::kMultiplyAdds: break;
    }
    if (const int64_t tiles = count(64, 64); tiles >= kF32LargeTiles) return launch_f32_tile<64, 16, 2>(args, tiles, stream);
    const int64_t tiles = count(32, 32);
    return launch_f32_tile<32, 32, 2>(args, tiles, stream);
}

}  // namespace fm
