// Weight gradients of experts of few rows on the gfx950 matrix cores (row-sparse product, bf16 / fp16 operands, fp32
// accumulation): out_e [M_s, N] = lhs[rows of e, M_s]^T x rhs[rows of e, N], in tiles of 128 x 256, two workgroups per CU.
//
// The reduction is as long as an expert has rows. Where that is a few hundred, a tile of 256 x 256 that has a CU for itself
// (fm_gemm_mfma.hip) spends 10 to 20 of its 25 to 50 us on filling its pipeline and on its epilogue, with nothing else to run.
// Here the other workgroup of the CU multiplies meanwhile, and the hardware hands out the next tile, whatever each takes. Both
// gradients of a layer with 16 experts of 1280 x 3416: 163 -> 133 us at 94 rows per expert, 262 -> 241 at 375.
//   * Slices of kBK rows go straight from global memory into LDS (`buffer_load ... lds`, 16 bytes per lane), two slices ahead
//     of the multiplications, one barrier per slice. Lanes with nothing to fetch (columns past the operand's, rows past the
//     expert's) are sent out of the buffer's range and bring zeros: a ragged reduction costs nothing, and what padding rows
//     hold cannot leak. Slices of 64 rows with one workgroup per CU and three slots: 340 us where this takes 241.
//   * LDS holds the slices as memory does, [row][column], XOR-swizzled on the global side; `ds_read_b64_tr_b16` hands every
//     lane consecutive rows of its column.
//   * 4 wavefronts in a 2 x 2 grid, 64 x 128 of the tile each, as 2 x 4 accumulators of v_mfma_f32_32x32x16. The order of a sum
//     is that of a tile of 256 x 256: the results are the same bits.
#include <atomic>
#include "fm_gemm_common.h"

namespace fm {

namespace row_sparse {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4_t;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4_t;
typedef __attribute__((__vector_size__(2 * sizeof(uint32_t)))) uint32_t u32x2_t;
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short i16x4_t;

constexpr int kTileM = 128, kTileN = 256, kBK = 32, kStages = 3, kThreads = 256, kWorkgroups = 2;
constexpr int kBlocksM = kTileM / 64, kBlocksN = kTileN / 64, kWaveCols = kTileN / 2;

__device__ __forceinline__ f32x16_t mfma(bf16_t, u32x4_t a, u32x4_t b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x16_t mfma(f16_t, u32x4_t a, u32x4_t b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// One operand's slice in LDS, [kBK rows][kColumns], and the loads that fill it.
template <int kColumns>
struct Operand {
    static constexpr int kBytes = kColumns * kBK * 2, kChunks = kColumns / 8;  // 16-byte chunks per row
    static constexpr int kLoads = kBytes / 16 / kThreads;                      // per lane and slice
    static constexpr uint32_t kOutOfRange = 0x80000000u, kRange = 0x7fffffffu;

    // Where chunk `c` of row `k` sits among the row's chunks: the four rows x 32 bytes that a transpose read takes from one
    // column of chunks then lie in different banks.
    static __device__ __forceinline__ int swizzled(int k, int c) { return c ^ ((k & 3) << 2); }

    const char *base;         // wave-uniform: element (first row of the next slice to fetch, first column of the tile)
    int64_t step;             // bytes from one slice to the next
    uint32_t offset[kLoads];  // per lane, bytes from `base`; out of range where there is nothing to fetch
    int row[kLoads];          // of the slice
    int rows_left;            // from `base` on

    // `stride`: bytes between rows. `valid`: columns that exist, a multiple of 8.
    __device__ __forceinline__ void setup(const char *first, int64_t stride, int valid, int rows, int wave, int lane) {
        base = uniform_pointer(first);
        step = kBK * stride;
        rows_left = rows;
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const int slot = (wave * kLoads + j) * 64 + lane, chunk = swizzled(slot / kChunks, slot % kChunks);
            row[j] = slot / kChunks;
            offset[j] = chunk * 8 < valid ? static_cast<uint32_t>(row[j] * stride + chunk * 16) : kOutOfRange;
        }
    }

    // Fetches the next slice into the LDS slot at byte address `slot`.
    __device__ __forceinline__ void fetch(int slot, int wave) {
        const __amdgpu_buffer_rsrc_t resource = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<char *>(uniform_pointer(base)), 0, static_cast<int>(kRange), kBufferResourceFlags);
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const uint32_t lane_offset = row[j] < rows_left ? offset[j] : kOutOfRange;
            const int target = __builtin_amdgcn_readfirstlane(slot + (wave * kLoads + j) * 1024);
            asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                         :
                         : "s"(target), "v"(lane_offset), "s"(resource)
                         : "memory");
        }
        base += step;
        rows_left -= kBK;
    }

    // Per lane, the byte addresses (from a slot's) of the fragments of the wavefront's blocks of 32 columns from `first` on;
    // 16 rows further on is a constant. Lane s of a group of 16 supplies the address of four columns (column + 4 (s % 4) ..)
    // of row k + s / 4 and receives rows k .. k + 3 of column + s.
    static __device__ __forceinline__ void fragment_addresses(int first, int lane, int (&addresses)[kColumns / 64]) {
        const int s = lane & 15, group = lane >> 4, k = ((group >> 1) << 3) + (s >> 2);
#pragma unroll
        for (int i = 0; i < kColumns / 64; ++i) {
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

// A lane holds, of each 32 x 32 accumulator, one row and four groups of four consecutive columns. Per block of 32 rows a
// wavefront passes its values, rounded, through its own LDS region and stores row segments of 16 bytes per lane.
constexpr int kRowBytes = kWaveCols * 2 + 16, kStagingBytes = 32 * kRowBytes;

template <typename T>
__device__ __forceinline__ void store_tile(const f32x16_t (&acc)[kBlocksM][kBlocksN], int staging, T *out, int64_t stride,
                                           int rows_valid, int cols_valid, int wave_m, int wave_n, int lane) {
    constexpr int kLanesPerRow = kWaveCols / 8, kRowsPerRead = 64 / kLanesPerRow, kReads = 32 / kRowsPerRead;
    const int write_base = staging + (lane & 31) * kRowBytes + (lane >> 5) * 8;
    const int read_row = lane / kLanesPerRow, read_column = lane % kLanesPerRow * 8;
    const int read_base = staging + read_row * kRowBytes + read_column * 2;
    const int column = wave_n * kWaveCols + read_column, first_row = wave_m * kBlocksM * 32 + read_row;
    const bool column_ok = column < cols_valid;  // a multiple of 8
#pragma unroll
    for (int i = 0; i < kBlocksM; ++i) {
#pragma unroll
        for (int j = 0; j < kBlocksN; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                struct {
                    T v[4];
                } group;
#pragma unroll
                for (int c = 0; c < 4; ++c) group.v[c] = from_float<T>(acc[i][j][4 * g + c]);
                *(FM_LDS(u32x2_t) *)static_cast<uintptr_t>(write_base + (j * 32 + 8 * g) * 2) = __builtin_bit_cast(u32x2_t, group);
            }
        // One wavefront's own region, and its LDS operations execute in order: no barrier.
        asm volatile("" ::: "memory");
        u32x4_t staged[kReads];
#pragma unroll
        for (int t = 0; t < kReads; ++t)
            staged[t] = *(FM_LDS(u32x4_t) *)static_cast<uintptr_t>(read_base + t * kRowsPerRead * kRowBytes);
#pragma unroll
        for (int t = 0; t < kReads; ++t) {
            const int row = first_row + i * 32 + t * kRowsPerRead;
            if (row < rows_valid && column_ok)
                __builtin_nontemporal_store(staged[t], reinterpret_cast<u32x4_t *>(out + row * stride + column));
        }
        asm volatile("" ::: "memory");
    }
}

template <typename T>
__global__ __launch_bounds__(kThreads, kWorkgroups) void grouped_gemm_row_sparse_kernel(GemmArgs args) {
    typedef Operand<kTileM> Lhs;
    typedef Operand<kTileN> Rhs;
    constexpr int kSlotBytes = Lhs::kBytes + Rhs::kBytes, kLoads = Lhs::kLoads + Rhs::kLoads;
    extern __shared__ __attribute__((aligned(1024))) char lds_generic[];
    const int lds = static_cast<int>(reinterpret_cast<uintptr_t>((FM_LDS(char) *)lds_generic));

    // Consecutive workgroup ids go to the 8 XCDs in turn; an XCD gets runs of `chunk_tiles` consecutive logical tiles.
    const int pid = blockIdx.x, local = pid / 8;
    const int logical = (local / args.chunk_tiles * 8 + pid % 8) * args.chunk_tiles + local % args.chunk_tiles;
    if (logical >= args.tiles_m * args.tiles_n) return;
    int tile_m, tile_n;
    tile_coordinates(logical, args.tiles_m, args.tiles_n, tile_m, tile_n);
    const int tiles_per_expert = static_cast<int>((args.sparse_size + kTileM - 1) / kTileM), expert = tile_m / tiles_per_expert;
    const int64_t row = static_cast<int64_t>(tile_m - expert * tiles_per_expert) * kTileM;
    const int64_t col0 = static_cast<int64_t>(tile_n) * kTileN;
    const int rows_valid = __builtin_amdgcn_readfirstlane(static_cast<int>(min(static_cast<int64_t>(kTileM), args.sparse_size - row)));
    const int cols_valid = __builtin_amdgcn_readfirstlane(static_cast<int>(min(static_cast<int64_t>(kTileN), args.cols - col0)));
    const int64_t begin = expert > 0 ? max(load_index(args.expert_ends, args.index_dtype, expert - 1), static_cast<int64_t>(0)) : 0;
    const int64_t end = min(load_index(args.expert_pad_begins, args.index_dtype, expert), args.inner);
    const int count = __builtin_amdgcn_readfirstlane(static_cast<int>(max(end - begin, static_cast<int64_t>(0))));
    const int num_slices = (count + kBK - 1) / kBK;

    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wave_m = wave / 2, wave_n = wave % 2;
    Lhs lhs;
    Rhs rhs;
    lhs.setup(reinterpret_cast<const char *>(static_cast<const T *>(args.lhs) + begin * args.lhs_stride_inner + row),
              args.lhs_stride_inner * 2, rows_valid, count, wave, lane);
    rhs.setup(reinterpret_cast<const char *>(static_cast<const T *>(args.rhs) + begin * args.rhs_stride_inner + col0),
              args.rhs_stride_inner * 2, cols_valid, count, wave, lane);
    int lhs_addresses[kBlocksM], rhs_addresses[kBlocksN];
    Lhs::fragment_addresses(wave_m * kTileM / 2, lane, lhs_addresses);
    Rhs::fragment_addresses(wave_n * kTileN / 2, lane, rhs_addresses);
    f32x16_t acc[kBlocksM][kBlocksN];
#pragma unroll
    for (int i = 0; i < kBlocksM; ++i)
#pragma unroll
        for (int j = 0; j < kBlocksN; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.f;

    // Slice t sits in slot t % kStages. The barrier of iteration t makes slice t visible (every wavefront has waited for its
    // own loads of it first; loads complete in order) and ends the reads of slice t - 1, whose slot the loads of slice
    // t + kStages - 1 then fill. Slices past the last one are fetched as zeros.
    int fetch_slot = 0;
    const auto fetch_slice = [&]() {
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
        for (int step = 0; step < kBK / 16; ++step) {
            u32x4_t a[kBlocksM], b[kBlocksN];
#pragma unroll
            for (int i = 0; i < kBlocksM; ++i) a[i] = Lhs::fragment(slot + lhs_addresses[i], step);
#pragma unroll
            for (int j = 0; j < kBlocksN; ++j) b[j] = Rhs::fragment(slot + Lhs::kBytes + rhs_addresses[j], step);
            // Operands swapped: a lane holds one row of the tile and groups of four consecutive columns.
#pragma unroll
            for (int i = 0; i < kBlocksM; ++i)
#pragma unroll
                for (int j = 0; j < kBlocksN; ++j) acc[i][j] = mfma(T(), b[j], a[i], acc[i][j]);
        }
        slot = slot == lds + (kStages - 1) * kSlotBytes ? lds : slot + kSlotBytes;
    }
    wait_for_loads<0>();  // the zero-filling loads past the end still write LDS
    __syncthreads();      // the slots become the wavefronts' staging regions
    T *out = static_cast<T *>(args.out) + (expert * args.sparse_size + row) * args.out_stride_row + col0;
    store_tile<T>(acc, lds + wave * kStagingBytes, out, args.out_stride_row, rows_valid, cols_valid, wave_m, wave_n, lane);
}

constexpr int kLdsBytes = kStages * (kTileM + kTileN) * kBK * 2;
static_assert(kLdsBytes * kWorkgroups <= 160 * 1024 && kLdsBytes >= 4 * kStagingBytes, "the workgroups of a CU share its LDS");

template <typename T>
static int launch(const GemmArgs &args, int64_t grid, hipStream_t stream) {
    const auto kernel = grouped_gemm_row_sparse_kernel<T>;
    static std::atomic<uint64_t> configured{0};
    if (int status = allow_lds(reinterpret_cast<const void *>(kernel), kLdsBytes, configured)) return status;
    kernel<<<static_cast<uint32_t>(grid), kThreads, kLdsBytes, stream>>>(args);
    return FM_OK;
}

}  // namespace row_sparse

// Where fm_gemm_row_panel.hip takes no part, up to this many rows per expert, of the rows that the operands have (a layer's buffers have
// about 128 per expert more than it fills). us, 256 x 256 / here, larger and smaller gradient of a layer: 16 rows of 128 experts of 2048 x 768 218 / 163, 115 /
// 88; 250 rows 362 / 344, 198 / 179; 350 rows 421 / 421, 247 / 216; 500 rows 493 / 512, 289 / 260; 1024 rows 770 / 835, 394 /
// 424. 8 experts of 4096 x 14336: 200 rows 726 / 716, 416 / 365; 383 rows 959 / 981, 539 / 492; 600 rows 1210 / 1295, 618 / 643.
// Results that are added to what is there, or stored in 32 bits, are bound by that traffic and no faster here (adding in 32
// bits 5 to 15 % slower).
constexpr int64_t kMaxRowsPerExpert = 512;

// `args` as `mfma_gemm_eligible` takes them.
bool row_sparse_gemm_chosen(const GemmArgs &args, int dtype) {
    return args.mode == kInputRowSparse && args.expert_ends != nullptr && !args.accumulate && args.out_dtype == dtype &&
           args.lhs_stride_row == 1 && args.rhs_stride_col == 1 && args.inner <= kMaxRowsPerExpert * args.num_experts;
}

int row_sparse_gemm_launch(GemmArgs args, int dtype, hipStream_t stream) {
    using namespace row_sparse;
    args.tiles_m = static_cast<int>((args.sparse_size + kTileM - 1) / kTileM) * args.num_experts;
    args.tiles_n = static_cast<int>((args.cols + kTileN - 1) / kTileN);
    const int64_t tiles = static_cast<int64_t>(args.tiles_m) * args.tiles_n;
    // Runs of 64 tiles per XCD (8 row tiles x 8 column tiles), shorter if they would not reach all XCDs.
    args.chunk_tiles = static_cast<int>(min(int64_t(64), (tiles + 7) / 8));
    const int64_t round = 8 * static_cast<int64_t>(args.chunk_tiles), grid = (tiles + round - 1) / round * round;
    if (grid >= (int64_t(1) << 31)) return fail(FM_ERR_UNSUPPORTED, "grouped gemm: too many tiles");
    return dtype == FM_DTYPE_BF16 ? launch<bf16_t>(args, grid, stream) : launch<f16_t>(args, grid, stream);
}

}  // namespace fm
