// Arguments and small device helpers shared by the grouped-GEMM kernels.
#pragma once

#include <atomic>

#include "fm_common.h"

namespace fm {

enum GemmMode { kOutputSparse = 0, kInputInnerSparse = 1, kInputRowSparse = 2 };

// What the MFMA kernel's epilogue does besides storing the product (output-sparse mode, gated MLP):
//   kFusionGatedForward: the product is layer 1's output [rows, 2 * half] = [gate | up]; a tile holds 128 gate columns
//     and the 128 up columns that go with them, `out` (may be null) receives both and `fused_out` [rows, half] receives
//     act(gate) * up;
//   kFusionGatedBackward: the product is the gradient of the activation's output [rows, half]; it is not stored:
//     `fused_in` is layer 1's output, `out` receives the gradient of it (both [rows, 2 * half], same strides) and
//     `fused_out` (may be null) the recomputed activation output.
enum GemmFusion { kFusionNone = 0, kFusionGatedForward = 1, kFusionGatedBackward = 2 };

struct GemmArgs {
    const void *lhs;
    const void *rhs;
    void *out;
    const void *expert_ends;        // null: dense product
    const void *expert_pad_begins;  // row-sparse mode: where a reduction ends; the others: where the rows to compute end (null: at
                                    // `expert_ends`, padding rows too)
    int64_t lhs_stride_row, lhs_stride_inner, rhs_stride_inner, rhs_stride_col, out_stride_row, out_stride_col;
    int64_t rows;         // rows of out
    int64_t cols;         // columns of out
    int64_t inner;        // length of the reduction axis as stored (per expert for input-inner-sparse)
    int64_t sparse_size;  // N_s, K_s or M_s
    int num_experts;
    int mode;
    int accumulate;
    int index_dtype;
    int out_dtype;
    int tiles_m, tiles_n;
    float *partials;  // the caller's workspace when the MFMA kernel splits reductions, else null; set by its launcher
    int fusion;       // GemmFusion
    int activation;   // fm_activation tag, for the fused epilogues
    const void *fused_in;
    void *fused_out;
    int64_t fused_stride;  // row stride of fused_out, elements
    int64_t half;          // columns of the activation output per expert
    int any_half;          // gated forward: it need not be a multiple of 128
    int num_ids;           // workgroup ids that may have a tile (set by the MFMA kernel's launcher)
    void *tile_table;      // one record per id, written by the plan kernel into the caller's workspace, or null
    int64_t piece_length;  // row-sparse mode without a map: group e reduces over [e, e + 1) * piece_length instead of
                           // everything (0: everything)
    int planned;           // `tile_table` (and `partials`) have been set up by mfma_gemm_plan
    int chunk_tiles;       // consecutive tiles that go to one XCD (set by the launchers of the fp32, few-row and few-tile kernels)
};

#define FM_LDS(T) __attribute__((address_space(3))) T

constexpr int kBufferResourceFlags = 0x00020000;  // raw buffer, 32-bit data format, no swizzle

// The same value, but the compiler cannot tell: what is computed from it is computed where it is written, not hoisted
// out of an enclosing loop into registers that stay occupied across the loop.
__device__ __forceinline__ int opaque(int value) {
    asm volatile("" : "+v"(value));
    return value;
}

// Tell the compiler that a pointer computed from tile coordinates is the same in every lane (it then lives in
// scalar registers and the loads use the scalar-base addressing form).
__device__ __forceinline__ const char *uniform_pointer(const char *pointer) {
    const uint64_t bits = reinterpret_cast<uint64_t>(pointer);
    const uint32_t low = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(bits));
    const uint32_t high = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(bits >> 32));
    return reinterpret_cast<const char *>((static_cast<uint64_t>(high) << 32) | low);
}

// ---- where reductions start ------------------------------------------------------------------------------
// Which slice of the reduction axis the tiles of an expert start with, where both operands are K-contiguous and the axis is whole
// slices of kRotationSlice. The CUs take slices at about the same pace, and 128 bytes of rows that are a few KiB apart lie in few of the memory's
// channels: with every expert's weights read from slice 0 on, all CUs ask the same channels at the same time. Experts that run at
// the same time are spread evenly over the axis instead (the fractional parts of multiples of the golden ratio). Per tile it would
// be worse: the tiles of an expert share its activations in L2. Row-contiguous weights, 512 bytes of every row at a time, are no
// faster for it, and neither is a launch that is bound by its MFMAs (kFewRows). Layer 1 (and layer 2's input gradient), us: 44 rows for each of
// 128 experts of 2048 x 768 218 -> 168 (125 -> 111), 94 for each of 64 of 2048 x 1408 200 -> 158 (106 -> 99), 125 of the 128 228 -> 218 and
// 218 -> 186 (120 -> 119), 469 of the 64 361 -> 348 (210 -> 210); 1024 of the 128 783 -> 789 (409 -> 409) without the bound.
// Where a tile starts and how far its operands reach is counted in 32 bits (fm_gemm_mfma.hip): axes are below kMaxRotatedAxis, as all
// are whose rows do not overlap (their strides are).
constexpr int kRotationSlice = 64, kFewRows = 1024;
constexpr int64_t kMaxRotatedAxis = int64_t(1) << 21;

__host__ __device__ inline bool starts_anywhere(const GemmArgs &args) {
    return args.mode != kInputRowSparse && args.num_experts > 1 && args.rows <= static_cast<int64_t>(kFewRows) * args.num_experts &&
           args.lhs_stride_inner == 1 && args.rhs_stride_inner == 1 && args.inner % kRotationSlice == 0 &&
           args.inner < kMaxRotatedAxis;
}

__device__ __forceinline__ int first_slice_of(const GemmArgs &args, int expert) {
    if (!starts_anywhere(args)) return 0;
    const uint32_t fraction = (static_cast<uint32_t>(expert) * 40503u) & 0xffffu;  // 40503 / 65536 = 0.618...
    return static_cast<int>((fraction * static_cast<uint64_t>(args.inner / kRotationSlice)) >> 16);
}

// ---- which tile ----------------------------------------------------------------------------------------
constexpr int kGroupRows = 8;

// The rows of an expert end where its padding begins, if the caller says where that is.
__device__ __forceinline__ void rows_of_expert(const GemmArgs &args, int expert, int64_t &begin, int64_t &end) {
    const void *ends = args.expert_pad_begins != nullptr ? args.expert_pad_begins : args.expert_ends;
    end = min(load_index(ends, args.index_dtype, expert), args.rows);
    begin = expert > 0 ? load_index(args.expert_ends, args.index_dtype, expert - 1) : 0;
}

// Logical order of the tiles of a product whose rows are grouped by expert (output-sparse, input-inner-sparse,
// dense): expert after expert; within an expert its row tiles (ceil(rows_e / kTile)) are cut into ceil(count / 8)
// groups of nearly equal size (9 row tiles: 5 + 4), and a group is walked column tile by column tile, row tiles
// fastest. 32 consecutive tiles (what an XCD runs at one time) are then about 8 row tiles x 4 column tiles of ONE
// expert, i.e. 8 lhs panels and 4 rhs panels shared in that XCD's L2; with groups that ignore the expert boundaries
// most chunks straddled two experts and needed twice the rhs panels.
// Every wavefront scans `expert_ends` 64 experts at a time; returns false if `logical` is past the last tile.
struct RowTile {
    int expert, tile_n, rows_valid;
    int64_t row0;
};

__device__ __forceinline__ void place_in_expert(int local, int count, int tiles_n, int &row_tile, int &tile_n) {
    const int groups = (count + kGroupRows - 1) / kGroupRows;
    const int base = count / groups, larger = count % groups;  // the first `larger` groups have base + 1 row tiles
    const int larger_tiles = larger * (base + 1) * tiles_n;
    int first_row, rows, in_group;
    if (local < larger_tiles) {
        const int group = local / ((base + 1) * tiles_n);
        rows = base + 1;
        first_row = group * rows;
        in_group = local - group * rows * tiles_n;
    } else {
        const int rest = local - larger_tiles;
        const int group = rest / (base * tiles_n);
        rows = base;
        first_row = larger * (base + 1) + group * rows;
        in_group = rest - group * rows * tiles_n;
    }
    row_tile = first_row + in_group % rows;
    tile_n = in_group / rows;
}

template <int kTile>
__device__ __forceinline__ bool locate_tile(const GemmArgs &args, int logical, RowTile &tile) {
    const int tiles_n = args.tiles_n;
    if (args.expert_ends == nullptr) {
        const int count = static_cast<int>((args.rows + kTile - 1) / kTile);
        if (logical >= count * tiles_n) return false;
        int row_tile;
        place_in_expert(logical, count, tiles_n, row_tile, tile.tile_n);
        tile.expert = 0;
        tile.row0 = static_cast<int64_t>(row_tile) * kTile;
        tile.rows_valid = static_cast<int>(min(static_cast<int64_t>(kTile), args.rows - tile.row0));
        return true;
    }
    const int lane = opaque(static_cast<int>(threadIdx.x & 63));
    int tiles_before = 0;  // row tiles of the experts before this block of 64
    for (int base = 0; base < args.num_experts; base += 64) {
        const int e = base + lane;
        int64_t begin = 0, end = 0;
        if (e < args.num_experts) rows_of_expert(args, e, begin, end);
        const int count = end > begin ? static_cast<int>((end - begin + kTile - 1) / kTile) : 0;
        int inclusive = count;
#pragma unroll
        for (int offset = 1; offset < 64; offset <<= 1) {
            const int other = __shfl_up(inclusive, offset, 64);
            if (lane >= offset) inclusive += other;
        }
        const int total = __shfl(inclusive, 63, 64);
        if (logical < (tiles_before + total) * tiles_n) {
            const uint64_t owners = __ballot((tiles_before + inclusive) * tiles_n > logical);
            const int owner = __ffsll(static_cast<unsigned long long>(owners)) - 1;
            const int owner_count = __shfl(count, owner, 64);
            const int first_tile = tiles_before + __shfl(inclusive - count, owner, 64);
            const int64_t owner_begin = __shfl(begin, owner, 64), owner_end = __shfl(end, owner, 64);
            int row_tile;
            place_in_expert(logical - first_tile * tiles_n, owner_count, tiles_n, row_tile, tile.tile_n);
            tile.expert = base + owner;
            tile.row0 = owner_begin + static_cast<int64_t>(row_tile) * kTile;
            tile.rows_valid = static_cast<int>(min(static_cast<int64_t>(kTile), owner_end - tile.row0));
            return true;
        }
        tiles_before += total;
    }
    return false;
}

// Logical tile -> (row tile, column tile) for the row-sparse product, whose row tiles are expert-aligned by
// construction: groups of 8 row tiles, column by column inside a group.
__device__ __forceinline__ void tile_coordinates(int logical, int tiles_m, int tiles_n, int &tile_m, int &tile_n) {
    const int width = kGroupRows * tiles_n;
    const int group = logical / width;
    const int first_m = group * kGroupRows;
    const int group_rows = min(tiles_m - first_m, kGroupRows);
    const int in_group = logical - group * width;
    tile_m = first_m + in_group % group_rows;
    tile_n = in_group / group_rows;
}

template <typename OutT>
__device__ __forceinline__ void store_out(void *out, int64_t offset, float value, bool accumulate) {
    OutT *pointer = static_cast<OutT *>(out) + offset;
    if (accumulate) value += to_float(*pointer);
    *pointer = from_float<OutT>(value);
}

__device__ __forceinline__ void store_out_dyn(void *out, int out_dtype, int64_t offset, float value, bool accumulate) {
    if (out_dtype == FM_DTYPE_F32) store_out<float>(out, offset, value, accumulate);
    else if (out_dtype == FM_DTYPE_BF16) store_out<bf16_t>(out, offset, value, accumulate);
    else store_out<f16_t>(out, offset, value, accumulate);
}

// Fast path (fm_gemm_mfma.hip). `eligible` says whether the MFMA kernel can take the problem as described by
// `args` (with `dtype` operands); `launch` fills in the tile counts and launches it.
bool mfma_gemm_eligible(const GemmArgs &args, int dtype);
bool mfma_gemm_fusion_eligible(const GemmArgs &args, int dtype);  // with args.fusion set
// `workspace` (may be null: no split) must hold mfma_gemm_workspace_size(args) bytes when that is not 0.
size_t mfma_gemm_workspace_size(GemmArgs args);
int mfma_gemm_launch(GemmArgs args, int dtype, void *workspace, size_t workspace_size, hipStream_t stream);

// The kernel that such a product runs on, and whether it would cut reductions into pieces, given a workspace.
enum GemmKernel { kLargeTiles = 0, kRowPanel = 1, kRowSparse = 2, kWeightStream = 3, kFewTiles = 4 };
GemmKernel mfma_gemm_kernel(GemmArgs args, int dtype, bool &splits);

// Tile tables of several products that follow one another on `stream`, in one launch: sets `planned`, `tile_table` and `partials`
// of those that want them (they share the space for pieces). `workspace`: mfma_gemm_plan_size(...) bytes, 64-byte aligned, kept
// until the last of them has run. A product with a table has to run as `run_gemm` (or the fused product) would have run it.
constexpr int kMaxPlanned = 5;
size_t mfma_gemm_plan_size(const GemmArgs *products, int count, int dtype);
int mfma_gemm_plan(GemmArgs *products, int count, int dtype, void *workspace, size_t workspace_size, hipStream_t stream);

// What the entry points of fm_gemm.hip check, dispatch and launch.
int run_gemm(const char *name, GemmArgs args, int dtype, void *workspace, size_t workspace_size, void *stream);
int run_fused_gemm(const char *name, GemmArgs args, int dtype, void *stream);

// Allows `kernel` that many bytes of dynamic LDS. `configured`: the kernel's own bit mask of devices done.
int allow_lds(const void *kernel, int bytes, std::atomic<uint64_t> &configured);

// Row-sparse products of experts of few rows (fm_gemm_row_panel.hip), of those that `mfma_gemm_eligible` accepts.
bool row_panel_gemm_chosen(const GemmArgs &args, int dtype);
int row_panel_gemm_launch(const GemmArgs &args, int dtype, hipStream_t stream);
// Row-sparse products of experts of some more rows (fm_gemm_row_sparse.hip), of those that `mfma_gemm_eligible` accepts.
bool row_sparse_gemm_chosen(const GemmArgs &args, int dtype);
int row_sparse_gemm_launch(GemmArgs args, int dtype, hipStream_t stream);
// Products that memory bounds, or of few tiles (fm_gemm_weight_stream.hip). `splits`: the large tiles' kernel would split the reductions,
// given a workspace.
bool weight_stream_gemm_chosen(const GemmArgs &args, int dtype, bool splits);
int weight_stream_gemm_launch(const GemmArgs &args, int dtype, hipStream_t stream);
// Those of fewer tiles still (fm_gemm_few_tiles.hip), of the ones that the above refuses.
bool few_tiles_gemm_chosen(const GemmArgs &args, int dtype, bool splits);
int few_tiles_gemm_launch(const GemmArgs &args, int dtype, hipStream_t stream);

// fp32 operands with a unit stride and 16-byte aligned lines (fm_gemm_f32.hip).
bool f32_gemm_eligible(const GemmArgs &args, int dtype);
int f32_gemm_launch(GemmArgs args, hipStream_t stream);

}  // namespace fm
