// Operand slices of the half-precision products that keep 64 along K at a time in LDS: where they lie there, the loads that fill them
// and the MFMA fragments that are read from them.
#pragma once

#include "fm_gemm_common.h"

namespace fm {

namespace slices {

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8_t;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float f32x16_t;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4_t;
typedef __attribute__((__vector_size__(2 * sizeof(uint32_t)))) uint32_t u32x2_t;
typedef __attribute__((__vector_size__(4 * sizeof(short)))) short i16x4_t;

constexpr int kBK = kRotationSlice, kSteps = kBK / 16, kLoadingThreads = 256;  // four wavefronts fill a slice

__device__ __forceinline__ f32x16_t mfma(bf16_t, u32x4_t a, u32x4_t b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
__device__ __forceinline__ f32x16_t mfma(f16_t, u32x4_t a, u32x4_t b, f32x16_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
}

// One operand's slice in LDS and the loads that fill it: lines [row][kBK] where it is contiguous along K, [kBK][row] otherwise.
template <int kTile, bool kContiguousK, int kBlocks>
struct Operand {
    static constexpr int kBytes = kTile * kBK * 2, kChunks = (kContiguousK ? kBK : kTile) / 8;  // 16-byte chunks per line
    static constexpr int kLoads = kBytes / 16 / kLoadingThreads;                              // per lane and slice
    static constexpr uint32_t kOutOfRange = 0x80000000u, kRange = 0x7fffffffu;

    // Where chunk `c` of line `line` sits among the line's chunks: the lines that a fragment takes one column of chunks from lie in
    // different banks.
    static __device__ __forceinline__ int swizzled(int line, int c) {
        if constexpr (kContiguousK) return c ^ ((line / (16 / kChunks)) & (kChunks - 1));
        else return c ^ (((line & 3) << 2) & (kChunks - 1));
    }

    const char *start, *base;  // wave-uniform: the tile's first element; that of the next slice to fetch
    int64_t step;              // bytes from one slice to the next
    uint32_t offset[kLoads];   // per lane, bytes from `base`; out of range where the tile has no such line or column
    int k[kLoads];             // of the load's first element in the slice
    int k_count, k_left;       // of the reduction; from `base` on
    int slices, next, unfetched;

    // `stride`: bytes between lines. `valid`: rows (columns of the product) that exist, a multiple of 8 where they are not lines.
    // `kPaired`: of every 64 lines the first 32 follow one another in memory and the last 32 lie `pair_distance` lines after those;
    // `valid` of each.
    template <bool kPaired>
    __device__ __forceinline__ void setup(const char *first, int64_t stride, int valid, int k_count_, int first_slice, int wave, int lane,
                                          int64_t pair_distance) {
        static_assert(kContiguousK || !kPaired, "lines are rows");
        start = uniform_pointer(first);
        step = kContiguousK ? kBK * 2 : kBK * stride;
        k_count = k_count_;
        slices = unfetched = (k_count + kBK - 1) / kBK;
        next = first_slice;
        base = start + first_slice * step;
        k_left = k_count - first_slice * kBK;
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const int slot = (wave * kLoads + j) * 64 + lane, line = slot / kChunks, chunk = swizzled(line, slot % kChunks);
            const int single = kPaired ? line / 64 * 32 + line % 32 : line;
            const bool exists = kContiguousK ? single < valid : chunk * 8 < valid;
            const int64_t memory_line = kPaired && line % 64 >= 32 ? single + pair_distance : single;
            offset[j] = exists ? static_cast<uint32_t>(memory_line * stride + chunk * 16) : kOutOfRange;
            k[j] = kContiguousK ? chunk * 8 : line;
        }
    }

    // The next slice -> the slot at LDS address `slot`: the last slice is followed by the first one, and when all have been fetched
    // zeros come, without an access to memory. What lies past the reduction comes as zeros too.
    __device__ __forceinline__ void fetch(int slot, int wave) {
        const __amdgpu_buffer_rsrc_t resource = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<char *>(uniform_pointer(base)), 0, static_cast<int>(kRange), kBufferResourceFlags);
#pragma unroll
        for (int j = 0; j < kLoads; ++j) {
            const uint32_t lane_offset = k[j] < k_left ? offset[j] : kOutOfRange;
            const int target = __builtin_amdgcn_readfirstlane(slot + (wave * kLoads + j) * 1024);
            // M0 is not handed out by the register allocator and nothing else in this file uses it.
            asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, 0 offen lds"
                         :
                         : "s"(target), "v"(lane_offset), "s"(resource)
                         : "memory");
        }
        base += step;
        ++next;
        --unfetched;
        if (next == slices) {
            next = 0;
            base = start;
        }
        k_left = unfetched > 0 ? k_count - next * kBK : 0;
    }

    // MFMA fragments (8 consecutive k of one row per lane; lane l: row l % 32, k half l / 32) of the 32 rows from `first` on, per lane:
    // an address per step of 16 (K-contiguous; the next 32 rows and the slot are added), or one per 32 rows (the step is added).
    static constexpr int kAddresses = kContiguousK ? kSteps : kBlocks;
    static __device__ __forceinline__ void fragment_addresses(int first, int lane, int (&addresses)[kAddresses]) {
        if constexpr (kContiguousK) {
            const int row = first + (lane & 31);
#pragma unroll
            for (int s = 0; s < kSteps; ++s) addresses[s] = (row * kChunks + swizzled(row, 2 * s + (lane >> 5))) * 16;
        } else {
            const int s = lane & 15, group = lane >> 4, k = ((group >> 1) << 3) + (s >> 2);
#pragma unroll
            for (int i = 0; i < kBlocks; ++i) {
                const int column = first + i * 32 + ((group & 1) << 4) + ((s & 3) << 2);
                addresses[i] = k * kTile * 2 + swizzled(k, column >> 3) * 16 + (column & 7) * 2;
            }
        }
    }
    static __device__ __forceinline__ u32x4_t fragment(const int (&addresses)[kAddresses], int slot, int i, int step) {
        if constexpr (kContiguousK) {
            return *(FM_LDS(u32x4_t) *)static_cast<uintptr_t>(addresses[step] + slot + i * 32 * kChunks * 16);
        } else {
            const uintptr_t at = static_cast<uintptr_t>(addresses[i] + slot + step * 16 * kTile * 2);
            const i16x4_t low = __builtin_amdgcn_ds_read_tr16_b64_v4i16((FM_LDS(i16x4_t) *)at);
            const i16x4_t high = __builtin_amdgcn_ds_read_tr16_b64_v4i16((FM_LDS(i16x4_t) *)(at + 4 * kTile * 2));
            const u32x2_t low_words = __builtin_bit_cast(u32x2_t, low), high_words = __builtin_bit_cast(u32x2_t, high);
            return u32x4_t{low_words[0], low_words[1], high_words[0], high_words[1]};
        }
    }
};

// Returns once at most `kNewest` of the loads this wavefront has issued are still on their way, and all that it has asked LDS for is
// there: after a barrier the others' loads may replace what it read.
template <int kNewest>
__device__ __forceinline__ void wait_for_loads() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(kNewest) : "memory");
}

}  // namespace slices

}  // namespace fm
