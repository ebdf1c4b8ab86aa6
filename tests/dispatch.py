"""Which kernel the library runs a product on, asked of its own rules without a GPU: tests that are about one kernel say so with this."""

import ctypes
import pathlib
import subprocess

CSRC = pathlib.Path(__file__).resolve().parent.parent / "fast_llm_amd" / "csrc"
KERNELS = ("large tiles", "row panel", "row sparse", "weight stream", "few tiles")
OUTPUT_SPARSE, INPUT_INNER_SPARSE, INPUT_ROW_SPARSE = range(3)

_PROGRAM = """
#include "fm_gemm_common.h"
using namespace fm;

// bf16 operands as the layer has them: contiguous activations and weights [experts * columns, inner] (output-sparse) or
// [experts * inner, columns]; the weight gradient of [rows, size] and [rows, columns]. The kernel, + 16 if it cuts reductions; -1: generic.
extern "C" int kernel_of(int mode, int64_t rows, int64_t columns, int64_t inner, int experts, int grouped, int accumulate, int out_dtype,
                         int gated) {
    static char operand[16] __attribute__((aligned(16)));
    const int64_t size = mode == kOutputSparse ? columns : inner;
    GemmArgs args{operand, operand, gated ? nullptr : operand, grouped ? operand : nullptr, grouped ? operand : nullptr};
    args.lhs_stride_row = mode == kInputRowSparse ? 1 : inner;
    args.lhs_stride_inner = mode == kInputRowSparse ? inner : 1;
    args.rhs_stride_inner = mode == kOutputSparse ? 1 : columns;
    args.rhs_stride_col = mode == kOutputSparse ? inner : 1;
    args.out_stride_row = columns, args.out_stride_col = 1;
    args.rows = mode == kInputRowSparse ? inner * experts : rows;
    args.cols = columns;
    args.inner = mode == kInputRowSparse ? rows : inner;
    args.sparse_size = size;
    args.num_experts = grouped ? experts : 1;
    args.mode = mode, args.accumulate = accumulate, args.index_dtype = FM_INDEX_I32, args.out_dtype = out_dtype;
    if (gated) {
        args.fusion = kFusionGatedForward, args.fused_out = operand, args.any_half = 1;
        args.half = args.fused_stride = columns / 2;
        if (!mfma_gemm_fusion_eligible(args, FM_DTYPE_BF16)) return -1;
    }
    if (!mfma_gemm_eligible(args, FM_DTYPE_BF16)) return -1;
    bool splits;
    const int kernel = mfma_gemm_kernel(args, FM_DTYPE_BF16, splits);
    return kernel + (splits ? 16 : 0);
}
"""


class Dispatch:
    """`library`: the built kernel library."""

    def __init__(self, folder: pathlib.Path, library: pathlib.Path):
        from fast_llm_amd.build import _hipcc

        source, probe = folder / "dispatch.hip", folder / "dispatch.so"
        source.write_text(_PROGRAM)
        subprocess.run(
            [_hipcc(), "--offload-host-only", "-std=c++17", "-fPIC", "-shared", f"-I{CSRC}", str(source), "-o", str(probe),
             f"-L{library.parent}", f"-l:{library.name}", f"-Wl,-rpath,{library.parent}"],
            check=True, capture_output=True,
        )  # fmt: skip
        self._kernel_of = ctypes.CDLL(str(probe)).kernel_of
        self._kernel_of.argtypes = [ctypes.c_int] + [ctypes.c_int64] * 3 + [ctypes.c_int] * 5

    def __call__(self, mode, rows, columns, inner, experts=None, accumulate=False, fp32_out=False, gated=False) -> str:
        """`rows` are those of the operands, padding included; `experts` None: a dense product; `inner` of a weight gradient: the rows
        of the gradient of one expert. With " in pieces" where the reductions are cut, given a workspace."""
        kernel = self._kernel_of(mode, rows, columns, inner, experts or 1, experts is not None, accumulate, 0 if fp32_out else 1, gated)
        assert kernel >= 0, "the generic kernel"
        return KERNELS[kernel % 16] + (" in pieces" if kernel >= 16 else "")
