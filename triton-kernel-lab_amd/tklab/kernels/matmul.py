"""GEMM on CDNA4 MFMA through ``tk_gemm``: ``matmul_fp32acc`` and ``matmul_fp16acc``.

Contract of ``src/tklab/kernels/matmul.py``: two 2-D matrices with matching
inner dimension, same device and dtype, strictly positive strides within the
int32 range, float16 (and here also bfloat16) inputs, a contiguous output of
the input dtype. Validation order and messages follow ``matmul.py:167-186``.

The reference autotunes 25 Triton configurations per shape
(``matmul.py:23-75``); this build picks a kernel from the operands' layout and
reports it in the same metadata keys. Operands whose rows are 16-byte aligned and
multiples of 8 elements long, each row-major or transposed, take buffer->LDS DMA
kernels (tiles from 64 x 64 to 256 x 256 by problem size, eight wave64s,
``v_mfma_f32_16x16x32``): ``gemm_dma_kernel`` for row-major operands with K % 32 == 0 (every registry shape),
``gemm_kernel`` for transposed ones (a linear layer's gradients) and other K, and
``gemm_split_kernel`` where few tiles meet a long K (:func:`split_k`).
Every other layout takes the register-staged ``gemm_kernel`` (64 x 64 to 256 x 128).
``matmul_fp16acc`` keeps its registry entry, but gfx950 MFMA
accumulates f16 products in float32 only, so both entry points run the same
FP32-accumulate kernel (its result is at least as accurate as an FP16
accumulation and meets the looser 5e-2 bound the reference sets for it).
"""

from __future__ import annotations

import torch

from tklab import _hip
from tklab.harness.addressing import assert_int32_addressable
from tklab.harness.tolerances import assert_relative_frobenius
from tklab.registry import (
    BenchmarkMetadataFn,
    BenchmarkScalar,
    KernelSpec,
    LaunchFn,
    TensorArgs,
    register,
)

_DTYPES = (torch.float16, torch.bfloat16)

# csrc/gemm_dma.hip (BM, BN, BK, kGroupM, kThreads / 64 waves, kBStages): row-major operands
# with K % 32 == 0. "num_warps" counts wave64s; "num_stages" is the ring of 32-wide K steps
# (the B operand's; A is loaded in 64-wide tiles into a ring of kAStages = 3).
TILE = {"hip_kernel": "gemm_dma_kernel", "block_m": 256, "block_n": 256, "block_k": 32, "group_m": 4,
        "num_warps": 8, "num_stages": 4}
# tk_gemm_tile's kernels. The 256 x 256 one of gemm_dma.hip is TILE; the smaller DMA tiles
# (csrc/gemm_tile.hpp) step K by 64 with the stages that fit a CU's LDS (half of it for the smallest
# tiles, two workgroups per CU), the register-staged ones (csrc/gemm.hip) with two stages.
_KERNELS = {1: "gemm_dma_kernel", 2: "gemm_kernel", 3: "gemm_kernel"}
_STAGED = 3
_MFMA = {
    torch.float16: "v_mfma_f32_16x16x32_f16",
    torch.bfloat16: "v_mfma_f32_16x16x32_bf16",
}


def _dma_rows(rows: int, cols: int, row_stride: int, col_stride: int) -> bool:
    """Rows the DMA kernels can load: unit inner stride, whole aligned 16-byte groups, < 2 GiB."""
    return (
        col_stride == 1
        and not (cols | row_stride) & 7
        and ((rows - 1) * row_stride + cols) * 2 < 2**31
    )


def _dma_operand(rows: int, cols: int, row_stride: int, col_stride: int) -> bool:
    """Layouts the DMA kernels take: stored by rows or by columns (``plan``, csrc/gemm_dma.hip).

    The base must be 16-byte aligned too.
    """
    return _dma_rows(rows, cols, row_stride, col_stride) or _dma_rows(cols, rows, col_stride, row_stride)


def split_k(m: int, n: int, k: int) -> int:
    """Runs of K for ``tk_gemm_splitk``; 1: one workgroup per output tile walks all of K.

    A workgroup takes 0.2 to 0.4 us per 64-wide K tile of a 64 x 64 tile (10 KiB with 16 rows of A,
    16 KiB with 64); the second kernel and the float32 sums take ~4 us of the device and ~5 of the
    host. One round of the 256 CUs and runs of at least 16 K tiles were the best or within 8 % of
    it: 64x4096x14336 (64 tiles) 84.6 us unsplit, 4 runs 31.9, 6 40.1, 8 35.3; 16x512x8192 (8 tiles) 27.4, 8 runs 10.6, 16 12.0. Past
    128 tiles nothing is left to fill (256x4096x8192: 46.7, 2 runs 49.4). Below the least depth
    a call is shorter than its host time: with the norm of a QKV projection 1x4096x4096 19.3
    unsplit, 23.9 split, the product 8x512x3072 11.6 and 14.0; from 96 tiles HBM traffic moves
    the line: 16x6144x4096 25.6 and 23.9, SwiGLU 8x8192x4096 38.6 and 33.0. Sums: at most 4 MiB
    (8 MiB with SwiGLU).

    The sizes decide, so that every layout the DMA kernels take and the fused variants add in the
    same order. Two things follow for the bits of a result (its error does not grow). A row's bits
    depend on M where K is split: 64x4096x14336 is summed in 4 runs, the same rows among 1024 in
    one. And operands the DMA kernels do not take (odd strides, unaligned bases) are never split,
    so they have the bits of the unsplit product. ``tk_gemm`` and the registry's launchers never
    split: every tile and layout sums a row alike whatever M is.
    """
    tiles = -(-m // 64) * -(-n // 64)
    depth = -(-k // 64)
    if tiles > 128 or depth < (64 if tiles >= 96 else 80):
        return 1
    return min(256 // tiles, depth // 16)


def enqueue_split(
    a: torch.Tensor, b: torch.Tensor, out: torch.Tensor, splits: int, *, up: torch.Tensor | None = None,
    row_scale: torch.Tensor | None = None,
) -> None:
    """``tk_gemm_splitk`` on checked operands: ``a @ b``, row-scaled, or SwiGLU with gate ``b``."""
    (m, k), n = a.shape, b.shape[1]
    # Float32 sums of the runs, on the stream the kernels run on.
    sums = torch.empty(splits * m * n * (1 if up is None else 2), device=a.device, dtype=torch.float32)
    _hip.call(
        "tk_gemm_splitk", _hip.dtype_code(a.dtype), a.data_ptr(), b.data_ptr(),
        None if up is None else up.data_ptr(), None if row_scale is None else row_scale.data_ptr(),
        out.data_ptr(), sums.data_ptr(), m, n, k, splits, *a.stride(), *b.stride(),
        *(b if up is None else up).stride(), *out.stride(), _hip.stream_of(a),
    )


def _tile_config(rows: int, cols: int, *, kernel: int = 1) -> dict[str, BenchmarkScalar]:
    """Metadata of a tile of one of :data:`_KERNELS`."""
    config = {**TILE, "hip_kernel": _KERNELS[kernel], "block_m": rows, "block_n": cols}
    if (rows, cols) == (256, 256):
        return config
    stage = (rows + cols) * 128
    stages = 81920 // stage if rows + cols <= 192 else min(5, 163840 // stage)
    return {**config, "block_k": 64, "group_m": 8 if cols > rows else 4,
            "num_stages": 2 if kernel == _STAGED else stages}


def _query_tile(
    a_ptr: int, b_ptr: int, m: int, n: int, k: int, a_strides: tuple[int, ...], b_strides: tuple[int, ...]
) -> tuple[int, int, int]:
    """(kernel, rows, columns) of ``tk_gemm_tile``."""
    tile = _hip.query("tk_gemm_tile", a_ptr, b_ptr, m, n, k, *a_strides, *b_strides)
    return tile >> 20, tile >> 10 & 1023, tile & 1023


def launch_config(a: torch.Tensor, b: torch.Tensor) -> dict[str, BenchmarkScalar]:
    """Tile configuration and MFMA of the kernel ``matmul_fp32acc`` launches for ``a @ b``."""
    (m, k), n = a.shape, b.shape[1]
    mma = {"mma_opcode": _MFMA.get(a.dtype, _MFMA[torch.float16])}
    kernel, rows, cols = _query_tile(a.data_ptr(), b.data_ptr(), m, n, k, a.stride(), b.stride())
    if kernel != _STAGED and split_k(m, n, k) > 1:
        return {**_tile_config(64, 64), **mma, "hip_kernel": "gemm_split_kernel"}
    return {**_tile_config(rows, cols, kernel=kernel), **mma}


def _validate(a: torch.Tensor, b: torch.Tensor) -> None:
    """GEMM input contract (reference ``matmul.py:167-186``)."""
    if a.ndim != 2 or b.ndim != 2:
        raise ValueError("matmul expects two 2D tensors")
    if a.shape[1] != b.shape[0]:
        raise ValueError(f"incompatible shapes: {a.shape} and {b.shape}")
    if 0 in (*a.shape, *b.shape):
        raise ValueError("matmul does not support empty dimensions")
    if a.device != b.device:
        raise ValueError(f"device mismatch: {a.device} != {b.device}")
    if a.dtype != b.dtype:
        raise ValueError(f"dtype mismatch: {a.dtype} != {b.dtype}")
    if a.dtype not in _DTYPES:
        raise ValueError("matmul supports float16 and bfloat16 inputs only")
    for name, tensor in (("left", a), ("right", b)):
        if any(stride <= 0 for stride in tensor.stride()):
            raise ValueError(f"{name} input requires strictly positive strides")
        assert_int32_addressable(tensor, name=name)
    if a.device.type != "cuda":
        raise ValueError("matmul requires CUDA (ROCm/HIP) tensors")


def _make_output(args: TensorArgs) -> torch.Tensor:
    """Contiguous output of the input dtype."""
    a, b = args
    return torch.empty((a.shape[0], b.shape[1]), device=a.device, dtype=a.dtype)


def _launch_factory(*, fp16_accumulate: bool) -> LaunchFn:
    """Allocation-free launcher for one accumulation mode (K is never split)."""

    def launch(args: TensorArgs, output: torch.Tensor) -> None:
        a, b = args
        _validate(a, b)
        if output.shape != (a.shape[0], b.shape[1]):
            raise ValueError("output shape does not match matmul result")
        if output.device != a.device or output.dtype != a.dtype:
            raise ValueError("output metadata must match the inputs")
        if not output.is_contiguous():
            raise ValueError("matmul output must be contiguous")
        _enqueue(a, b, output, fp16_accumulate=fp16_accumulate, whole=True)

    return launch


def _enqueue(
    a: torch.Tensor, b: torch.Tensor, output: torch.Tensor, *, fp16_accumulate: bool, whole: bool = False
) -> None:
    """``output = a @ b`` for operands and an output already checked; ``whole``: never split K."""
    (m, k), n = a.shape, b.shape[1]
    a_strides, b_strides, a_ptr, b_ptr = a.stride(), b.stride(), a.data_ptr(), b.data_ptr()
    splits = 1 if whole else split_k(m, n, k)
    if (splits > 1 and not (a_ptr | b_ptr) & 15 and _dma_operand(m, k, *a_strides)
            and _dma_operand(k, n, *b_strides)):
        sums = torch.empty(splits * m * n, device=a.device, dtype=torch.float32)
        _hip.call(
            "tk_gemm_splitk", _hip.dtype_code(a.dtype), a_ptr, b_ptr, None, None, output.data_ptr(),
            sums.data_ptr(), m, n, k, splits, *a_strides, *b_strides, *b_strides, *output.stride(),
            _hip.stream_of(a),
        )
        return
    _hip.call(
        "tk_gemm", _hip.dtype_code(a.dtype), a_ptr, b_ptr, output.data_ptr(), m, n, k, *a_strides,
        *b_strides, *output.stride(), int(fp16_accumulate), _hip.stream_of(a),
    )


_launch_fp32acc = _launch_factory(fp16_accumulate=False)
_launch_fp16acc = _launch_factory(fp16_accumulate=True)


def matmul_fp32acc(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """``a @ b`` with float32 MFMA accumulation, summed over K in the order :func:`split_k` states."""
    _validate(a, b)
    output = _make_output((a, b))
    _enqueue(a, b, output, fp16_accumulate=False)
    return output


def matmul_fp16acc(a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """Registry-compatible FP16-accumulate entry point (runs the FP32-accumulate kernel)."""
    _validate(a, b)
    output = _make_output((a, b))
    _enqueue(a, b, output, fp16_accumulate=True)
    return output


def _launch_reference(args: TensorArgs, output: torch.Tensor) -> None:
    """Allocation-free PyTorch GEMM (hipBLASLt)."""
    a, b = args
    torch.mm(a, b, out=output)


def _make_inputs(size: int, device: torch.device, dtype: torch.dtype) -> TensorArgs:
    """Square standard-normal matrices."""
    return (
        torch.randn(size, size, device=device, dtype=dtype),
        torch.randn(size, size, device=device, dtype=dtype),
    )


def _make_adversarial(device: torch.device) -> TensorArgs:
    """Strided 129 x 193 @ 193 x 257: M, N and K tails at once."""
    left = torch.randn(129, 386, device=device, dtype=torch.float16)
    right = torch.randn(386, 257, device=device, dtype=torch.float16)
    return left[:, ::2], right[::2, :]


def _assert_fp32acc(output: torch.Tensor, reference: torch.Tensor) -> None:
    """Relative Frobenius error below 1e-2 (reference ``matmul.py:282-284``)."""
    assert_relative_frobenius(output, reference, max_relative_error=1e-2)


def _assert_fp16acc(output: torch.Tensor, reference: torch.Tensor) -> None:
    """Relative Frobenius error below 5e-2 (reference ``matmul.py:287-289``)."""
    assert_relative_frobenius(output, reference, max_relative_error=5e-2)


def _metadata_factory() -> BenchmarkMetadataFn:
    """Tile configuration in the reference's metadata keys (``matmul.py:292-312``)."""

    def metadata(size: int, dtype: torch.dtype) -> dict[str, BenchmarkScalar]:
        # Registry inputs are contiguous, aligned size x size matrices; the launcher never splits K.
        kernel, rows, cols = _query_tile(0, 0, size, size, size, (size, 1), (size, 1))
        return {**_tile_config(rows, cols, kernel=kernel), "mma_opcode": _MFMA.get(dtype, _MFMA[torch.float16])}

    return metadata


_SIZES = (512, 1024, 2048, 4096, 8192)


def _flops(size: int, _dtype: torch.dtype) -> int:
    """``2 * M * N * K`` for a square problem."""
    return 2 * size**3


MATMUL_FP32ACC = register(
    KernelSpec(
        name="matmul_fp32acc",
        description="FP16/BF16 GEMM with FP32 MFMA accumulation.",
        triton_fn=matmul_fp32acc,
        launch_fn=_launch_fp32acc,
        ref_fn=torch.matmul,
        reference_launch_fn=_launch_reference,
        make_inputs=_make_inputs,
        make_output=_make_output,
        make_adversarial=_make_adversarial,
        sizes=_SIZES,
        correctness_sizes=(512, 1024),
        bound="compute",
        flops=_flops,
        dtypes=(torch.float16, torch.bfloat16),
        assert_fn=_assert_fp32acc,
        benchmark_metadata=_metadata_factory(),
        compute_mode="fp16_fp32acc",
        supports_interpreter=False,
    )
)

MATMUL_FP16ACC = register(
    KernelSpec(
        name="matmul_fp16acc",
        description="FP16 GEMM registry entry; MFMA accumulates in FP32 on gfx950.",
        triton_fn=matmul_fp16acc,
        launch_fn=_launch_fp16acc,
        ref_fn=torch.matmul,
        reference_launch_fn=_launch_reference,
        make_inputs=_make_inputs,
        make_output=_make_output,
        make_adversarial=_make_adversarial,
        sizes=_SIZES,
        correctness_sizes=(512, 1024),
        bound="compute",
        flops=_flops,
        dtypes=(torch.float16,),
        assert_fn=_assert_fp16acc,
        benchmark_metadata=_metadata_factory(),
        compute_mode="fp16_fp16acc",
        supports_interpreter=False,
    )
)
