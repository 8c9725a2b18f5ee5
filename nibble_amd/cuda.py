"""Python wrappers of the torch ops ``w4a16::linear``, ``w4a16::dequantize`` and
``w4a16::quantize``.

Mirrors reference ``w4a16/cuda.py``: importing the compiled extension
(``nibble_amd._C``, here a thin libtorch shim over the HIP C ABI) registers
the ops; a missing extension is recorded, ``cuda_extension_available()``
reports it and the wrappers raise ``RuntimeError``. There is no fallback:
GPU tensors only ever run the HIP kernels. On PyTorch-ROCm "cuda" tensors
are HIP tensors, so the reference's names are kept.
"""

from __future__ import annotations

import importlib

import torch

try:
    importlib.import_module("nibble_amd._C")
except (ImportError, OSError) as error:
    _EXTENSION_LOAD_ERROR: Exception | None = error
else:
    _EXTENSION_LOAD_ERROR = None


if _EXTENSION_LOAD_ERROR is None:
    # Shape/dtype-only implementations so torch.compile can trace through the
    # ops with fake tensors (reference w4a16/cuda.py:14-36).
    @torch.library.register_fake("w4a16::linear")
    def _linear_fake(activations, packed_weights, scales, group_size):
        return activations.new_empty((activations.shape[0], packed_weights.shape[0]))

    @torch.library.register_fake("w4a16::dequantize")
    def _dequantize_fake(packed_weights, scales, group_size):
        return packed_weights.new_empty(
            (packed_weights.shape[0], packed_weights.shape[1] * 2), dtype=torch.float16
        )

    @torch.library.register_fake("w4a16::quantize")
    def _quantize_fake(weights, group_size):
        rows, cols = weights.shape
        return (
            weights.new_empty((rows, cols // 2), dtype=torch.uint8),
            weights.new_empty((rows, cols // group_size), dtype=torch.float16),
        )


def cuda_extension_available() -> bool:
    """Whether the compiled W4A16 HIP extension is loaded."""
    return _EXTENSION_LOAD_ERROR is None


def extension_load_error() -> Exception | None:
    return _EXTENSION_LOAD_ERROR


def _require_extension() -> None:
    if _EXTENSION_LOAD_ERROR is not None:
        raise RuntimeError(
            "The W4A16 HIP extension is not built. Build it with "
            "`python -c 'import __graft_entry__ as g; g.build()'`."
        ) from _EXTENSION_LOAD_ERROR


_PLAIN = (torch.Tensor, torch.nn.Parameter)
_transformed = torch._C._functorch.is_functorch_wrapped_tensor
_dispatch_modes = torch._C._len_torch_dispatch_stack


def addressable(*tensors: torch.Tensor) -> bool:
    """Whether a choice may look at where these tensors' memory starts: ordinary
    tensors of a call that runs now. False for a traced call (its graph also
    serves other tensors), under a dispatch mode, for a wrapper of
    ``torch.func`` and for a subclass, which may have no memory of their own."""
    if torch.compiler.is_compiling() or torch.jit.is_tracing() or _dispatch_modes():
        return False
    for tensor in tensors:
        if type(tensor) not in _PLAIN or _transformed(tensor):
            return False
    return True


def linear_cuda(
    activations: torch.Tensor,
    packed_weights: torch.Tensor,
    scales: torch.Tensor,
    group_size: int = 128,
) -> torch.Tensor:
    """Fused W4A16 linear on the GPU (reference ``w4a16/cuda.py:52-69``).

    group_size 128 with 16-byte aligned operands runs the tuned gfx950 kernels
    (up to 16 rows) and the W4A16 GEMM (above); group sizes 32 and 64 at M <= 8
    with K a multiple of 128 run their matrix-core kernel; anything else runs
    the scalar HIP kernel.
    """
    _require_extension()
    # the overload itself: naming the packet looks it up on every call (about 1 us)
    return torch.ops.w4a16.linear.default(activations, packed_weights, scales, group_size)


def dequantize_cuda(
    packed_weights: torch.Tensor,
    scales: torch.Tensor,
    group_size: int = 128,
) -> torch.Tensor:
    """Packed INT4 -> fp16 [N, K] in one pass (reference ``w4a16/cuda.py:72-83``).

    Bit-identical to ``dequantize_weights(...).to(torch.float16)``; needs
    group_size a multiple of 32 and 16-byte aligned packed weights.
    """
    _require_extension()
    return torch.ops.w4a16.dequantize(packed_weights, scales, group_size)


def quantize_cuda(weights: torch.Tensor, group_size: int = 128) -> tuple[torch.Tensor, torch.Tensor]:
    """fp16 / fp32 weights [N, K] -> (packed uint8 [N, K / 2], fp16 scales) in
    one pass, the bytes of ``quantize_and_pack_weights``; group_size a power of
    two from 16 to 512, weights contiguous and 16-byte aligned."""
    _require_extension()
    return torch.ops.w4a16.quantize(weights, group_size)
