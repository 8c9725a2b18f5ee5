"""``QuantizedLinear`` (alias ``Int4Linear``): an inference-only linear layer
that keeps packed INT4 weights and runs them through the HIP kernels.

Mirrors reference ``w4a16/linear.py`` (constructor checks, buffers
``packed_weights`` / ``scales`` / ``bias`` in the state dict, ``from_float``,
``empty``, ``forward`` routing). Routing of ``forward``:

* CPU tensors: the pure-PyTorch ``linear_reference``;
* GPU tensors, ``fused`` and M <= ``FUSED_MAX_ROWS``: ``w4a16::linear``
  (the gfx950 GEMV / small-batch kernels);
* GPU tensors, ``fused``, group_size 128 and M <= ``native_max_rows``
  (prompts; 512, 704 or 1024 rows by the layer's sizes, see
  ``gemm_max_rows``): ``w4a16::linear`` as well, which runs the W4A16 MFMA GEMM (at
  9..16 rows of long rows, its 16-row paired form) on weights decoded in
  registers, bit-identical to the dequantized fp16 weights, with fp32
  accumulation; the reference sends these rows to dequantize + cuBLAS, and
  the result agrees with that path within its own prefill tolerance
  (reference tests/test_linear.py:207-225, rtol = atol = 1e-3);
* GPU tensors otherwise (longer prompts, ``fused=False``):
  ``w4a16::dequantize`` then ``F.linear`` (hipBLASLt) when group_size is a
  multiple of 32, else ``w4a16::linear``'s generic kernel (any M, any even
  group size).

GPU tensors never take a torch or CPU fallback: without the extension they
raise ``RuntimeError``.
"""

from __future__ import annotations

import torch
import torch.nn.functional as F

from nibble_amd.cuda import addressable, dequantize_cuda, linear_cuda
from nibble_amd.quantization import quantize_and_pack_weights
from nibble_amd.reference import dequantize_weights, linear_reference

# Largest M routed to the fused kernels; larger M dequantizes and uses a GEMM.
FUSED_MAX_ROWS = 8
# Largest M routed to the W4A16 GEMM when fused (group size 128) on any layer:
# measured against dequantize + hipBLASLt on the 1.1B / 8B / 70B layers (K x N,
# us: M = 256, 4096 x 14336 43.7 against 74.2; M = 64, 5632 x 2048 11.6 against
# 26.7; M = 512, 4096 x 14336 72.7 against 84.2, 14336 x 4096 86.5 against
# 109.0, 8192 x 28672 275 against 281, and every other swept layer faster too).
# Wide layers lose from M = 1024 (4096 x 14336 141.8 against 117.7) and nearly
# every one at M = 2048 (2048 x 11264 118.0 against 97.2).
NATIVE_GEMM_MAX_ROWS = 512


def gemm_max_rows(n: int, k: int) -> int:
    """Rows up to which the W4A16 GEMM of a layer keeps up with dequantize + the
    dense GEMM: a sweep of 513..1024 rows over layers of up to 24M weights
    (graph timing, rotated weights), in which it loses no more than 1%
    anywhere below these lines. Its tiles fill whole rounds of the 256 CUs on
    small and narrow layers (K x N at 1024 rows, us: 5632 x 2048 35.2 against
    44.4, 14336 x 1024 55.3 against 60.8, 2048 x 4096 25.9 against 34.4).
    Others start a further round past 704 rows (4096 x 5632 at 704 46.6
    against 54.1, at 705 59.1 against 54.9; 1408 x 16384 at 704 43.2 against
    49.5, at 960 57.9 against 55.6), the widest at once (1024 x 20480 at 576
    44.7 against 43.0). Rows shorter than 1024 weights run shapes chosen by
    their grid alone, which lose here and there past 512 outputs (128 x 1024
    at 576 12.0 against 8.3)."""
    weights = n * k
    if weights > 24_000_000 or (k < 1024 and n > 512):
        return NATIVE_GEMM_MAX_ROWS
    if n <= 2048 or weights <= 12_000_000 or (n <= 4096 and weights <= 17_500_000):
        return 2 * NATIVE_GEMM_MAX_ROWS
    return 704 if n <= 16384 else NATIVE_GEMM_MAX_ROWS


class QuantizedLinear(torch.nn.Module):
    """Inference-only linear layer backed by packed INT4 weights."""

    def __init__(
        self,
        packed_weights: torch.Tensor,
        scales: torch.Tensor,
        group_size: int = 128,
        bias: torch.Tensor | None = None,
        fused: bool = True,
    ) -> None:
        super().__init__()
        if packed_weights.dtype != torch.uint8 or packed_weights.ndim != 2:
            raise ValueError("packed_weights must be uint8 with shape [N, K / 2]")
        if scales.dtype != torch.float16 or scales.ndim != 2:
            raise ValueError("scales must be float16 with shape [N, K / group_size]")
        if packed_weights.device != scales.device:
            raise ValueError("packed_weights and scales must share a device")
        if group_size <= 0:
            raise ValueError("group_size must be greater than zero")

        self.out_features = packed_weights.shape[0]
        self.in_features = packed_weights.shape[1] * 2
        self.group_size = group_size
        if self.in_features % group_size != 0:
            raise ValueError("K must be divisible by group_size")
        expected = (self.out_features, self.in_features // group_size)
        if tuple(scales.shape) != expected:
            raise ValueError(f"scales must have shape {expected}")
        if bias is not None:
            if bias.dtype != torch.float16 or tuple(bias.shape) != (self.out_features,):
                raise ValueError("bias must be float16 with shape [N]")
            if bias.device != packed_weights.device:
                raise ValueError("bias and packed_weights must share a device")

        self.register_buffer("packed_weights", packed_weights.detach())
        self.register_buffer("scales", scales.detach())
        self.register_buffer("bias", None if bias is None else bias.detach())
        self.fused = fused
        # prompt rows up to this count take the W4A16 GEMM when fused (set it
        # to FUSED_MAX_ROWS for the reference's routing: dequantize + GEMM for
        # every M > 8; a value that is set stands as it is, whatever the layer)
        self.native_max_rows = gemm_max_rows(self.out_features, self.in_features)

    @classmethod
    def from_float(cls, layer: torch.nn.Linear, group_size: int = 128, fused: bool = True) -> "QuantizedLinear":
        """Quantize an ``nn.Linear`` (reference ``w4a16/linear.py:58-83``)."""
        if not isinstance(layer, torch.nn.Linear):
            raise TypeError("layer must be an instance of torch.nn.Linear")
        packed, scales = quantize_and_pack_weights(layer.weight.detach(), group_size)
        bias = None if layer.bias is None else layer.bias.detach().to(torch.float16)
        return cls(packed, scales, group_size=group_size, bias=bias, fused=fused)

    @classmethod
    def empty(
        cls,
        out_features: int,
        in_features: int,
        group_size: int = 128,
        bias: bool = False,
        fused: bool = True,
        device: torch.device | str | None = None,
    ) -> "QuantizedLinear":
        """Uninitialised packed storage of the right shapes (reference ``w4a16/linear.py:85-130``)."""
        if out_features <= 0 or in_features <= 0:
            raise ValueError("out_features and in_features must be greater than zero")
        if in_features % 2 != 0:
            raise ValueError("in_features must be even")
        if group_size <= 0:
            raise ValueError("group_size must be greater than zero")
        if in_features % group_size != 0:
            raise ValueError("K must be divisible by group_size")
        device = torch.device("cpu") if device is None else device
        packed = torch.empty((out_features, in_features // 2), dtype=torch.uint8, device=device)
        scales = torch.empty((out_features, in_features // group_size), dtype=torch.float16, device=device)
        bias_tensor = torch.empty((out_features,), dtype=torch.float16, device=device) if bias else None
        return cls(packed, scales, group_size=group_size, bias=bias_tensor, fused=fused)

    def extra_repr(self) -> str:
        return (
            f"in_features={self.in_features}, out_features={self.out_features}, "
            f"group_size={self.group_size}, bias={self.bias is not None}, fused={self.fused}"
        )

    def _takes_gemm(self, flat: torch.Tensor) -> bool:
        """Whether these prompt rows take the W4A16 GEMM: up to ``native_max_rows``.
        Past NATIVE_GEMM_MAX_ROWS only rows and weights that start on 16 bytes,
        which the GEMM needs: the library's scalar kernel, which takes the
        others, is far behind the dense GEMM there, and dequantize refuses such
        weights. Where a tensor has no address to test (torch.compile and the
        like) these rows keep dequantize + the dense GEMM."""
        rows = flat.shape[0]
        if rows > self.native_max_rows or rows <= NATIVE_GEMM_MAX_ROWS:
            return rows <= self.native_max_rows
        packed = self.packed_weights
        return addressable(flat, packed) and (flat.data_ptr() | packed.data_ptr()) % 16 == 0

    def _dequant_linear(self, activations: torch.Tensor) -> torch.Tensor:
        """fp16 weight matrix from the packed codes, then a dense GEMM."""
        if self.packed_weights.is_cuda:
            weight = dequantize_cuda(self.packed_weights, self.scales, self.group_size)
        else:
            weight = dequantize_weights(self.packed_weights, self.scales, self.group_size).to(torch.float16)
        return F.linear(activations, weight)

    def forward(self, activations: torch.Tensor) -> torch.Tensor:
        if activations.ndim < 1:
            raise ValueError("activations must have at least one dimension")
        in_features = self.in_features
        if activations.shape[-1] != in_features:
            raise ValueError("activations last dimension must equal in_features")
        if activations.dtype != torch.float16:
            raise TypeError("activations must have dtype torch.float16")
        if activations.requires_grad:
            raise RuntimeError("activations must not require grad")
        packed, scales = self.packed_weights, self.scales   # buffers: each look-up costs about 0.3 us
        if activations.device != packed.device:
            raise ValueError("activations and packed_weights must share a device")

        # The kernels need a dense [M, K] matrix; views from attention reshapes are copied.
        # Rows of no features have no row count to infer, and the reshape refuses them.
        matrix = activations.ndim == 2 and in_features > 0
        flat = activations.contiguous() if matrix else activations.contiguous().reshape(-1, in_features)
        rows = flat.shape[0]
        if flat.is_cuda:
            if not packed.is_contiguous():
                raise ValueError("packed_weights must be contiguous")
            if not scales.is_contiguous():
                raise ValueError("scales must be contiguous")
            if self.fused and rows <= FUSED_MAX_ROWS:
                out = linear_cuda(flat, packed, scales, self.group_size)
            elif self.fused and self.group_size == 128 and self._takes_gemm(flat):
                out = linear_cuda(flat, packed, scales, self.group_size)
            elif self.group_size % 32 == 0:
                out = self._dequant_linear(flat)
            else:
                out = linear_cuda(flat, packed, scales, self.group_size)
        else:
            out = linear_reference(flat, packed, scales, self.group_size)
        if not matrix:
            out = out.reshape(*activations.shape[:-1], self.out_features)
        bias = self.bias
        return out if bias is None else out + bias


# The name the W4A16 API documentation uses for the same class.
Int4Linear = QuantizedLinear
