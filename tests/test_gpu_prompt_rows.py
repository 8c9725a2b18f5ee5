"""Prompt rows (M > 16) where the library chooses the GEMM shape by estimated
time, and the rows past which QuantizedLinear hands over to the dense GEMM."""

from __future__ import annotations

import pytest
import torch

from nibble_amd.cuda import dequantize_cuda
from nibble_amd.linear import NATIVE_GEMM_MAX_ROWS, QuantizedLinear, gemm_max_rows
from tests._cases import make_case


# a row past a tile of 16, 32, 64 and 128, and past a second round of tiles;
# K from the least that is chosen by time, and group counts that no K split
# divides (9, 11, 13); N below one tile, ragged, and an even number of tiles
@pytest.mark.gpu
@pytest.mark.parametrize("m", [17, 24, 32, 33, 65, 127, 200, 385, 513, 700, 1024])
@pytest.mark.parametrize("k,n", [(1024, 24), (1152, 515), (1408, 4100), (1664, 1000), (2048, 5632), (5632, 2049)])
def test_prompt_rows_by_estimated_time(gpu, m, k, n):
    """The op against 64-bit sums over the dequantized weights: half an ulp of
    the fp16 output, and for the fp32 sums 2^-23 of the sum of magnitudes for
    each of the K / 16 + 32 additions that one output passes through at most."""
    x, p, s = (t.to(gpu) for t in make_case(m, k, n, seed=m + k + n))
    print(f"[case] M={m} K={k} N={n}", flush=True)
    out = torch.ops.w4a16.linear(x, p, s, 128)
    torch.cuda.synchronize()
    wt = dequantize_cuda(p, s, 128).double().t().contiguous()
    ref, size = x.double() @ wt, x.double().abs() @ wt.abs()
    bound = ref.abs() * 2 ** -11 + (k / 16 + 32) * 2 ** -23 * size + 2 ** -25
    err = (out.double() - ref).abs()
    assert torch.all(err <= bound), f"worst {float((err / bound).max()):.3f} of the bound"


def _layer(n, k):
    return QuantizedLinear(torch.zeros((n, k // 2), dtype=torch.uint8), torch.ones((n, k // 128), dtype=torch.float16))


def test_rows_that_take_the_gemm():
    top = NATIVE_GEMM_MAX_ROWS
    rows = torch.zeros((2 * top + 2, 256), dtype=torch.float16)
    small = _layer(8, 256)
    assert [small._takes_gemm(rows[:m]) for m in (top, top + 1, 2 * top, 2 * top + 1)] == [True, True, True, False]
    shifted = rows.reshape(-1)[1:1 + (top + 1) * 256].view(top + 1, 256)   # contiguous, 2 bytes past the alignment
    assert not small._takes_gemm(shifted) and small._takes_gemm(shifted[:top])
    small.native_max_rows = 100
    assert small._takes_gemm(rows[:100]) and not small._takes_gemm(rows[:101])
    large = _layer(96000, 256)   # 24.6M weights
    assert large._takes_gemm(rows[:top]) and not large._takes_gemm(rows[:top + 1])


@pytest.mark.parametrize("k,n,rows", [
    (2048, 2048, 1024), (5632, 2048, 1024), (11008, 2048, 1024), (14336, 1536, 1024), (2048, 4096, 1024),
    (4096, 4096, 1024), (2048, 5632, 1024), (1024, 8192, 1024), (128, 512, 1024),    # faster up to 1024 rows
    (8192, 2560, 704), (4096, 5632, 704), (2048, 11264, 704), (1408, 16384, 704), (1024, 16384, 704),
    (2816, 8192, 704),                                                               # slower past 704
    (1024, 20480, 512), (128, 1024, 512), (512, 16384, 512), (4096, 6144, 512)])
def test_rows_up_to_which_the_gemm_keeps_up(k, n, rows):
    assert gemm_max_rows(n, k) == rows


def test_rows_that_a_caller_sets_stand():
    """512 set by a caller is no more than 512, on a small layer, too; a larger value counts on a large one."""
    top = NATIVE_GEMM_MAX_ROWS
    rows = torch.zeros((2 * top + 2, 256), dtype=torch.float16)
    small, large = _layer(8, 256), _layer(96000, 256)
    small.native_max_rows = top
    assert small._takes_gemm(rows[:top]) and not small._takes_gemm(rows[:top + 1])
    large.native_max_rows = 2 * top + 1
    assert large._takes_gemm(rows[:2 * top + 1]) and not large._takes_gemm(rows)


def _past_alignment(dtype, shape, shift):
    """A tensor whose own storage starts `shift` bytes past 16, at storage offset 0."""
    size = torch.zeros(shape, dtype=dtype).nbytes
    buffer = bytearray(size + 32)
    start = -torch.frombuffer(buffer, dtype=torch.uint8).data_ptr() % 16 + shift
    out = torch.frombuffer(buffer, dtype=dtype, offset=start, count=size // dtype.itemsize).view(shape)
    assert out.data_ptr() % 16 == shift and out.storage_offset() == 0
    return out


def test_rows_that_take_the_gemm_start_on_16_bytes():
    """The address decides, not the offset within a storage that may itself start anywhere."""
    rows = NATIVE_GEMM_MAX_ROWS + 1
    layer = _layer(8, 256)
    for shift in range(0, 16, 2):
        assert layer._takes_gemm(_past_alignment(torch.float16, (rows, 256), shift)) == (shift == 0)
    store = _past_alignment(torch.float16, (rows * 256 + 1,), 14)   # one element on: 16-byte aligned
    assert layer._takes_gemm(store[1:].view(rows, 256))
    odd = QuantizedLinear(_past_alignment(torch.uint8, (8, 128), 4), torch.ones((8, 2), dtype=torch.float16))
    assert odd._takes_gemm(torch.zeros((rows - 1, 256), dtype=torch.float16))
    assert not odd._takes_gemm(torch.zeros((rows, 256), dtype=torch.float16))


@pytest.mark.gpu
def test_module_refuses_misaligned_weights_past_the_gemm(gpu):
    """dequantize refuses weights that do not start on 16 bytes; the module does at these rows, too."""
    _, p, s = make_case(1, 256, 8, seed=0)
    store = torch.empty((p.numel() + 4,), dtype=torch.uint8, device=gpu)
    store[4:] = p.reshape(-1).to(gpu)
    layer = QuantizedLinear(store[4:].view_as(p), s.to(gpu))
    for rows in (513, 1024, 1025):
        with pytest.raises(RuntimeError, match="16-byte aligned"):
            layer(torch.zeros((rows, 256), dtype=torch.float16, device=gpu))


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [513, 1024, 1025])
@pytest.mark.parametrize("shift", [0, 1])
def test_module_rows_past_the_gemm(gpu, rows, shift):
    k, n = 1024, 520
    x, p, s = (t.to(gpu) for t in make_case(rows, k, n, seed=rows))
    store = torch.empty((rows * k + 1,), dtype=torch.float16, device=gpu)
    store[shift:shift + rows * k] = x.reshape(-1)
    view = store[shift:shift + rows * k].view(rows, k)
    print(f"[case] rows={rows} shift={shift}", flush=True)
    out = QuantizedLinear(p, s, group_size=128)(view)
    ref = x.double() @ dequantize_cuda(p, s, 128).double().t().contiguous()
    # the bound of the other module tests on dequantized weights
    torch.testing.assert_close(out.double(), ref, rtol=1e-3, atol=1e-3)
