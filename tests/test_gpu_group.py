"""Group sizes 32 and 64 at M = 1..8 on the matrix-core form of the generic
family (w4a16_group.hip), through the default route and every launch shape,
against the fp32 oracle."""

from __future__ import annotations

import pytest
import torch

from tests._cases import assert_parity, expected, make_case
from nibble_amd import _lib

pytestmark = pytest.mark.gpu


def _on(gpu, *tensors):
    return [t.to(gpu) for t in tensors]


# one run, an odd run count (a padded half pair), ragged N, rows that fill LDS (14336 at M = 8: two launches)
@pytest.mark.parametrize("k,n", [(128, 8), (128, 5), (384, 19), (640, 250), (1024, 64), (2176, 515), (4096, 4100),
                                 (2048, 8200), (14336, 24)])
@pytest.mark.parametrize("group", [32, 64])
@pytest.mark.parametrize("m", [1, 2, 4, 5, 8])
def test_group_default_route(gpu, m, group, k, n):
    x, p, s = make_case(m, k, n, seed=k + n + m, all_nibbles=True, group_size=group)
    xd, pd, sd = _on(gpu, x / 8, p, s)
    plan = _lib.plan_linear(xd.data_ptr(), pd.data_ptr(), m, n, k, group)
    print(f"[case] M={m} K={k} N={n} G={group} {plan}", flush=True)
    assert plan["kernel"] == "generic" and plan["max_blocks"] == 1
    out = torch.full((m, n), float("nan"), dtype=torch.float16, device=gpu)
    _lib.linear_f16(xd, pd, sd, out, group)
    torch.cuda.synchronize()
    assert_parity(out, expected(x / 8, p, s, group), f"M={m} K={k} N={n} G={group}")


@pytest.mark.parametrize("splits,rows", [(1, 1), (1, 8), (2, 3), (4, 2), (8, 1)])
@pytest.mark.parametrize("depth", [1, 2, 4])
@pytest.mark.parametrize("m,group", [(1, 64), (1, 32), (3, 32), (8, 64)])
def test_group_launch_shapes(gpu, m, group, splits, rows, depth):
    k, n = 9 * 128, 100   # 5 run pairs, the last half padded: wavefronts with none at 8 splits
    x, p, s = make_case(m, k, n, seed=splits + depth, group_size=group)
    xd, pd, sd = _on(gpu, x, p, s)
    out = torch.full((m, n), float("nan"), dtype=torch.float16, device=gpu)
    print(f"[case] M={m} G={group} splits={splits} rows={rows} depth={depth}", flush=True)
    _lib.linear_f16_tuned(xd, pd, sd, out, group, _lib.KERNEL_GENERIC, rows, splits, depth, 1)
    torch.cuda.synchronize()
    assert_parity(out, expected(x, p, s, group), f"M={m} G={group} {splits}x{rows} D={depth}")


@pytest.mark.parametrize("rows,splits,depth", [(1, 3, 1), (0, 0, 0), (-1, 1, 1), (2, 8, 1), (9, 1, 1), (1, 16, 1),
                                               (1, 2, 3), (1, 1, 8)])
def test_generic_takes_any_other_arguments(gpu, rows, splits, depth):
    """Arguments that are no shape of the matrix-core form are ignored: the scalar kernel's bits."""
    x, p, s = make_case(2, 384, 24, seed=7, group_size=64)
    xd, pd, sd = _on(gpu, x, p, s)
    got = []
    for max_blocks in (0, 1):
        out = torch.full((2, 24), float("nan"), dtype=torch.float16, device=gpu)
        print(f"[case] rows={rows} splits={splits} depth={depth} max_blocks={max_blocks}", flush=True)
        _lib.linear_f16_tuned(xd, pd, sd, out, 64, _lib.KERNEL_GENERIC, rows, splits, depth, max_blocks)
        torch.cuda.synchronize()
        got.append(out)
    assert_parity(got[0], expected(x, p, s, 64), "scalar")
    assert torch.equal(*got)


def test_group_scales_of_other_alignment_and_inf(gpu):
    """Scales that are only 2-byte aligned keep the scalar kernel; a non-finite
    scale or activation of one group reaches only its own outputs."""
    for group in (32, 64):
        x, p, s = make_case(2, 640, 24, seed=group, group_size=group)
        s[3, 1] = float("inf")
        x[1, 7] = float("inf")
        xd, pd = _on(gpu, x, p)
        store = torch.empty((s.numel() + 1,), dtype=torch.float16, device=gpu)
        store[1:] = s.to(gpu).reshape(-1)
        got = []
        for sd in (s.to(gpu), store[1:].view_as(s)):
            out = torch.empty((2, 24), dtype=torch.float16, device=gpu)
            print(f"[case] G={group} scales at {sd.data_ptr() % 16}", flush=True)
            _lib.linear_f16(xd, pd, sd, out, group)
            torch.cuda.synchronize()
            got.append(out.float().cpu())
        finite = torch.isfinite(got[1])
        assert torch.equal(finite, torch.isfinite(got[0]))
        assert finite[0].sum() == 23 and not finite[0, 3]
        assert torch.allclose(got[0][finite], got[1][finite], rtol=1e-3, atol=1e-3)


@pytest.mark.parametrize("group", [32, 64])
@pytest.mark.parametrize("m,k,splits", [(1, 128, 0), (1, 1152, 0), (4, 640, 0), (8, 384, 0), (8, 2176, 8), (3, 1152, 1)])
def test_group_infinite_scales(gpu, m, k, group, splits):
    """An infinite scale gives what the sum over code * scale * x gives: NaN
    with a code or an activation of 0 in its group or products of both signs,
    else an infinity of their sign; other rows of the layer keep their bits."""
    n, groups = 12, k // group
    x, p, s = make_case(m, k, n, seed=k + m + group, group_size=group)
    plain = s.clone()
    x[0] = 1.0 + x[0].abs()                       # one sign in activation row 0
    inf = float("inf")
    s[0, groups // 2] = inf                       # random codes: both signs
    s[1, 0], p[1, :group // 2] = inf, 0x33        # one sign
    s[2, groups - 1], p[2, -group // 2:] = -inf, 0x33
    s[3, 0], p[3, :group // 2], p[3, 0] = inf, 0x33, 0x03   # one code of 0
    s[4, 0], s[4, groups - 1] = inf, -inf         # one sign each, of different signs
    p[4, :group // 2], p[4, -group // 2:] = 0x33, 0x33
    s[5, groups // 2] = float("nan")
    xd, pd, sd = _on(gpu, x, p, s)
    out = torch.full((m, n), float("nan"), dtype=torch.float16, device=gpu)
    print(f"[case] infinite scales M={m} K={k} G={group} splits={splits}", flush=True)
    if splits:
        _lib.linear_f16_tuned(xd, pd, sd, out, group, _lib.KERNEL_GENERIC, 1, splits, 2, 1)
    else:
        _lib.linear_f16(xd, pd, sd, out, group)
    torch.cuda.synchronize()
    got = out.float().cpu()
    codes = ((torch.stack((p & 15, p >> 4), dim=-1).reshape(n, k).int() ^ 8) - 8).float()
    wide = codes * s.float().repeat_interleave(group, dim=1)
    terms = x.float().unsqueeze(1) * wide.unsqueeze(0)           # [m, n, k]
    want = terms.sum(dim=2)
    assert torch.equal(got.isnan(), want.isnan())
    assert torch.equal(got.isposinf(), want.isposinf()) and torch.equal(got.isneginf(), want.isneginf())
    assert got[0, 0].isnan() and got[0, 1] == inf and got[0, 2] == -inf and got[0, 3:6].isnan().all()
    assert_parity(out[:, 6:], expected(x, p[6:], plain[6:], group), f"M={m} K={k} G={group}")
