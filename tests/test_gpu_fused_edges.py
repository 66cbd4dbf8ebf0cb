"""The fused element-wise kernels bit for bit against the PyTorch ops where their loops and
rounding can go wrong: rows past a workgroup, strided and odd rows, RoPE's several heads per
thread and tokens per workgroup, NaN and infinity, the row scale's rsqrt."""

from __future__ import annotations

import pytest
import torch
import torch.nn.functional as F

from engine.kernels import fused

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
DTYPES = [torch.float32, torch.bfloat16, torch.float16]


def _same(got, want):
    """Equal values, NaN where NaN; for 16-bit types PyTorch's own NaN bits."""
    if got.dtype == torch.float32:
        return torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0)) and torch.equal(got.isnan(), want.isnan())
    return torch.equal(got.view(torch.int16), want.view(torch.int16))


def _rms(x, w, eps):
    xf = x.float()
    return w * (xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + eps)).to(x.dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize(("rows", "cols"), [(1, 8), (3, 2048), (5, 2056), (70000, 8), (9, 4099), (2, 16384)])
def test_rms_norm(rows, cols, dtype):
    print("[case] rms", rows, cols, dtype, flush=True)
    x = torch.randn(rows, cols + 8, device=DEV).to(dtype)[:, :cols]  # strided rows
    w = torch.randn(cols, device=DEV).to(dtype)
    assert _same(fused.rms_norm(x, w, 1e-5), _rms(x, w, 1e-5))
    x = x.contiguous()
    x[0, 0] = float("inf")
    x[-1, cols // 2] = float("nan")
    assert _same(fused.rms_norm(x, w, 0.0), _rms(x, w, 0.0))


@pytest.mark.parametrize("scale", [1e-20, 1e-3, 1.0, 300.0, 1e15])
def test_row_scale_has_pytorch_bits(scale):
    """One value per row: the scale is rsqrt(x^2 + eps) of 200,000 different x."""
    x = (torch.randn(200000, 1, device=DEV) * scale).abs() + 1e-38
    w = torch.ones(1, device=DEV)
    for eps in (0.0, 1e-6):
        assert _same(fused.rms_norm(x, w, eps), _rms(x, w, eps))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize(("n", "heads", "hd"), [(1, 1, 16), (3, 5, 64), (700, 3, 32), (2200, 31, 128),
                                                (2200, 33, 256), (9000, 9, 64), (40, 300, 256),
                                                (600, 130, 512)])  # fmt: skip
def test_rope(n, heads, hd, dtype):
    """Below and above the size where a thread takes four heads, heads no multiple of four,
    tokens with more and fewer items than a workgroup has threads."""
    print("[case] rope", n, heads, hd, dtype, flush=True)
    x = torch.randn(n, heads + 3, hd, device=DEV).to(dtype)
    x[0, 0, 0], x[-1, 0, 3] = float("inf"), float("nan")
    ang = torch.randn(n, hd, device=DEV) * 50
    cos, sin = ang.cos(), ang.sin()
    p = x[:, 1 : 1 + heads].clone()
    want = p * cos[:, None].to(dtype) + torch.cat((-p[..., hd // 2 :], p[..., : hd // 2]), -1) * sin[:, None].to(dtype)
    rest = x.clone()
    fused.rope_(x[:, 1 : 1 + heads], cos, sin)
    assert _same(x[:, 1 : 1 + heads], want)
    assert _same(x[:, :1], rest[:, :1]) and _same(x[:, 1 + heads :], rest[:, 1 + heads :])


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_silu_mul_every_value(dtype):
    """All 65,536 gates, NaNs and infinities among them."""
    g = torch.arange(65536, device=DEV, dtype=torch.int32).to(torch.int16).view(dtype)
    for u in (1.0, -0.37, 3.0e4, float("inf"), float("nan")):
        up = torch.full_like(g, u)
        assert _same(fused.silu_mul(g, up), F.silu(g) * up)


@pytest.mark.parametrize("dtype", DTYPES)
def test_silu_mul_streamed(dtype):
    """Outputs past the L2s take streaming accesses: the first size and one vector less."""
    vec = 16 // torch.empty(0, dtype=dtype).element_size()
    n = (32 << 20) // 16 * vec
    for m in (n - vec, n):
        print("[case] silu", m, dtype, flush=True)
        g, u = (torch.randn(m, device=DEV).to(dtype) for _ in range(2))
        g[-3], u[5] = float("nan"), float("inf")
        assert _same(fused.silu_mul(g, u), F.silu(g) * u)


def test_rms_norm_more_rows_than_a_grid_holds():
    """2^24 workgroups of 256 threads are past HIP's 2^32 threads along x."""
    rows = (1 << 24) + 3
    x = torch.randn(rows, 8, device=DEV).bfloat16()
    w = torch.randn(8, device=DEV).bfloat16()
    got = fused.rms_norm(x, w, 1e-5)
    for lo in range(0, rows, 1 << 22):
        assert _same(got[lo : lo + (1 << 22)], _rms(x[lo : lo + (1 << 22)], w, 1e-5))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("cols", [1, 3, 4, 8, 12, 33, 64, 72, 128, 256, 264, 511, 512, 520, 1032])
@pytest.mark.parametrize("rows", [1, 7, 2053])
def test_rms_norm_several_rows_per_workgroup(rows, cols, dtype):
    """Rows of 1 to 64 vectors share workgroups, in both widths of access; the last workgroup is
    partly filled. 65,535 workgroups along y and a row more go round the loop."""
    x = torch.randn(rows, cols + 8, device=DEV).to(dtype)[:, :cols]
    w = torch.randn(cols, device=DEV).to(dtype)
    assert _same(fused.rms_norm(x, w, 1e-5), _rms(x, w, 1e-5))
    w32 = w.float()  # another weight dtype: one element per access
    assert _same(fused.rms_norm(x, w32, 1e-5), _rms(x, w32, 1e-5))


def test_rms_norm_rows_past_the_grid():
    x = torch.randn(65535 * 4 + 5, 33, device=DEV)
    w = torch.randn(33, device=DEV)
    assert _same(fused.rms_norm(x, w, 1e-5), _rms(x, w, 1e-5))
