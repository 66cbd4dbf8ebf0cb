"""Attention on rows of a step's q and out (``rows=``): which layouts the kernels take in
place (CPU), and that they give the gathered path's bits (GPU)."""

from __future__ import annotations

import pytest
import torch

from engine import workloads
from engine.kernels import paged_attention as pa
from engine.model.layers import mixed_attention
from engine.runtime.paged_cache import KVShape, PagedBatch, PagedKVCache

DEV = torch.device("cuda:0")


def test_layouts():
    rows = torch.arange(6)
    base = torch.zeros(2, 6, 4, 64, dtype=torch.bfloat16)
    q, out = base[0], base[1]
    ok = [(q, out), (q, q), (q[:3], q[3:]), (q[3:], q[:3]), (q[:0], out[:0])]
    head_major = torch.zeros(4, 6, 64, dtype=torch.bfloat16).transpose(0, 1)
    fused = torch.zeros(6, 12, 64, dtype=torch.bfloat16)
    ok += [(head_major, torch.empty_like(head_major)), (fused[:, :4], out), (head_major, out)]
    for a, b in ok:
        assert pa.rows_in_place(a, b, rows), (a.stride(), b.stride())
    bad = [(q, out.float()), (q[:4], q[2:]), (q, q.transpose(1, 2)), (q[..., :60], out[..., :60]),
           (q[:1].expand(6, 4, 64), out), (q[..., ::2], out[..., ::2]), (q, out[:5]),
           (torch.zeros(6 * 256 + 4, dtype=torch.bfloat16)[4:].view(6, 4, 64), out),
           (torch.zeros(6, 4, 68, dtype=torch.bfloat16)[..., :64], out),
           (fused[:, :4], fused[:, 2:6])]  # fmt: skip
    for a, b in bad[:3] + bad[4:]:
        assert not pa.rows_in_place(a, b, rows), (a.shape, a.stride(), b.stride())
    assert not pa.rows_in_place(q, out, rows.int())
    assert not pa.rows_in_place(q, out, torch.ones(6, dtype=torch.bool))
    assert not pa.rows_in_place(q, out, torch.arange(12)[::2])
    assert not pa.rows_in_place(q[0], out[0], rows)


def _layout(x, kind):
    if kind == "fused":  # a slice of a wider projection
        wide = torch.zeros(x.shape[0], x.shape[1] + 5, x.shape[2], dtype=x.dtype, device=x.device)
        wide[:, 2 : 2 + x.shape[1]] = x
        return wide[:, 2 : 2 + x.shape[1]]
    return x.transpose(0, 1).contiguous().transpose(0, 1) if kind == "head_major" else x


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["plain", "fused", "head_major", "in_place"])
@pytest.mark.parametrize(
    ("batch", "nh", "nkv", "hd", "dtype"),
    [(3, 8, 2, 64, torch.bfloat16),  # split pass
     (24, 64, 8, 128, torch.float16),  # split pass, wide
     (70, 32, 8, 128, torch.bfloat16),  # stream-K, staged
     (40, 32, 8, 64, torch.float16),  # stream-K
     (40, 40, 8, 128, torch.bfloat16),  # stream-K, wide
     (9, 6, 2, 32, torch.float32), (5, 4, 4, 256, torch.bfloat16)])  # fmt: skip
def test_decode_rows(batch, nh, nkv, hd, dtype, layout):
    step = workloads.custom([(61 * i) % 1500 for i in range(batch)], nh, nkv, hd, 16, dtype, DEV, seed=2)
    g = torch.Generator().manual_seed(4)
    n = 2 * batch + 3
    rows = torch.randperm(n, generator=g)[:batch]
    rows[0] -= n  # counts from the end
    rows = rows.to(DEV)
    q = _layout(torch.randn(n, nh, hd, device=DEV).to(dtype), layout)
    args = (step.k_cache, step.v_cache, step.block_tables, step.context_lens, 16)
    print("[case] rows", batch, nh, nkv, hd, dtype, layout, flush=True)
    for wgs in (None, 1, 37):
        q1 = q.clone(memory_format=torch.preserve_format)
        out = q1 if layout == "in_place" else torch.full_like(q1, 7.0)
        want = out.clone()
        want[rows] = pa.paged_decode_attention(q1[rows], *args, num_workgroups=wgs)
        pa.paged_decode_attention(q1, *args, out=out, num_workgroups=wgs, rows=rows)
        torch.cuda.synchronize()
        assert torch.equal(out, want), wgs


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["plain", "fused", "head_major", "in_place"])
@pytest.mark.parametrize(("hd", "dtype"), [(128, torch.bfloat16), (64, torch.float16), (64, torch.bfloat16),
                                           (256, torch.float16), (64, torch.float32), (16, torch.bfloat16)])  # fmt: skip
def test_prefill_rows(hd, dtype, layout):
    lens, cached = [70, 1, 0, 130], [0, 40, 9, 300]
    nh, nkv = 6, 2
    step = workloads.custom([a + b for a, b in zip(lens, cached, strict=True)], nh, nkv, hd, 16, dtype,
                            DEV, seed=3)  # fmt: skip
    cu = torch.tensor([0, 70, 71, 71, 201], dtype=torch.int32, device=DEV)
    n = 260
    rows = torch.randperm(n, generator=torch.Generator().manual_seed(1))[: sum(lens)]
    rows[5] -= n
    rows = rows.to(DEV)
    q = _layout(torch.randn(n, nh, hd, device=DEV).to(dtype), layout)
    out = q if layout == "in_place" else torch.full_like(q, 7.0)
    args = (step.k_cache, step.v_cache, step.block_tables, step.context_lens, 16, cu, 130)
    print("[case] prefill rows", hd, dtype, layout, flush=True)
    want = out.clone()
    want[rows] = pa.paged_prefill_attention(q[rows], *args)
    pa.paged_prefill_attention(q, *args, out=out, rows=rows)
    torch.cuda.synchronize()
    assert torch.equal(out, want)


@pytest.mark.gpu
def test_rows_outside_are_skipped():
    step = workloads.custom([30, 40, 50], 8, 2, 64, 16, torch.bfloat16, DEV, seed=2)
    q = torch.randn(4, 8, 64, device=DEV).bfloat16()
    args = (step.k_cache, step.v_cache, step.block_tables, step.context_lens, 16)
    for wgs in (None, 1, 9):
        out = torch.full_like(q, 7.0)
        rows = torch.tensor([1, 4, -5], device=DEV)
        pa.paged_decode_attention(q, *args, out=out, rows=rows, num_workgroups=wgs)
        torch.cuda.synchronize()
        assert (out[[0, 2, 3]] == 7).all() and not (out[1] == 7).any()
    with pytest.raises(ValueError, match="rows"):
        pa.paged_decode_attention(q, *args, rows=rows)


@pytest.mark.gpu
def test_plain_decode_keeps_its_registers():
    """The row lookup is a form of its own: in the plain one it cost registers, and fp32 at hd 64
    (4 heads per wave: 168 of them) a wave per SIMD, 2 workgroups of 4 waves per CU for 3."""
    cus = torch.cuda.get_device_properties(DEV).multi_processor_count
    assert pa.decode_workgroups(DEV, torch.float32, 64, 16, 4) == 3 * cus


def test_a_step_larger_than_q_is_refused():
    """A mixed step's row indices reach past a q (or out) of fewer rows: an IndexError, as from
    q[rows], and before any kernel that would skip such rows."""
    cache = PagedKVCache(KVShape(1, 2, 64), 8, 16, "cpu", torch.bfloat16)
    batch = PagedBatch.build(cache, [[0], [1, 2], [3]], [5, 20, 9], [1, 20, 9], "cpu", use_kernel=True)
    assert batch.num_tokens == 30
    q = torch.zeros(30, 4, 64, dtype=torch.bfloat16)
    with pytest.raises(IndexError, match="30 tokens"):
        mixed_attention(0, q[:29], batch)
    with pytest.raises(IndexError, match="30 tokens"):
        mixed_attention(0, q, batch, out=q[:29].clone())
