"""Chunked prefill in fp32 arithmetic (fp32 caches, and 16-bit ones at head_dim 16) against
attention in float64, at the edges of its tiles: 64 query rows, 16 / 32 / 64 keys, two halves."""

from __future__ import annotations

import pytest
import torch

from engine import workloads
from engine.kernels import paged_attention as pa

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
# |V| < 6 times fp32 scores of a few ulps (|s| < 16) and fp32 sums
TOL = 6 * 16 * 2.0**-22


def _exact(step, lens):
    q, k, v = step_q(step), step.k_cache.cpu().double(), step.v_cache.cpu().double()
    g, bs = q.shape[1] // k.shape[1], step.block_size
    out, at = torch.zeros(q.shape, dtype=torch.float64), 0
    for c, (m, n) in enumerate(zip(lens, step.context_lens.tolist(), strict=True)):
        p = torch.arange(n)
        slots = step.block_tables[c].cpu().long()[p // bs] * bs + p % bs
        kb, vb = (x[slots].repeat_interleave(g, 1).transpose(0, 1) for x in (k, v))
        s = (q[at : at + m].transpose(0, 1) @ kb.transpose(1, 2)) * q.shape[-1] ** -0.5
        s = s.masked_fill(p[None, None] > (n - m + torch.arange(m))[None, :, None], float("-inf"))
        out[at : at + m] = (torch.softmax(s, -1) @ vb).transpose(0, 1)
        at += m
    return out


def step_q(step):
    return step.info["q"].cpu().double()


@pytest.mark.parametrize(("hd", "dtype"), [(16, torch.float32), (32, torch.float32), (64, torch.float32),
                                           (128, torch.float32), (256, torch.float32),
                                           (16, torch.bfloat16), (16, torch.float16)])  # fmt: skip
@pytest.mark.parametrize(("nh", "nkv", "bs"), [(4, 4, 16), (6, 2, 5), (8, 2, 16), (7, 1, 64)])
def test_tile_edges(nh, nkv, bs, hd, dtype):
    lens = [1, 15, 16, 17, 64, 65, 9, 33]
    cached = [0, 0, 16, 111, 1, 0, 500, 31]
    step = workloads.custom([a + b for a, b in zip(lens, cached, strict=True)], nh, nkv, hd, bs,
                            dtype, DEV, seed=hd)  # fmt: skip
    q = torch.randn(sum(lens), nh, hd, device=DEV).to(dtype)
    step.info["q"] = q
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], dtype=torch.int32, device=DEV)
    print("[case] prefill f32", nh, nkv, hd, bs, dtype, flush=True)
    out = torch.full(q.shape, float("nan"), device=DEV)
    args = (step.k_cache, step.v_cache, step.block_tables, step.context_lens, bs, cu, max(lens))
    pa.paged_prefill_attention(q, *args, out=out)
    rounded = pa.paged_prefill_attention(q, *args)
    torch.cuda.synchronize()
    err = (out.cpu().double() - _exact(step, lens)).abs().max().item()
    assert err <= TOL, err
    assert torch.equal(rounded, out.to(dtype))


def test_more_items_than_one_grid_dimension_holds():
    """A bound on the chunks' lengths far above them: 2,100 x 512 x 8 items of 512 threads, past
    HIP's 2^32 along x; nearly all of them empty."""
    lens = [1 + i % 3 for i in range(2100)]
    step = workloads.custom([n + i % 40 for i, n in enumerate(lens)], 8, 8, 16, 16, torch.float32, DEV, seed=1)
    q = torch.randn(sum(lens), 8, 16, device=DEV)
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], dtype=torch.int32, device=DEV)
    args = (q, step.k_cache, step.v_cache, step.block_tables, step.context_lens, 16, cu)
    assert torch.equal(pa.paged_prefill_attention(*args, 32768), pa.paged_prefill_attention(*args, 3))


@pytest.mark.parametrize(("hd", "dtype"), [(16, torch.float32), (16, torch.bfloat16), (64, torch.float32),
                                           (128, torch.float32), (256, torch.float32)])  # fmt: skip
@pytest.mark.parametrize("groups", [1, 2, 3, 8])
@pytest.mark.parametrize("value", [float("inf"), float("nan")])
def test_later_values_do_not_reach_earlier_rows(groups, hd, dtype, value):
    """An infinite or NaN V of a token shows in its own row and the later ones of its chunk, in its
    dim, and nowhere else (an earlier row's P is 0 there, and 0 x inf is NaN): also where out is q."""
    lens, cached = [90, 33], [37, 0]
    step = workloads.custom([127, 33], 2 * groups, 2, hd, 16, dtype, DEV, seed=hd)
    q = torch.randn(sum(lens), 2 * groups, hd, device=DEV).to(dtype)
    step.info["q"] = q
    cu = torch.tensor([0, 90, 123], dtype=torch.int32, device=DEV)
    want = _exact(step, lens)
    for c, t in ((0, 40), (0, 89), (1, 20)):  # token t of chunk c
        p = cached[c] + t
        step.v_cache[int(step.block_tables[c, p // 16]) * 16 + p % 16, :, hd // 2] = value
    args = (step.k_cache, step.v_cache, step.block_tables, step.context_lens, 16, cu, 90)
    out = torch.empty(q.shape, device=DEV)
    rounded = q.clone()
    pa.paged_prefill_attention(q, *args, out=out)
    pa.paged_prefill_attention(rounded, *args, out=rounded, rows=torch.arange(123, device=DEV))
    assert torch.equal(rounded.nan_to_num(7.0), out.to(dtype).nan_to_num(7.0))
    out = out.cpu().double()
    hit = torch.zeros(out.shape, dtype=torch.bool)
    hit[[*range(40, 90), *range(110, 123)], :, hd // 2] = True
    assert (out[~hit] - want[~hit]).abs().max().item() <= TOL
    assert (out[hit].isnan() if value != value else out[hit] == value).all()
