"""Decode with 5 to 32 query heads per KV head at head_dim 64 and 128: one wave takes the
whole group (up to 16 heads), P.V on the matrix cores. Against attention in float64."""

from __future__ import annotations

import pytest
import torch

from engine import workloads
from engine.kernels import paged_attention as pa

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _exact(step):
    out = torch.zeros(step.q.shape, dtype=torch.float64)
    q, k, v = step.q.cpu().double(), step.k_cache.cpu().double(), step.v_cache.cpu().double()
    tables, bs = step.block_tables.cpu().long(), step.block_size
    g = q.shape[1] // k.shape[1]
    for b, n in enumerate(step.context_lens.tolist()):
        if n == 0:
            continue
        p = torch.arange(n)
        slots = tables[b, p // bs] * bs + p % bs
        kb, vb = (x[slots].repeat_interleave(g, 1).transpose(0, 1) for x in (k, v))
        w = torch.softmax((kb @ q[b, :, :, None])[..., 0] * q.shape[-1] ** -0.5, -1)
        out[b] = (w[:, None] @ vb)[:, 0]
    return out


def _tol(step):
    """|V| < 6 times P's relative error -- 2^-22 holds it at hd 128 (fp32, or three bf16 terms) and
    for two fp16 terms at hd 64, 2^-17 two bf16 terms at hd 64 -- plus fp32 scores of a few ulps (|s| < 16) and fp32 sums."""
    p = 2.0**-17 if step.q.shape[-1] == 64 and step.q.dtype == torch.bfloat16 else 2.0**-22
    return 6 * (p + 16 * 2.0**-23)


def _check(step, wgs=None):
    print("[case]", step.name, step.q.dtype, "wgs", wgs, flush=True)
    args = (step.q, step.k_cache, step.v_cache, step.block_tables, step.context_lens, step.block_size)
    out = torch.empty(step.q.shape, dtype=torch.float32, device=DEV)
    pa.paged_decode_attention(*args, out=out, num_workgroups=wgs)
    rounded = pa.paged_decode_attention(*args, num_workgroups=wgs)
    torch.cuda.synchronize()
    err = (out.cpu().double() - _exact(step)).abs().max().item()
    assert err <= _tol(step), err
    assert torch.equal(rounded, out.to(step.q.dtype))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("group", [5, 7, 8, 12, 16, 17, 32])
def test_groups(group, hd, dtype):
    nkv = 8 if group <= 8 else 2
    # tiles of 16: one token, one short of and past a tile, none, several ranges
    ctx = [1, 15, 16, 17, 0, 33, 700, 2100]
    _check(workloads.custom(ctx, group * nkv, nkv, hd, 16, dtype, DEV, seed=group))
    _check(workloads.custom(ctx, group * nkv, nkv, hd, 16, dtype, DEV, seed=group), wgs=61)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize(("nkv", "bs", "batch"), [(1, 16, 3), (3, 8, 5), (8, 32, 70), (4, 5, 130)])
def test_shapes(nkv, bs, batch, dtype):
    """KV heads that do not fill a workgroup, blocks that a tile crosses, staged batches."""
    ctx = [(37 * i) % 401 for i in range(batch)]
    _check(workloads.custom(ctx, 8 * nkv, nkv, 128, bs, dtype, DEV, seed=bs))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize(("nkv", "group", "bs"), [(8, 8, 16), (8, 7, 4), (4, 11, 16), (8, 16, 48)])
def test_split_pass(nkv, group, bs, hd, dtype):
    """Batches whose (sequence, KV head) pairs just fit the CUs: one launch, a workgroup per
    pair, at 1 to 2,016 tokens (some waves without any)."""
    ctx = [1 + (i * 211) % 2016 for i in range(256 // (8 * (2 if nkv == 4 else 1)) - 1)]
    ctx[3] = 0
    step = workloads.custom(ctx, group * nkv, nkv, hd, bs, dtype, DEV, seed=bs, width=2048 // bs)
    assert pa.default_workgroups(DEV, dtype, hd, group * nkv, nkv, len(ctx), 2048 // bs, bs) == 0
    _check(step)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_infinite_values_stay_infinite(dtype):
    """P enters P.V in terms of which some are 0: 0 x inf must not reach the output."""
    step = workloads.custom([90, 400], 64, 8, 128, 16, dtype, DEV, seed=3)
    slot = int(step.block_tables[1, 2]) * 16 + 5
    step.v_cache[slot, 3, 7] = float("inf")
    step.v_cache[slot, 5, 100] = float("-inf")
    out = pa.paged_decode_attention(step.q, step.k_cache, step.v_cache, step.block_tables,
                                    step.context_lens, 16)  # fmt: skip
    want = _exact(step)
    assert torch.equal(out.cpu().isinf(), want.isinf()) and not out.isnan().any()
    assert torch.equal(out.cpu()[want.isinf()].sign().double(), want[want.isinf()].sign())


@pytest.mark.parametrize(("nkv", "hd"), [(8, 128), (4, 128), (8, 64), (2, 128)])
def test_cascade(nkv, hd):
    """Cascade decode of 8 heads per KV head: wide waves (8 KV heads), narrow ones (4, to fill
    a workgroup), two launches (2); against the plain decode."""
    step = workloads.custom([320 + 9 * (i % 40) for i in range(96)], 8 * nkv, nkv, hd, 16,
                            torch.bfloat16, DEV, seed=1)  # fmt: skip
    step.block_tables[:, :20] = step.block_tables[:1, :20]
    groups = pa.find_prefix_groups(step.block_tables, step.context_lens, 16, 8 * nkv, nkv, DEV,
                                   dtype=torch.bfloat16, head_dim=hd)  # fmt: skip
    args = (step.q, step.k_cache, step.v_cache, step.block_tables, step.context_lens, 16)
    print("[case] cascade", nkv, hd, flush=True)
    outs = [torch.empty(step.q.shape, dtype=torch.float32, device=DEV) for _ in range(3)]
    pa.paged_decode_attention(*args, out=outs[0])
    pa.paged_decode_attention(*args, out=outs[1], prefix_groups=groups)
    pa.paged_decode_attention(*args, out=outs[2], prefix_groups=groups, prefix_workgroups=-1)
    torch.cuda.synchronize()
    # the prefix pass is the chunked prefill, whose bar is 2e-3
    assert (outs[1] - outs[0]).abs().max().item() <= 2e-3
    assert (outs[2] - outs[0]).abs().max().item() <= 2e-3


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("group", [4, 8, 16])
@pytest.mark.parametrize("wgs", [None, 1, 3])
def test_small_weights_keep_their_bits(group, wgs, dtype):
    """P is fp32 in P.V at every group size (hd 128): a weight of e^-25 (2^-36) beside one of 1,
    where the large V is the small weight's, and an infinite V at such a weight. The score -25
    carries an fp32 rounding of 25 2^-24, which the exponential makes the result's relative
    error; 2^-18 covers it and the sums."""
    step = workloads.custom([40, 90], 2 * group, 2, 128, 16, dtype, DEV, seed=5)
    step.q.zero_()
    step.q[..., 0] = 16
    step.k_cache.zero_()
    step.v_cache.zero_()
    p = torch.arange(90)
    for b, n in enumerate([40, 90]):
        slots = step.block_tables[b].cpu().long()[p[:n] // 16] * 16 + p[:n] % 16
        step.k_cache[slots.to(DEV), :, 0] = -17.6875  # scores -17.6875 sqrt(2) = -25.01
        step.k_cache[slots[7], :, 0] = 0
        step.v_cache[slots[11], :, 3:] = 6e4
        step.v_cache[slots[n - 3], 0, 1] = float("inf")
        step.v_cache[slots[n - 3], 1, 2] = float("-inf")
    out = torch.empty(step.q.shape, dtype=torch.float32, device=DEV)
    pa.paged_decode_attention(step.q, step.k_cache, step.v_cache, step.block_tables, step.context_lens,
                              16, out=out, num_workgroups=wgs)  # fmt: skip
    got, want = out.cpu().double(), _exact(step)
    assert torch.equal(got.isinf(), want.isinf()) and not got.isnan().any()
    assert torch.equal(got[want.isinf()], want[want.isinf()])
    fin = ~want.isinf()
    assert ((got - want)[fin].abs() <= 2.0**-18 * want[fin].abs()).all()


@pytest.mark.parametrize(("nh", "nkv", "ctx", "most"), [
    (128, 8, [2500], 64), (128, 8, [8000], 128), (64, 4, [20011], 256), (32, 2, [3000, 2800, 3300, 2900], 256),
    (16, 1, [20 + i % 80 for i in range(300)], 256), (8, 1, [20 + i % 80 for i in range(300)], 512),
    (16, 1, [250 + i % 50 for i in range(300)], 512), (32, 2, [250 + i % 50 for i in range(300)], 512),
    (40, 8, [300 + i for i in range(40)], 256),
    (15, 3, [2000 + i for i in range(300)], 512), (160, 16, [2500], 64)])  # fmt: skip
def test_default_ranges(nh, nkv, ctx, most):
    """The default split of the wide form cuts short batches into fewer ranges than the GPU holds:
    a range's records are a fraction of the K/V it reads."""
    step = workloads.custom(ctx, nh, nkv, 128, 16, torch.bfloat16, DEV, seed=2)
    wgs = pa.default_workgroups(DEV, torch.bfloat16, 128, nh, nkv, len(ctx), step.block_tables.shape[1], 16)
    cus = torch.cuda.get_device_properties(DEV).multi_processor_count
    print("[case] ranges", nh, nkv, len(ctx), wgs, flush=True)
    assert 32 <= wgs <= pa.decode_workgroups(DEV, torch.bfloat16, 128, nh, nkv)
    if cus == 256:
        assert wgs <= most
    if len(ctx) < 300:
        _check(step)
