"""The combine gives a (sequence, head) pair 1 to 16 waves by the number of pairs: every form
against one workgroup's single pass, at the edges of the rule, with more ranges than units
(empty ranges), sequences cut into few and many pieces, and cascade parts."""

from __future__ import annotations

import pytest
import torch

from engine import workloads
from engine.kernels import paged_attention as pa

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")
# |V| < 6 times the fp32 rounding of scores (|s| < 16, a few ulps) and of the merged sums
TOL = 6 * 16 * 2.0**-22


@pytest.mark.parametrize(("batch", "nh"), [(1, 8), (2, 32), (5, 13), (8, 32), (257, 1), (16, 32),
                                           (27, 19), (32, 32), (41, 25)])  # fmt: skip
@pytest.mark.parametrize(("hd", "dtype"), [(128, torch.bfloat16), (64, torch.float16), (16, torch.float32),
                                           (256, torch.float32)])  # fmt: skip
def test_waves_per_pair(batch, nh, hd, dtype):
    nkv = 1 if nh in (1, 13, 19, 25) else nh // 4
    ctx = [(i * 331 + 1900) % 2500 for i in range(batch)]
    ctx[batch // 2] = 0 if batch > 1 else ctx[0]
    step = workloads.custom(ctx, nh, nkv, hd, 16, dtype, DEV, seed=batch)
    args = (step.q, step.k_cache, step.v_cache, step.block_tables, step.context_lens, 16)
    print("[case]", step.name, batch, dtype, flush=True)
    one = torch.empty(step.q.shape, dtype=torch.float32, device=DEV)
    pa.paged_decode_attention(*args, out=one, num_workgroups=1)
    for wgs in (2, 61, 256, 3000):
        out = torch.full_like(one, float("nan"))
        pa.paged_decode_attention(*args, out=out, num_workgroups=wgs)
        torch.cuda.synchronize()
        assert (out - one).abs().max().item() <= TOL, wgs


@pytest.mark.parametrize(("batch", "nh"), [(2, 8), (3, 32), (8, 32), (16, 32), (30, 24)])
def test_cascade_parts(batch, nh):
    """Prefix parts go to a pair's first wave; sequences the stream pass finished too."""
    step = workloads.custom([400 + 50 * i for i in range(batch)], nh, nh // 4, 128, 16,
                            torch.bfloat16, DEV, seed=1)  # fmt: skip
    step.block_tables[:, :24] = step.block_tables[:1, :24]
    groups = pa.find_prefix_groups(step.block_tables, step.context_lens, 16, nh, nh // 4, DEV, pieces=3)
    args = (step.q, step.k_cache, step.v_cache, step.block_tables, step.context_lens, 16)
    print("[case] cascade", batch, nh, flush=True)
    plain, casc = (torch.empty(step.q.shape, dtype=torch.float32, device=DEV) for _ in range(2))
    pa.paged_decode_attention(*args, out=plain)
    for wgs in (1, 7, 500):
        pa.paged_decode_attention(*args, out=casc, prefix_groups=groups, num_workgroups=wgs)
        torch.cuda.synchronize()
        assert (casc - plain).abs().max().item() <= 2e-3, wgs  # the prefix pass's own bar
