"""Decode waves with both products on MFMA (GQA groups of 4 heads and more,
head_dim 128, 16-bit types) vs the float64 oracle where the form can go wrong:
block edges, heads that do not fill the 16 columns, split rows, an infinite V,
large and tiny scores.  Bars as for decode: 2e-3 max-abs plus one rounding of
the output."""

import numpy as np
import pytest
import torch

from oracle import paged_decode as opd
from pagelora_amd.attention_backend import PagedDecodeAttention
from tests.gpu_cases import ragged_case

pytestmark = pytest.mark.gpu

REL = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}


def _run(case, hq, hkv, ps, device, **kw):
    be = PagedDecodeAttention(device=device, workspace_mb=64, num_qo_heads=hq, num_kv_heads=hkv, head_dim=128,
                              page_size=ps, **kw)
    be.plan_decode(paged_kv_indptr=case["indptr"], paged_kv_indices=case["indices"],
                   paged_kv_last_page_len=case["last"])
    out = be.run_decode(case["q"], case["cache"])
    torch.cuda.synchronize()
    return out[:, :, 0].float().cpu().numpy()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("group", [4, 5, 6, 7, 8, 16])
@pytest.mark.parametrize("page_size,target_waves", [(16, None), (16, 8), (64, None), (8, None)])
def test_block_edges_and_splits(gpu_device, dtype, group, page_size, target_waves):
    hkv = 2
    lens = [1, 15, 16, 17, 33, 700]
    case = ragged_case(lens=lens, hq=group * hkv, hkv=hkv, head_dim=128, page_size=page_size, dtype=dtype,
                       device=gpu_device, seed=group, pool_extra=3)
    # scores far apart, so that the running maximum moves late and far
    case["q"][1:].mul_(8.0)
    case["q_host"][1:].mul_(8.0)
    got = _run(case, group * hkv, hkv, page_size, gpu_device, target_waves=target_waves)
    want, _ = opd.paged_decode(case["q_host"].float().numpy(), case["cache_host"].float().numpy(),
                               case["indptr"].numpy(), case["indices"].numpy(), case["last"].numpy())
    err = np.abs(got - want)
    assert (err <= 2e-3 + REL[dtype] * np.abs(want)).all(), f"max err {err.max():.3e}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_infinite_v_stays_infinite(gpu_device, dtype):
    """+inf in one dim of one token's V: that output dim is +inf, the others are the oracle's."""
    case = ragged_case(lens=[200, 40], hq=14, hkv=2, head_dim=128, page_size=16, dtype=dtype, device=gpu_device,
                       seed=3, pool_extra=2)
    page = int(case["indices"][0])
    case["cache"][page, 1, 5, 0, 9] = float("inf")
    got = _run(case, 14, 2, 16, gpu_device)
    want, _ = opd.paged_decode(case["q_host"].float().numpy(), case["cache_host"].float().numpy(),
                               case["indptr"].numpy(), case["indices"].numpy(), case["last"].numpy())
    assert np.isposinf(got[0, :7, 9]).all()
    mask = np.isfinite(got)
    assert mask.sum() == got.size - 7
    assert (np.abs(got - want)[mask] <= 2e-3 + REL[dtype] * np.abs(want)[mask]).all()
