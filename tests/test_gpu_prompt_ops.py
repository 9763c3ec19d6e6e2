"""The prompt-sized fused element-wise kernels (one adapter bound to every row,
MFMA tiles) vs the row kernels they take over from, which the same call
with per-token ids still runs.

Both form round(base + scale * y . B^T) with fp32 sums in another order, so a
value may round to the neighbouring 16-bit one; the operations after it and
the final rounding then move a result by up to four units of its type."""

import pytest
import torch

from pagelora_amd import fused_ops

pytestmark = pytest.mark.gpu

ULP = {torch.bfloat16: 2.0**-7, torch.float16: 2.0**-10}


def _close(got, want, dtype, scale=1.0):
    got, want = got.float(), want.float()
    assert torch.isfinite(got).all()
    err = (got - want).abs()
    assert (err <= 4 * ULP[dtype] * torch.clamp(want.abs(), min=scale)).all(), f"max err {err.max()}"
    # most elements round alike
    assert (err > 0).float().mean() < 0.05


def _module(gen, rows, n, width, rank, dtype, device, y, y_offset):
    B = (torch.randn((n, width, rank), generator=gen) * 0.1).to(dtype).to(device)
    return [fused_ops.LoraUp(y, y_offset, B, 2.0, a) for a in (1, -1)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rank", [8, 16, 32])
@pytest.mark.parametrize("rows", [24, 33, 101, 1003])
@pytest.mark.parametrize("inter", [8, 264, 1024])
def test_silu_mul(gpu_device, dtype, rank, rows, inter):
    gen = torch.Generator().manual_seed(rows + inter + rank)
    n = 3
    gu = torch.randn((rows, 2 * inter + 2 * n * rank), generator=gen).to(dtype).to(gpu_device)
    gate = _module(gen, rows, n, inter, rank, dtype, gpu_device, gu, 2 * inter)
    up = _module(gen, rows, n, inter, rank, dtype, gpu_device, gu, 2 * inter + n * rank)
    ids = torch.ones(rows, dtype=torch.int32, device=gpu_device)
    got, want = (fused_ops.silu_mul(gu[:, : 2 * inter], lora=(g, u), adapter_ids=ids) for g, u in zip(gate, up))
    torch.cuda.synchronize()
    _close(got, want, dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rank", [8, 16, 32])
@pytest.mark.parametrize("rows,hq,hkv,norm", [(512, 7, 1, True), (600, 32, 8, True), (527, 4, 4, False),
                                              (2001, 7, 1, True), (1503, 4, 4, False)])
def test_qk_norm_rope_append(gpu_device, dtype, rank, rows, hq, hkv, norm):
    gen = torch.Generator().manual_seed(rows + hq + rank)
    n, D, ps = 2, 128, 16
    width = (hq + 2 * hkv) * D
    qkv = torch.randn((rows, width + 3 * n * rank), generator=gen).to(dtype).to(gpu_device)
    outs_w = (hq * D, hkv * D, hkv * D)
    mods = [_module(gen, rows, n, w, rank, dtype, gpu_device, qkv, width + j * n * rank)
            for j, w in enumerate(outs_w)]
    wq, wk = ((1 + 0.1 * torch.randn(D, generator=gen)).to(dtype).to(gpu_device) if norm else None for _ in range(2))
    pos = torch.randint(0, 40000, (rows,), generator=gen)
    pages = 40 if rows <= 600 else 130
    slots = torch.randperm(pages * ps, generator=gen)[:rows]
    page, off = slots // ps, slots % ps
    page[3], off[5] = -1, ps  # outside the pool: skipped
    ids = torch.ones(rows, dtype=torch.int32, device=gpu_device)
    results = []
    for j in range(2):
        cache = torch.zeros((pages, 2, ps, hkv, D), dtype=dtype, device=gpu_device)
        q = fused_ops.qk_norm_rope_append(
            qkv[:, :width], wq, wk, pos.to(gpu_device), page.to(gpu_device), off.to(gpu_device), cache,
            num_qo_heads=hq, num_kv_heads=hkv, head_dim=D, page_size=ps, rope_theta=1e6,
            lora=tuple(m[j] for m in mods), adapter_ids=ids)
        results.append((q, cache))
    torch.cuda.synchronize()
    for got, want in zip(*results):
        _close(got, want, dtype)
    assert ((results[0][1] != 0) == (results[1][1] != 0)).all()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rank", [8, 16])
@pytest.mark.parametrize("rows,hidden", [(320, 8), (321, 520), (1027, 4096), (323, 4088), (321, 1032)])
@pytest.mark.parametrize("chunk8", [False, True])
def test_add_rmsnorm_rows(gpu_device, dtype, rank, rows, hidden, chunk8):
    """Rows sharing B in registers vs a row per workgroup."""
    gen = torch.Generator().manual_seed(rows + hidden + rank)
    n = 2
    x = torch.randn((rows, hidden + n * rank), generator=gen).to(dtype).to(gpu_device)
    res = torch.randn((rows, hidden), generator=gen).to(dtype).to(gpu_device)
    w = (1 + 0.1 * torch.randn(hidden, generator=gen)).to(dtype).to(gpu_device)
    B = (torch.randn((n, hidden, rank), generator=gen) * 0.1).to(dtype).to(gpu_device)
    Bs = fused_ops.lora_b_chunk8(B) if chunk8 else B
    ids = torch.ones(rows, dtype=torch.int32, device=gpu_device)
    outs = []
    for a in (1, -1):
        r = res.clone()
        m = fused_ops.LoraUp(x, hidden, Bs, 2.0, a)
        outs.append((fused_ops.add_rmsnorm(r, x[:, :hidden], w, 1e-6, lora=m, adapter_ids=ids), r))
    torch.cuda.synchronize()
    for got, want in zip(*outs):
        _close(got, want, dtype)
