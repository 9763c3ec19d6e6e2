"""DecoderWeights.logits past the decode GEMM's rows: every x that the library
GEMM takes -- column and row strides, shapes, rows at any alignment, gradients
-- with the lm_head stored row-major beside the shuffled copy, or shuffled
alone."""

import pytest
import torch
import torch.nn.functional as F

from pagelora_amd.decoder import DecoderConfig, DecoderWeights

pytestmark = pytest.mark.gpu

CFG = DecoderConfig(num_layers=1, hidden=256, num_qo_heads=8, num_kv_heads=2, head_dim=64, intermediate=512,
                    vocab=1000, lora_rank=16, lora_alpha=32.0)
ROWS = 70  # past both limits, 16 and 64


def _inputs(device):
    x = torch.randn((ROWS, 256), generator=torch.Generator().manual_seed(1)).to(device, torch.bfloat16)
    odd = torch.empty(ROWS * 260 + 3, dtype=x.dtype, device=device)[3:].view(ROWS, 260)[:, 1:257]
    return {
        "plain": x,
        "rows 4 bytes off": odd.copy_(x),
        "columns strided": x.t().contiguous().t(),
        "one row for all": x[:1].expand(ROWS, 256),
        "three dims": x.view(ROWS, 1, 256).expand(ROWS, 2, 256),
        "one dim": x[0],
    }


@pytest.mark.parametrize("keep_row_major", [False, True])
def test_any_x_past_the_decode_rows(gpu_device, keep_row_major):
    w = DecoderWeights(CFG, n_adapters=1, device=gpu_device, seed=3, keep_row_major=keep_row_major)
    head = w.lm_head.clone()
    for name, x in _inputs(gpu_device).items():
        print(f"[logits] {name}", flush=True)
        got, want = w.logits(x), F.linear(x.float(), head.float())
        assert got.shape == want.shape and got.dtype == torch.bfloat16, name
        # one rounding of the result, and the order of 256 fp32 sums
        assert ((got.float() - want).abs() <= 2.0**-8 * want.abs() + 1e-4).all(), name


def test_gradients_past_the_decode_rows(gpu_device):
    w = DecoderWeights(CFG, n_adapters=1, device=gpu_device, seed=3)
    x = _inputs(gpu_device)["plain"].clone().requires_grad_()
    w.logits(x).float().sum().backward()
    want = w.lm_head.float().sum(0).expand(ROWS, 256)
    # one rounding of the result, and the order of 1000 fp32 sums
    assert ((x.grad.float() - want).abs() <= 2.0**-8 * want.abs() + 1e-3).all()
