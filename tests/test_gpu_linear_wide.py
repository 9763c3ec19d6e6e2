"""The GEMM on shuffled weights past 16 tokens (pl_linear_shuffled_wide) vs
the oracle's linear term in float64: one rounding of the output (2^-8
relative for bf16, 2^-11 for fp16) plus the fp32 accumulation's error, 2e-3
max-abs, as for pl_linear_shuffled."""

import numpy as np
import pytest
import torch

from pagelora_amd import _lib
from pagelora_amd.linear import ShuffledWeight, linear_shuffled, linear_shuffled_wide

pytestmark = pytest.mark.gpu

REL = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}


# Edges of the token tiles (32 .. 256 rows), of the column tiles (128 .. 384)
# and of the K steps: 64-wide ones fewer than the buffers in flight, K not a
# multiple of 64, K split over workgroups (few tokens, wide
# K), the tile shapes of many tokens.
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tokens,n,k", [
    (17, 4112, 4096), (32, 1000, 96), (33, 6192, 64), (48, 24608, 192), (49, 37, 320), (64, 4112, 12288),
    (65, 1000, 4096), (77, 4112, 4096), (81, 24608, 128), (100, 130, 224), (129, 2064, 4096), (191, 6192, 2048),
    (257, 4112, 1024), (513, 24608, 256), (1000, 6192, 448), (2111, 4112, 320), (2112, 24608, 128),
    (2200, 6192, 256), (2113, 24600, 64)])
def test_linear_wide_vs_oracle(gpu_device, dtype, tokens, n, k):
    print(f"[wide gemm] {tokens} x {n} x {k} {dtype}", flush=True)
    g = torch.Generator(device=gpu_device).manual_seed(n + k + tokens)
    x = torch.randn((tokens, k), generator=g, device=gpu_device).to(dtype)
    w = (torch.randn((n, k), generator=g, device=gpu_device) * k ** -0.5).to(dtype)
    bias = (torch.randn(n, generator=g, device=gpu_device) * 0.1).to(dtype) if tokens % 2 else None
    sw = ShuffledWeight(w)
    wide = torch.full((tokens, n + 9), 7.0, dtype=dtype, device=gpu_device)  # odd row stride, neighbours kept
    out = linear_shuffled_wide(x, sw, bias, out=wide[:, :n])
    whole = linear_shuffled_wide(x, sw, bias)
    torch.cuda.synchronize()
    assert torch.equal(out, whole) and (wide[:, n:] == 7.0).all()
    want = x.double().cpu().numpy() @ w.double().cpu().numpy().T
    if bias is not None:
        want = want + bias.double().cpu().numpy()
    err = np.abs(whole.float().cpu().numpy() - want)
    assert (err <= 2e-3 + REL[dtype] * np.abs(want)).all(), f"max err {err.max():.3e}"


# K steps that their splits do not divide evenly (33, 42, 65 by 8, 55 and 27 by 4, 69 by 2)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tokens,n,k,splits", [(65, 1000, 2112, 8), (65, 1000, 2688, 8), (65, 1000, 4160, 8),
                                               (33, 4112, 3520, 4), (77, 4096, 1728, 4), (77, 8208, 4416, 2)])
def test_uneven_splits(gpu_device, dtype, tokens, n, k, splits):
    assert _lib.load().pl_linear_shuffled_wide_splits(tokens, k, n, None) == splits
    test_linear_wide_vs_oracle(gpu_device, dtype, tokens, n, k)


# K an odd multiple of 32: the tile kernel's last half step, in one piece and
# in the last of several, and a K below one step
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("tokens,n,k", [(33, 4112, 96), (65, 1000, 2080), (77, 8208, 4128), (200, 12320, 160),
                                        (48, 24608, 1056), (2112, 6192, 96), (1000, 37, 3488), (2050, 2064, 32),
                                        (40, 4112, 32)])
def test_last_half_step(gpu_device, dtype, tokens, n, k):
    test_linear_wide_vs_oracle(gpu_device, dtype, tokens, n, k)


# Up to 64 tokens, either side of where the 16-token kernel takes over: one
# round of workgroups, two that share weights, an unsplit product of few steps
@pytest.mark.parametrize("tokens,n,k", [(18, 2048, 160), (18, 2064, 160), (32, 2040, 4704), (33, 1360, 96),
                                        (33, 1376, 96), (64, 2048, 352), (64, 2064, 352), (64, 1000, 1024),
                                        (40, 8192, 1280), (33, 4096, 1600), (56, 2300, 3072)])
def test_few_columns(gpu_device, tokens, n, k):
    test_linear_wide_vs_oracle(gpu_device, torch.bfloat16, tokens, n, k)


def test_strided_x_without_workspace(gpu_device):
    """x as a column slice of a wider buffer; no workspace: the same product
    with its K sums in one piece."""
    g = torch.Generator(device=gpu_device).manual_seed(5)
    big = torch.randn((77, 4096 + 64), generator=g, device=gpu_device).to(torch.bfloat16)
    w = (torch.randn((4112, 4096), generator=g, device=gpu_device) * 0.02).to(torch.bfloat16)
    sw, lib = ShuffledWeight(w), _lib.load()
    x = big[:, 64:]
    assert lib.pl_linear_shuffled_wide_workspace_size(77, 4096, 4112) > 0
    out = torch.empty((77, 4112), dtype=torch.bfloat16, device=gpu_device)
    _lib.check(lib.pl_linear_shuffled_wide(x.data_ptr(), x.stride(0), 77, 4096, sw.data.data_ptr(), 4112, None,
                                           out.data_ptr(), 4112, None, 0, _lib.dtype_code(x.dtype),
                                           _lib.stream_handle(x.device)), "pl_linear_shuffled_wide")
    split = linear_shuffled_wide(x, sw)
    torch.cuda.synchronize()
    want = x.double().cpu().numpy() @ w.double().cpu().numpy().T
    for got in (out, split):
        err = np.abs(got.float().cpu().numpy() - want)
        assert (err <= 2e-3 + 2.0**-8 * np.abs(want)).all(), f"max err {err.max():.3e}"


@pytest.mark.parametrize("tokens", [17, 64, 70])
def test_rows_far_apart(gpu_device, tokens):
    """A row stride of 2^22 elements, past the tile kernels' 32-bit offsets:
    the same product, by the 16-token kernel."""
    k, n = 96, 40
    g = torch.Generator(device=gpu_device).manual_seed(tokens)
    x = torch.empty(((tokens - 1) << 22) + k, dtype=torch.bfloat16, device=gpu_device).as_strided(
        (tokens, k), (1 << 22, 1))
    x.copy_(torch.randn((tokens, k), generator=g, device=gpu_device))
    w = (torch.randn((n, k), generator=g, device=gpu_device) * k ** -0.5).to(torch.bfloat16)
    sw = ShuffledWeight(w)
    want = x.double().cpu().numpy() @ w.double().cpu().numpy().T
    for call in (linear_shuffled_wide, linear_shuffled)[: 2 if tokens <= 64 else 1]:
        err = np.abs(call(x, sw).float().cpu().numpy() - want)
        assert (err <= 2e-3 + 2.0**-8 * np.abs(want)).all(), f"max err {err.max():.3e}"
