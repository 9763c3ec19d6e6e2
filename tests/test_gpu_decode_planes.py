"""The probability planes of the decode wave for groups of 4 heads and more, vs
the float64 oracle: one row of few items, scores and V chosen so that what the
planes drop or add shows in the result."""

import math

import numpy as np
import pytest
import torch

from oracle import paged_decode as opd
from tests.gpu_cases import ragged_case
from tests.test_gpu_decode_matrix import _run

pytestmark = pytest.mark.gpu

DTYPES = [torch.bfloat16, torch.float16]
REL = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}


def _one_row(scores, v, group, dtype, device):
    """One row of ``group`` heads that all score token t ``scores[t]`` (in
    powers of two) and read V rows ``v`` [tokens, 128]."""
    n = len(scores)
    case = ragged_case(lens=[n], hq=group, hkv=1, head_dim=128, page_size=16, dtype=dtype, device="cpu", seed=1)
    # q = 8 in dim 0, K = the score there: q . K / sqrt(128) * log2(e) = score
    q, cache = torch.zeros_like(case["q"]), torch.zeros_like(case["cache"])
    q[:, :, 0] = 8.0
    pages = case["indices"].long()
    k = torch.zeros((len(pages) * 16, 128))
    k[:n, 0] = torch.as_tensor(scores, dtype=torch.float32) * (math.sqrt(128) / 8.0 / math.log2(math.e))
    vv = torch.zeros((len(pages) * 16, 128))
    vv[:n] = torch.as_tensor(v, dtype=torch.float32)
    cache[pages, 0, :, 0] = k.reshape(-1, 16, 128).to(dtype)
    cache[pages, 1, :, 0] = vv.reshape(-1, 16, 128).to(dtype)
    case["q_host"], case["cache_host"] = q, cache
    case["q"], case["cache"] = q.to(device), cache.to(device)
    return case


def _want(case):
    return opd.paged_decode(case["q_host"].float().numpy(), case["cache_host"].float().numpy(),
                            case["indptr"].numpy(), case["indices"].numpy(), case["last"].numpy())[0]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("group", [4, 7])
@pytest.mark.parametrize("n", [2048, 16384])
@pytest.mark.parametrize("below", [30.0, 60.0])
def test_tokens_far_below_the_maximum_add_nothing(gpu_device, dtype, group, n, below):
    """One token (an attention sink with a small V) far above n others with V =
    1, in one item: the others weigh n 2^-below.  Bar: one rounding of the
    result, and 2^-36 of V for every token."""
    scores = np.zeros(n)
    scores[0] = below
    v = np.ones((n, 128))
    v[0] = 0.05
    case = _one_row(scores, v, group, dtype, gpu_device)
    got = _run(case, group, 1, 16, gpu_device, target_waves=1)
    want = _want(case)
    err = np.abs(got - want)
    assert (err <= REL[dtype] * np.abs(want) + n * 2.0**-36).all(), f"max err {err.max():.3e}"


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("group", [2, 4, 7])
@pytest.mark.parametrize("first", [True, False])
def test_infinite_v_at_a_probability_of_zero_is_nan(gpu_device, dtype, group, first):
    """A token 400 powers of two below the maximum has probability 0 in fp32:
    an infinite V there gives 0 * inf = NaN in its dim for every group size
    (2 heads: the vector wave), whichever of the two tokens comes first, and
    nothing in the other dims."""
    n = 100
    scores = np.zeros(n)
    scores[0 if first else 90] = 400.0
    v = np.random.default_rng(2).standard_normal((n, 128))
    v[37, 9] = np.inf
    case = _one_row(scores, v, group, dtype, gpu_device)
    got = _run(case, group, 1, 16, gpu_device, target_waves=1)
    case["cache_host"][case["cache_host"].isinf()] = 0.0
    want = _want(case)
    assert np.isnan(got[:, :, 9]).all()
    rest = np.arange(128) != 9
    assert (np.abs(got - want)[:, :, rest] <= REL[dtype] * np.abs(want[:, :, rest]) + 1e-6).all()


def _cancelling_error(group, dtype, device, seed):
    """The relative error of a row whose three terms nearly cancel."""
    rng = np.random.default_rng(seed)
    scores = np.array([0.0, -rng.uniform(0.1, 0.9), -rng.uniform(1.1, 1.9)])
    v = np.zeros((3, 128))
    case = _one_row(scores, v, group, dtype, device)
    page = int(case["indices"][0])
    k0 = case["cache_host"][page, 0, :3, 0, 0].double().numpy()
    p = np.exp((k0 - k0.max()) * 8.0 / math.sqrt(128))
    cut = lambda x: torch.as_tensor(x, dtype=torch.float64).to(dtype).double().numpy()  # noqa: E731
    v[1] = cut(rng.uniform(1, 2, 128))
    v[0] = cut(-p[1] * v[1] / p[0])
    left = p[0] * v[0] + p[1] * v[1]
    v[2] = cut(-(left - np.sign(left) * 2.0**-12) / p[2])  # takes the rest down to about 2^-12 of the terms
    for key in ("cache", "cache_host"):
        case[key][page, 1, :3, 0] = torch.as_tensor(v).to(dtype).to(case[key].device)
    got, want = _run(case, group, 1, 16, device, target_waves=1), _want(case)
    return np.linalg.norm(got - want) / np.linalg.norm(want)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("group", [4, 7])
def test_probabilities_keep_their_32_bits(gpu_device, dtype, group):
    """Terms that cancel down to 2^-12 of themselves: a probability of 16 bits
    leaves an error of up to 2^-5 of the result, one of 22 bits 2^-11.  The
    vector wave (2 heads; fp32 probabilities, and the same scores, of which
    only one dim is not zero) is the measure; beyond its error 2^-13 for the
    order of the sums (2^-24 of the terms, twice)."""
    errs = [(_cancelling_error(group, dtype, gpu_device, s), _cancelling_error(2, dtype, gpu_device, s))
            for s in range(8)]
    print(f"[planes] {dtype} group {group}: worst " + ", vector wave ".join(f"{max(e):.2e}" for e in zip(*errs)),
          flush=True)
    assert all(a <= b + 2.0**-13 for a, b in errs), errs
