"""The split-range prefill kernel (head_dim 128, page sizes of a multiple of 4)
vs the float64 oracle where it can go wrong: 64-token tile and 128-row item
edges, kv ranges cut into parts, GQA groups that straddle items, strided q and
out, and junk in the pages' unused slots.  Bars as in test_gpu_prefill."""

import pytest
import torch

from tests.test_gpu_prefill import _backend, _case, _check, _oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("page_size", [4, 12, 16, 64])
@pytest.mark.parametrize("heads,qo_lens,kv_lens,causal", [
    ((2, 2), [1, 63, 64, 65], [64, 63, 128, 4097], True),      # a part per few tiles beside short requests
    ((7, 1), [19, 0, 40], [2100, 5, 1025], True),              # groups of 7 across 16- and 128-row edges
    ((8, 2), [3, 130], [1500, 300], False),
    ((4, 4), [300], [300], True),
])
def test_edges_vs_oracle(gpu_device, dtype, page_size, heads, qo_lens, kv_lens, causal):
    hq, hkv = heads
    case = _case(qo_lens, kv_lens, hq, hkv, 128, page_size, dtype, gpu_device, seed=hq + page_size)
    be = _backend(case, hq, hkv, 128, page_size, gpu_device, causal)
    assert be._prefill_plan["split"]
    # what lies past a request's last token in its last page is no part of the result
    cache, ip, ind, last = case["cache"].clone(), case["indptr"], case["indices"], case["last"]
    for r in range(len(kv_lens)):
        cache[ind[ip[r + 1] - 1].item(), :, last[r].item():] = float("nan")
    out = torch.empty((case["q"].shape[0], hq + 1, 128), dtype=dtype, device=gpu_device)[:, 1:]
    q = torch.empty_like(out)
    q.copy_(case["q"])
    be.run_prefill_into(q, cache, out)
    torch.cuda.synchronize()
    _check(out, _oracle(case, causal), dtype)


def test_long_range_is_cut(gpu_device):
    """77 queries behind 9000 tokens: the kv range is cut, and its parts merge to the oracle's result."""
    case = _case([77], [9077], 8, 2, 128, 16, torch.float16, gpu_device, seed=1)
    be = _backend(case, 8, 2, 128, 16, gpu_device)
    assert be._prefill_plan["num_merges"] > 0
    out = be.run_prefill(case["q"], case["cache"])
    torch.cuda.synchronize()
    _check(out, _oracle(case), torch.float16)


# the merge takes 64 parts a pass and eight loads at a time
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads,kv_len,parts", [((7, 1), 20002, 79), ((28, 4), 32002, 126), ((2, 2), 16385, 65)])
def test_more_parts_than_a_pass(gpu_device, dtype, heads, kv_len, parts):
    """Two queries behind a long prefix: one row item in more than 64 parts."""
    case = _case([2], [kv_len], *heads, 128, 16, dtype, gpu_device, seed=parts)
    be = _backend(case, *heads, 128, 16, gpu_device)
    plan = be._prefill_plan
    records = plan["tables"][-1].view(-1, 8).cpu()
    assert plan["num_items"] == parts and records[plan["num_items"]:, 6].tolist() == [parts]
    out = be.run_prefill(case["q"], case["cache"])
    torch.cuda.synchronize()
    _check(out, _oracle(case), dtype)


# either side of where the 64-row kernel takes short sequences
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("heads,qo_lens,kv_lens,split", [
    ((4, 1), [1], [1], False), ((7, 1), [64, 17], [256, 17], False), ((7, 1), [64, 17], [257, 17], True),
    ((8, 8), [128] * 16, [128] * 16, False),   # 256 workgroups
    ((8, 8), [128] * 17, [129] * 17, True),    # 272 of three tiles
    ((32, 32), [17] * 20, [17] * 20, False),   # 640, half of the 128-row items padding
    ((32, 32), [128] * 9, [128] * 9, True),
])
def test_short_sequences(gpu_device, dtype, heads, qo_lens, kv_lens, split):
    case = _case(qo_lens, kv_lens, *heads, 128, 16, dtype, gpu_device, seed=len(qo_lens))
    be = _backend(case, *heads, 128, 16, gpu_device)
    assert be._prefill_plan["split"] == split
    out = be.run_prefill(case["q"], case["cache"])
    torch.cuda.synchronize()
    _check(out, _oracle(case), dtype)


@pytest.mark.parametrize("scale", [-0.05, 0.0])
def test_scale_sign(gpu_device, scale):
    """A negative or zero softmax scale: the same as the 64-row kernel on pages of 2 tokens."""
    case = _case([50, 3], [200, 400], 4, 2, 128, 16, torch.bfloat16, gpu_device, seed=2)
    be = _backend(case, 4, 2, 128, 16, gpu_device)
    assert be._prefill_plan["split"]
    be.sm_scale = scale
    out = be.run_prefill(case["q"], case["cache"])
    pages = case["indices"].long()
    small = case["cache"].cpu()[pages]  # [pages, 2, 16, Hkv, D] -> pages of 2 tokens
    small = small.reshape(len(pages), 2, 8, 2, 2, 128).transpose(1, 2).reshape(-1, 2, 2, 2, 128).contiguous()
    from pagelora_amd.attention_backend import PagedDecodeAttention

    ref = PagedDecodeAttention(device=gpu_device, workspace_mb=8, num_qo_heads=4, num_kv_heads=2, head_dim=128,
                               page_size=2)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32)  # noqa: E731
    # 200 tokens are 13 pages of 16, the last of 8; 400 are 25 whole ones
    order = torch.cat([torch.arange(100), torch.arange(104, 304)]).to(torch.int32)
    ref.plan_prefill(qo_indptr=i32([0, 50, 53]), paged_kv_indptr=i32([0, 100, 300]), paged_kv_indices=order,
                     paged_kv_last_page_len=i32([2, 2]))
    assert not ref._prefill_plan["split"]
    ref.sm_scale = scale
    want = ref.run_prefill(case["q"], small.to(gpu_device))
    torch.cuda.synchronize()
    _check(out, want.float().cpu().numpy(), torch.bfloat16)


@pytest.mark.parametrize("wait", [True, False])
def test_run_on_another_stream_follows_the_plan(gpu_device, wait):
    """A run on a stream of its own, right after the plan and behind pending
    work on the planning stream, reads the plan's tables, and a later plan's
    upload does not disturb it: where the plan waits for its upload
    (plan_prefill) and where it does not (the decoder's prefill)."""
    cases = [_case([77], [9077], 8, 2, 128, 16, torch.bfloat16, gpu_device, seed=s) for s in (1, 2)]
    want = []
    for c in cases:
        want.append(_backend(c, 8, 2, 128, 16, gpu_device).run_prefill(c["q"], c["cache"]))
    be = _backend(cases[0], 8, 2, 128, 16, gpu_device)
    torch.cuda.synchronize()
    side, got = torch.cuda.Stream(), []
    big = torch.randn((4096, 4096), device=gpu_device)
    for c in cases:
        big = (big @ big).clamp_(-1, 1)  # the planning stream is busy when the upload is enqueued
        be._plan_prefill(c["qo_indptr"], c["indptr"], c["indices"], c["last"], wait=wait)
        with torch.cuda.stream(side):
            got.append(be.run_prefill(c["q"], c["cache"]))
    torch.cuda.synchronize()
    assert all(torch.equal(a, b) for a, b in zip(got, want))


def test_capture_right_after_the_plan(gpu_device):
    """plan_prefill has uploaded its tables when it returns: a capture begun
    without a synchronization, and replayed on a stream that waits for nothing,
    reads them."""
    case = _case([77], [9077], 8, 2, 128, 16, torch.bfloat16, gpu_device, seed=1)
    want = _backend(case, 8, 2, 128, 16, gpu_device).run_prefill(case["q"], case["cache"])
    be = _backend(case, 8, 2, 128, 16, gpu_device)
    big, side, graph = torch.randn((4096, 4096), device=gpu_device), torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    big = (big @ big).clamp_(-1, 1)  # the planning stream is busy when the upload is enqueued
    be.plan_prefill(qo_indptr=case["qo_indptr"], paged_kv_indptr=case["indptr"], paged_kv_indices=case["indices"],
                    paged_kv_last_page_len=case["last"])
    assert be._prefill_plan["ready"] is None
    with torch.cuda.stream(side):
        graph.capture_begin()
        got = be.run_prefill(case["q"], case["cache"])
        graph.capture_end()
        for _ in range(3):
            got.zero_()
            graph.replay()
            side.synchronize()
            assert torch.equal(got, want)
