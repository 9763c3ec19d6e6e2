"""The prompt-size path of the LoRA delta (past 64 tokens, or inputs past the
decode path's width) vs the float64 oracle: tile edges, tokens sorted by
adapter, module widths and ranks that fill no whole chunk.

Bars: fp32 sums of the rank-r product on the oracle's rounded intermediate
(2e-3, as for the decode path) plus one rounding of the result."""

import numpy as np
import pytest
import torch

from oracle import lora as ol
from pagelora_amd.lora import lora_delta_groups_

pytestmark = pytest.mark.gpu


def _case(T, n, spec, dtype, out_dtype, gen, device):
    """Groups ``spec`` = [(in, [(out, rank), ...]), ...], outputs column views of one buffer per group."""
    groups, host = [], []
    for fin, modules in spec:
        x = torch.randn((T, fin), generator=gen).to(dtype)
        base = torch.randn((T, sum(o for o, _ in modules) + 8), generator=gen).to(out_dtype)
        packed, col, mods = base.to(device), 0, []
        for out, rank in modules:
            A = (torch.randn((n, rank, fin), generator=gen) * fin ** -0.5).to(dtype)
            B = (torch.randn((n, out, rank), generator=gen) * 0.05).to(dtype)
            mods.append((A.to(device), B.to(device), packed[:, col:col + out], 2.0))
            host.append((x, A, B, base[:, col:col + out].float().numpy(), packed[:, col:col + out]))
            col += out
        host.append((None, None, None, base[:, col:].float().numpy(), packed[:, col:]))
        groups.append((x.to(device), mods))
    return groups, host


@pytest.mark.parametrize("dtype,out_dtype", [(torch.bfloat16, torch.bfloat16), (torch.float16, torch.float16),
                                             (torch.bfloat16, torch.float32), (torch.float16, torch.bfloat16)])
@pytest.mark.parametrize("T,n,spec", [
    (65, 1, [(1000, [(264, 16), (8, 8), (64, 24)]), (32, [(72, 8)])]),
    (80, 2, [(512, [(256, 16), (512, 16)]), (264, [(40, 40)])]),
    (333, 7, [(4096, [(96, 16), (328, 16), (24, 16)])]),
    (129, 64, [(256, [(64, 128)]), (40, [(64, 8), (64, 72)])]),
    (20, 3, [(16640, [(64, 16)]), (64, [(64, 64), (8, 48)])]),
    (4096, 2, [(64, [(16, 16)])]),
])
def test_tiles_match_the_oracle(gpu_device, T, n, spec, dtype, out_dtype):
    gen = torch.Generator().manual_seed(T * 131 + n)
    groups, host = _case(T, n, spec, dtype, out_dtype, gen, gpu_device)
    # -1 and n: tokens without an adapter; the last adapter is rare
    ids = torch.randint(-1, n + 1, (T,), generator=gen, dtype=torch.int32)
    lora_delta_groups_(groups, ids.to(gpu_device))
    torch.cuda.synchronize()
    inter = "bf16" if dtype == torch.bfloat16 else "f16"
    rtol = {torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11, torch.float32: 0.0}[out_dtype]
    for x, A, B, base, got in host:
        want = base
        if x is not None:
            want = base + ol.multi_adapter_delta(x.float().numpy(), ids.tolist(), A.float().numpy(),
                                                 B.float().numpy(), 2.0, intermediate=inter)
        err = np.abs(got.float().cpu().numpy() - want)
        assert (err <= 2e-3 + rtol * np.abs(want)).all(), f"max err {err.max():.3e}"


def test_groups_in_sequence_where_one_reads_anothers_output(gpu_device):
    """The second group's input is the first one's output: the same as two calls."""
    gen = torch.Generator().manual_seed(3)
    T = 100
    x = torch.randn((T, 256), generator=gen).to(torch.bfloat16).to(gpu_device)

    def module(fin, out):
        return ((torch.randn((2, 16, fin), generator=gen) * fin ** -0.5).to(torch.bfloat16).to(gpu_device),
                (torch.randn((2, out, 16), generator=gen) * 0.2).to(torch.bfloat16).to(gpu_device))

    A0, B0 = module(256, 128)
    A1, B1 = module(128, 64)
    ids = (torch.arange(T, dtype=torch.int32) % 2).to(gpu_device)
    results = []
    for joined in (True, False):
        mid = torch.zeros((T, 128), dtype=torch.bfloat16, device=gpu_device)
        out = torch.zeros((T, 64), dtype=torch.bfloat16, device=gpu_device)
        g0, g1 = (x, [(A0, B0, mid, 1.0)]), (mid, [(A1, B1, out, 1.0)])
        if joined:
            lora_delta_groups_([g0, g1], ids)
        else:
            lora_delta_groups_([g0], ids)
            lora_delta_groups_([g1], ids)
        results.append((mid, out))
    torch.cuda.synchronize()
    assert torch.equal(results[0][0], results[1][0]) and torch.equal(results[0][1], results[1][1])
    assert results[0][1].abs().sum() > 0


def test_capture_with_the_general_path_s_workspace(gpu_device, monkeypatch):
    """A capture of many tokens with a workspace that holds the general path's
    partials but not the tiles' buffers takes the general path; one that holds
    neither is refused before anything is recorded."""
    from pagelora_amd import _lib, lora

    gen = torch.Generator().manual_seed(5)
    T, spec = 4096, [(64, [(16, 16)])] * 4
    groups, host = _case(T, 2, spec, torch.bfloat16, torch.bfloat16, gen, gpu_device)
    ids = torch.randint(-1, 2, (T,), generator=gen, dtype=torch.int32).to(gpu_device)
    descs = (_lib.LoraGroup * len(groups))()
    keep = [lora._module_structs(mods, x)[0] for x, mods in groups]

    def need():
        for d, (x, mods), arr in zip(descs, groups, keep):
            d.x, d.ldx, d.in_features, d.num_modules, d.modules = x.data_ptr(), x.stride(0), x.shape[1], len(mods), arr
        return _lib.load().pl_lora_delta_workspace_size(descs, len(groups), T, 2)

    tiled = need()
    for arr in keep:
        arr[0].out += 2  # an unaligned output: the general path's need (sizes only, nothing is read)
    general = need()
    assert general < tiled
    for size in (general, general - 256):
        monkeypatch.setitem(lora._DELTA_WS, gpu_device.index, torch.zeros(size, dtype=torch.uint8, device=gpu_device))
        graph = torch.cuda.CUDAGraph()
        refused = False
        with torch.cuda.graph(graph):
            try:
                lora_delta_groups_(groups, ids)
            except RuntimeError as e:
                refused = "sized before graph capture" in str(e)
        assert refused == (size < general)
        if refused:
            continue
        graph.replay()
        torch.cuda.synchronize()
        for x, A, B, base, got in host:
            want = base
            if x is not None:
                want = base + ol.multi_adapter_delta(x.float().numpy(), ids.tolist(), A.float().numpy(),
                                                     B.float().numpy(), 2.0, intermediate="bf16")
            err = np.abs(got.float().cpu().numpy() - want)
            assert (err <= 2e-3 + 2.0**-8 * np.abs(want)).all(), f"max err {err.max():.3e}"
