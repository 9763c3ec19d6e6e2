"""The LoRA delta's workspace when it grows: a captured graph holds the address
of the buffer of its time, so that buffer has to outlive the growth."""

import weakref

import torch

from pagelora_amd import lora


def test_outgrown_buffers_outlive_the_growth(monkeypatch):
    monkeypatch.setattr(lora, "_DELTA_WS", {})
    monkeypatch.setattr(lora, "_OUTGROWN_WS", [], raising=False)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    device = torch.device("cpu", 0)
    sizes, refs = [], []
    for nbytes in (1 << 20, (1 << 20) + 256, 3 << 20, 3 << 20, 9 << 20):
        ws = lora._delta_workspace(device, nbytes)
        assert ws.numel() >= nbytes and not ws.any()
        if not refs or refs[-1]() is not ws:
            refs.append(weakref.ref(ws))
            sizes.append(ws.numel())
        del ws
    assert all(r() is not None for r in refs)
    assert sum(sizes[:-1]) < sizes[-1]  # bounded by the buffer in use
