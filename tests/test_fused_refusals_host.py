"""What the fused element-wise entries refuse before any launch, at prompt
sizes too: a dtype code that they do not know.  Host checks only (the pointers
are never read)."""

import pytest

from pagelora_amd import _lib

PTR = 4096  # aligned, never dereferenced


def _module(width, rank=32):
    return _lib.LoraUp(PTR, 1024, 0, PTR, width, rank, 1.0, 0, 0)


@pytest.mark.parametrize("rows", [1, 24, 4096])
def test_silu_mul_lora_unknown_dtype(rows):
    mods = (_lib.LoraUp * 2)(_module(512), _module(512))
    status = _lib.load().pl_silu_mul_lora(PTR, 1024, mods, None, 1, PTR, 512, rows, 512, 7, None)
    assert status == _lib.PL_ERR_UNSUPPORTED, _lib.last_error()


@pytest.mark.parametrize("rows", [1, 4096])
def test_qk_norm_rope_append_lora_unknown_dtype(rows):
    hq, hkv, d = 4, 2, 128
    mods = (_lib.LoraUp * 3)(_module(hq * d), _module(hkv * d), _module(hkv * d))
    status = _lib.load().pl_qk_norm_rope_append_lora(
        PTR, 8 * d, None, mods, None, 1, PTR, PTR, PTR, PTR, PTR, PTR, PTR, PTR, 2 * 16 * hkv * d, hkv * d, d, 64, 16,
        rows, hq, hkv, d, PTR, 1e-6, 7, None)
    assert status == _lib.PL_ERR_UNSUPPORTED, _lib.last_error()
