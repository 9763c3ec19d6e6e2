"""The K split of the GEMM on shuffled weights past 16 tokens, on the host: a
workgroup loads its first step before it looks at how many it has, so every
split of every K has at least one step, and together they are all of K."""

import numpy as np
import pytest

from pagelora_amd import _lib


@pytest.mark.parametrize("tokens", [33, 48, 64, 77, 128, 300])
def test_every_split_has_steps(tokens):
    lib = _lib.load()
    begin = np.zeros(9, dtype=np.int32)
    most = 0
    for n in (37, 1000, 2000, 4112, 6192):
        for k in range(64, 12800, 32):
            steps = k // 64
            splits = lib.pl_linear_shuffled_wide_splits(tokens, k, n, begin.ctypes.data)
            b = begin[:splits + 1]
            most = max(most, splits)
            assert b[0] == 0 and b[-1] == steps and (np.diff(b) >= 1).all(), (tokens, n, k, b)
            need = splits * tokens * -(-n // 16) * 16 * 4 if splits > 1 else 0
            assert lib.pl_linear_shuffled_wide_workspace_size(tokens, k, n) == need
    assert tokens > 128 or most == 8  # the widest split is among them
