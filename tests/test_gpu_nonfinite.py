"""asa_check_nonfinite (the reference-order calls' non-finite check) against
torch.isnan / torch.isinf: sizes around a lane's 16 bytes and a block's share,
each type, a single bad element at the start, the end and inside."""
import numpy as np
import pytest
import torch

import splash_attention as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n", [1, 3, 7, 8, 9, 2047, 4096, 4099, 5_000_011])
def test_nonfinite_flags(dev, dtype, n):
    print(f"[nonfinite] {dtype} n={n}", flush=True)
    big = torch.finfo(dtype).max
    base = torch.full((n,), big, dtype=dtype, device=dev)  # the largest finite value is no infinity
    base[::2] = -0.0
    assert sa.ops.nonfinite([base]) == [False]
    for at in sorted({0, n // 2, n - 1}):
        for bad in (float("nan"), float("inf"), float("-inf")):
            t = base.clone()
            t[at] = bad
            assert sa.ops.nonfinite([base, t]) == [False, True]
            assert sa.ops.nonfinite([t, base, base]) == [True, False, False]


def test_nonfinite_views_and_host_tensors_take_the_full_check(dev):
    t = torch.zeros(8, 9, device=dev)
    assert sa.ops.nonfinite([t[:, :8]]) == [True]   # not contiguous
    assert sa.ops.nonfinite([t.cpu()]) == [True]
    flat = torch.zeros(65, device=dev)
    assert sa.ops.nonfinite([flat[1:]]) == [True]   # not 16-byte aligned
