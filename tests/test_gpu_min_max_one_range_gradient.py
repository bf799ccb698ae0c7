"""MinMaxQuantize's input gradient under one range for the whole tensor, whose bounds every thread of the masking launch
forms itself: sizes around a vector, a block and a tile, addresses that are and are not 16-byte aligned, overwriting and
accumulating, non-finite inputs.  The result is exact: dy where the nudged range holds x, 0 elsewhere."""
import numpy as np
import pytest
import torch

from nnabla_amd import kernels
from util import to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [1, 3, 4, 1023, 4096, 4097, 70001])
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("accumulate", [False, True])
def test_mask_of_one_range(size, shift, accumulate):
    kernels.init(0)
    rng = np.random.RandomState(size)
    x = (rng.randn(size) * 2).astype(np.float32)
    dy = rng.randn(size).astype(np.float32)
    lo, hi, levels = np.float32(-1.3), np.float32(1.7), np.float32(255)
    scale = np.float32((hi - lo) / levels)
    zero = np.float32(0) - lo / scale
    nudged = np.float32(np.floor(zero + np.float32(0.5)))
    m, M = np.float32((0 - nudged) * scale), np.float32((levels - nudged) * scale)
    x[:min(size, 6)] = np.array([np.nan, np.inf, -np.inf, m, M, 0], np.float32)[:size]

    def dev(v):
        t = torch.empty(size + shift, device="cuda")
        t[shift:] = torch.from_numpy(v)
        return t[shift:]

    one = lambda v: torch.full((1,), float(v), device="cuda")
    old = rng.randn(size).astype(np.float32)
    want = np.where((x >= m) & (x <= M), dy, dy * np.float32(0))
    if accumulate:
        want = want + old
    dx, _, _ = kernels.min_max_quantize_backward(dev(dy), dev(x), one(lo), one(hi), one(0), one(levels), one(scale),
                                                 x_min_max=True, dx=dev(old) if accumulate else None, want_min=False,
                                                 want_max=False)
    assert np.array_equal(to_np(dx), want)
