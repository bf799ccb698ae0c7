"""Blocks of eight wavefronts of the real-weight convolution (csrc/kernels/conv_real.hip), which geometries of at most one
block per CU take: chunks of 32 and 64 channels with channels left over, taps that are no multiple of the wavefronts,
and windows that are recomputed, forward and input gradient against float64."""
import numpy as np
import pytest
import torch  # noqa: F401  (the device library's runtime)

from nnabla_amd import kernels
from test_gpu_convolution_real_weights import _bound, _conv64, _data, _grad64, _run

pytestmark = pytest.mark.gpu

# batch, channels, height, width, maps, kernel, pad, stride, group
CASES = [(16, 130, 28, 28, 70, (3, 3), (1, 1), 2, 1),   # chunks of 32, two channels in the last
         (128, 300, 7, 7, 65, (3, 3), (1, 1), 1, 1),    # of 64, 44 in the last; the gradient: one channel in the last
         (64, 512, 9, 9, 40, (1, 1), (0, 0), 1, 1),     # a tap: most wavefronts have no step
         (24, 200, 14, 14, 100, (3, 3), (1, 1), 2, 1)]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("bad", [False, True])
def test_against_float64(case, bad):
    kernels.init(0)
    B, C, H, W, O, k, p, s, g = case
    x, w, b, dy = _data(case)
    if bad:  # a window of tiny values, one with an infinity
        x[0, :, :4, :4] *= np.float32(1e-33)
        x[B - 1, C - 1, H - 1, W - 1] = np.inf
        dy[0, :, :2, :2] *= np.float32(1e-33)
    y, dx = _run(case, x, w, b, dy)
    with np.errstate(invalid="ignore"):
        ref, terms = _conv64(case, x, w, b), _conv64(case, np.abs(x), np.abs(w))
    fin = np.isfinite(ref)
    assert np.array_equal(np.isfinite(y), fin) and fin.sum() > 0.9 * ref.size
    bound = _bound(terms, C // g * k[0] * k[1]) + 2.0 ** -23 * np.abs(ref) + 2.0 ** -24 * 4
    assert (np.abs(y - ref)[fin] <= bound[fin]).all()
    ref = _grad64(case, w, dy)
    bound = _bound(_grad64(case, np.abs(w), np.abs(dy)), O // g * k[0] * k[1]) + 2.0 ** -23 * np.abs(ref) + 2.0 ** -149
    assert (np.abs(dx - ref) <= bound).all()
