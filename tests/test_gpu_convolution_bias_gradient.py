"""The bias gradient taken along by the weight gradient's product (csrc/kernels/conv_dw.hip): planes below and above a
block's width, several samples side by side, groups, strides, sums added to what is there, non-finite values, and the pass
of its own where the weight gradient is not wanted, against float64."""
import numpy as np
import pytest
import torch

from nnabla_amd import kernels
from util import to_np

pytestmark = pytest.mark.gpu

# batch, channels, height, width, maps, kernel, stride, group
CASES = [(1, 16, 7, 7, 16, 3, 1, 1), (37, 33, 5, 9, 70, 3, 1, 1), (5, 64, 31, 33, 300, 3, 2, 1), (3, 96, 28, 28, 64, 1, 1, 2),
         (130, 40, 14, 14, 257, 5, 1, 1)]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("binary", [False, True])
def test_against_float64(case, binary):
    kernels.init(0)
    B, C, H, W, O, k, s, g = case
    gen = torch.Generator(device="cuda").manual_seed(B + C + O)
    oh, ow = (H + 2 * (k // 2) - k) // s + 1, (W + 2 * (k // 2) - k) // s + 1
    x = torch.randn(B, C, H, W, generator=gen, device="cuda")
    w = torch.randn(O, C // g, k, k, generator=gen, device="cuda")
    dy = torch.randn(B, O, oh, ow, generator=gen, device="cuda") + 0.25
    geo = ((k // 2,) * 2, (s, s), (1, 1), g)

    def grads(**kw):
        if binary:
            return kernels.binary_convolution_backward(dy, x, w, None, None, *geo, **kw)
        return kernels.convolution_backward(dy, x, w, *geo, **kw)

    ref, terms = dy.double().sum((0, 2, 3)), dy.double().abs().sum((0, 2, 3))
    # chains of at most a slice's samples of one thread, six steps over the lanes, four wavefronts, the slices in double
    bound = terms * 2.0 ** -24 * (B * (oh * ow // 1024 + 1) + 12) + ref.abs() * 2.0 ** -23
    dx, dw, db = grads()
    assert bool(((db.double() - ref).abs() <= bound).all())
    alone = grads(want=(False, False, True))[2]
    assert bool(((alone.double() - ref).abs() <= bound).all())
    assert torch.equal(grads(want=(False, True, False))[1], dw)
    old = torch.full((O,), 3.0, device="cuda")
    grads(db=old, want=(False, True, True))
    assert bool(((old.double() - (ref + 3)).abs() <= bound + 2.0 ** -22 * (ref.abs() + 3)).all())
    dy[0, 1, 0, 0], dy[B - 1, O - 1, oh - 1, ow - 1] = float("inf"), float("nan")
    got = to_np(grads()[2])
    assert got[1] == np.inf and np.isnan(got[O - 1])
    rest = [o for o in range(O) if o not in (1, O - 1)]
    assert np.array_equal(got[rest], to_np(db)[rest])
