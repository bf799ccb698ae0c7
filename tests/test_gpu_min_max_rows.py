"""MinMaxQuantize with a range per channel over rows of any length and alignment (a wavefront or a block per row,
csrc/kernels/quantize.hip and quantize_backward.hip), against the oracle: lengths at the edges of a wavefront's and a
block's accesses, channels that do not fill a block's four rows, arrays that start off a 16-byte boundary."""
import numpy as np
import pytest
import torch

import oracle
from nnabla_amd import kernels
from util import bits_equal, to_np

pytestmark = pytest.mark.gpu


def _at(a, offset):
    """On the device, `offset` elements past a 16-byte boundary."""
    flat = torch.empty(a.size + 4, device="cuda")
    v = flat[offset:offset + a.size].view(a.shape)
    v.copy_(torch.from_numpy(a))
    return v


@pytest.mark.parametrize("batch,channels,length", [(1, 2, 256), (3, 5, 257), (2, 7, 729), (1, 3, 1023), (5, 3, 1025), (2, 2, 2047),
                                                   (3, 2, 2048), (1, 3, 2049), (2, 3, 3025), (1, 2, 9001)])
@pytest.mark.parametrize("offset", [0, 1])
def test_rows(batch, channels, length, offset):
    kernels.init(0)
    rng = np.random.RandomState(length + batch)
    shape, per = (batch, channels, length), (1, channels, 1)
    x, dy, odx = ((rng.randn(*shape) * s).astype(np.float32) for s in (3.0, 1.0, 1.0))
    qmin = (-2.0 - 0.1 * rng.rand(*per)).astype(np.float32)
    qmax = (2.5 + 0.1 * rng.rand(*per)).astype(np.float32)
    lmin, lmax = np.zeros(per, np.float32), np.full(per, 255.0, np.float32)
    ry, rmn, rmx, rscale = oracle.min_max_quantize(x, qmin, qmax, lmin, lmax, 0.999, False, False, 0.01)
    rdx, gmin, gmax = oracle.min_max_quantize_backward(dy, x, rmn, rmx, lmin, lmax, rscale, True, False, False)
    r = [torch.from_numpy(v.copy()).cuda() for v in (qmin, qmax, lmin, lmax)]
    xd, dyd = _at(x, offset), _at(dy, offset)
    y, scale = kernels.min_max_quantize(xd, *r)
    assert bits_equal(to_np(y), ry) and bits_equal(to_np(scale), rscale)
    dx, dmin, dmax = kernels.min_max_quantize_backward(dyd, xd, *r, scale, True)
    assert bits_equal(to_np(dx), rdx)
    total = np.abs(dy).astype(np.float64).sum(axis=(0, 2), keepdims=True)
    # fp32 sums of up to 9001 terms in runs of a lane's few and then a tree: well below 2^-20 of the sum of magnitudes
    for got, ref in ((dmin, gmin), (dmax, gmax)):
        assert (np.abs(to_np(got) - ref.astype(np.float64)) <= 2e-6 * total).all()
    old = _at(odx, offset)
    kernels.min_max_quantize_backward(dyd, xd, *r, scale, True, dx=old, want_min=False, want_max=False)
    rdx2, _, _ = oracle.min_max_quantize_backward(dy, x, rmn, rmx, lmin, lmax, rscale, True, False, False, dx=odx.copy())
    assert bits_equal(to_np(old), rdx2)
