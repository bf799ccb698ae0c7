"""Where the convolution kernels take a block's positions apart (short_divide, the extent of a slab, buffers that end with
the group's last channel): maps one position wide or high, lines as long as a tile and one off, three axes whose maps end
inside a tile, padding so wide that a line's first window starts before the end of the line above -- against float64.

Bounds: binary, x rounded to 2^-30 of the largest magnitude under a block's windows and two roundings of the result; real,
sums of n terms in fp32 one after the other at the worst.
"""
import numpy as np
import pytest
import torch
import torch.nn.functional as TF

from nnabla_amd import kernels
from util import to_np

pytestmark = pytest.mark.gpu

# x shape, maps, kernel, pad, stride
CASES = [
    ((2, 32, 300, 1), 64, (3, 1), (1, 0), (1, 1)), ((2, 32, 1, 300), 33, (1, 3), (0, 1), (1, 1)),
    ((1, 48, 9, 127), 64, (3, 3), (1, 1), (1, 1)), ((1, 48, 9, 128), 64, (3, 3), (1, 1), (1, 1)),
    ((1, 48, 9, 129), 64, (3, 3), (1, 1), (1, 1)), ((3, 64, 11, 7), 96, (3, 5), (4, 9), (1, 1)),
    ((2, 256, 5, 3), 256, (3, 3), (3, 6), (1, 1)), ((2, 256, 13, 13), 250, (3, 3), (1, 1), (3, 2)),
    ((2, 32, 5, 3, 4), 70, (3, 3, 3), (1, 1, 1), (1, 1, 1)), ((3, 128, 4, 6, 5), 256, (1, 3, 3), (0, 2, 4), (1, 1, 1)),
    ((2, 24, 6, 5, 9), 40, (2, 3, 2), (0, 1, 3), (2, 1, 2)),
]


@pytest.mark.parametrize("xs,O,k,pad,stride", CASES)
def test_binary_and_real_weights_against_float64(xs, O, k, pad, stride):
    kernels.init(0)
    rng = np.random.RandomState(O + xs[1])
    x = torch.from_numpy(rng.randn(*xs).astype(np.float32))
    w = torch.from_numpy(rng.randn(O, xs[1], *k).astype(np.float32))
    conv = {2: TF.conv2d, 3: TF.conv3d}[len(k)]
    n, dil = int(np.prod(w.shape[1:])), (1,) * len(k)
    signs = torch.where(w < 0, -1.0, 1.0).double()
    ref = conv(x.double(), signs, None, stride, pad).numpy()
    y, _ = kernels.binary_connect_convolution(x.cuda(), w.cuda(), None, pad, stride, dil, 1)
    assert (np.abs(to_np(y) - ref) <= n * 2.0 ** -30 * float(x.abs().max()) + 2.0 ** -23 * np.abs(ref)).all()
    I = torch.zeros(w.shape, dtype=torch.int32, device="cuda")
    yr = kernels.inq_convolution(x.cuda(), w.cuda(), I, w.cuda(), I.clone(), None, pad, stride, dil, 1, 4,
                                 kernels.INQ_NO_SELECTION)
    most = conv(x.abs().double(), w.abs().double(), None, stride, pad).numpy()
    assert (np.abs(to_np(yr) - conv(x.double(), w.double(), None, stride, pad).numpy()) <= most * (n + 8) * 2.0 ** -24).all()
