"""Convolutions of few channels to at most 64 maps, which the matrix-core forms take from four taps on where they are
estimated the faster ones and the fp32 kernel otherwise: both sides of the line, few windows and many, against float64."""
import numpy as np
import pytest
import torch
import torch.nn.functional as TF

from nnabla_amd import kernels
from util import to_np

pytestmark = pytest.mark.gpu

# batch, channels, height, width, maps, kernel, stride
CASES = [(1, 16, 8, 8, 16, 3, 1), (1, 23, 9, 9, 24, 2, 1), (2, 16, 27, 27, 64, 3, 1), (1, 16, 31, 33, 16, 3, 1),
         (1, 16, 32, 32, 16, 3, 1), (6, 23, 13, 14, 64, 3, 1), (5, 20, 28, 28, 33, 2, 2),
         (4, 18, 27, 27, 24, 5, 2), (3, 17, 20, 21, 30, 1, 1), (2, 22, 40, 40, 64, (1, 3), 1)]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("zero_to", [1.0, 0.0])
def test_both_weights_against_float64(case, zero_to):
    kernels.init(0)
    B, C, H, W, O, k, s = case
    k = k if isinstance(k, tuple) else (k, k)
    rng = np.random.RandomState(B + C + H + O)
    x = np.maximum(rng.randn(B, C, H, W), 0).astype(np.float32)
    w = (rng.randn(O, C, *k) * 0.1).astype(np.float32)
    w.ravel()[::9] = 0.0
    b = rng.randn(O).astype(np.float32)
    x[0, 0, 1, 1] = np.inf
    geo = ((k[0] // 2, k[1] // 2), (s, s), (1, 1))
    xd, wd, bd = (torch.from_numpy(v).cuda() for v in (x, w, b))
    signs = np.where(w > 0, 1.0, np.where(w < 0, -1.0, zero_to))
    alpha = np.abs(w.astype(np.float64)).mean((1, 2, 3))
    conv = lambda a, f, c=None: TF.conv2d(torch.from_numpy(a).double(), torch.from_numpy(f).double(),
                                          None if c is None else torch.from_numpy(c).double(), stride=s, padding=geo[0]).numpy()
    n, clean = C * k[0] * k[1], np.where(np.isfinite(x), x, 0).astype(np.float32)

    def check(got, f):
        with np.errstate(invalid="ignore"):
            ref = conv(x, f, b)
        fin = np.isfinite(ref)
        assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(np.isposinf(got), np.isposinf(ref))
        # sums of n terms in fp32 one after the other at the worst, terms good to 2^-23
        bound = conv(clean, np.abs(f)) * (n + 8) * 2.0 ** -24 + np.abs(ref) * 3e-6 + 2.0 ** -23
        assert (np.abs(got - ref)[fin] <= bound[fin]).all() and fin.mean() > 0.5

    y, Wb, al = kernels.binary_weight_convolution(xd, wd, bd, *geo, 1, zero_to)
    assert np.array_equal(to_np(Wb), signs.astype(np.float32))
    check(to_np(y), signs * alpha[:, None, None, None])
    I = torch.zeros(w.shape, dtype=torch.int32, device="cuda")
    yr = kernels.inq_convolution(xd, wd.clone(), I, wd.clone(), I.clone(), bd, *geo, 1, 4, kernels.INQ_NO_SELECTION)
    check(to_np(yr), w.astype(np.float64))


@pytest.mark.parametrize("B,C,sp,O,k", [(64, 16, (56, 56), 8, (1, 4)), (150, 2, (20, 20), 8, (2, 2)),
                                        (16, 8, (112, 112), 16, (3, 3))])
def test_real_weights_over_many_windows_stay_on_the_fp32_kernel(B, C, sp, O, k):
    """Its products one after the other in fp32, bit for bit: on the matrix cores such layers take two to six times as long,
    their rows of weights and channels being padding for the most part."""
    kernels.init(0)
    rng = np.random.RandomState(B + C + O)
    x, w = rng.randn(B, C, *sp).astype(np.float32), rng.randn(O, C, *k).astype(np.float32)
    pad = tuple(v // 2 for v in k)
    I = torch.zeros(w.shape, dtype=torch.int32, device="cuda")
    wd = torch.from_numpy(w).cuda()
    y = to_np(kernels.inq_convolution(torch.from_numpy(x).cuda(), wd, I, wd.clone(), I.clone(), None, pad, (1, 1), (1, 1), 1,
                                      4, kernels.INQ_NO_SELECTION))
    xp = np.pad(x[-1], ((0, 0), (pad[0],) * 2, (pad[1],) * 2))
    ref = np.zeros(y.shape[1:], np.float32)
    for c in range(C):
        for i in range(k[0]):
            for j in range(k[1]):
                ref = ref + xp[c, i:i + ref.shape[1], j:j + ref.shape[2]] * w[:, c, i, j, None, None]
    assert np.array_equal(y[-1], ref)
