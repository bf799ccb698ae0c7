"""Convolutions of real-valued weights on the bf16 matrix cores (csrc/kernels/conv_real.hip), forward and input gradient,
against float64: strides and remainder classes, paddings, odd extents, tiles that span rows and samples, groups, channel
counts around the chunks of 16 and 32, and values its bf16 parts cannot hold."""
import numpy as np
import pytest
import torch
import torch.nn.functional as TF

from nnabla_amd import kernels
from util import to_np

pytestmark = pytest.mark.gpu

# batch, channels, height, width, maps, kernel, pad, stride, group
CASES = [(1, 16, 7, 7, 16, (3, 3), (1, 1), 1, 1), (3, 17, 9, 5, 65, (3, 3), (1, 1), 2, 1), (2, 33, 14, 14, 70, (1, 1), (0, 0), 2, 1),
         (5, 48, 4, 6, 64, (5, 5), (2, 2), 1, 1), (2, 24, 13, 27, 31, (5, 5), (2, 2), 2, 1), (2, 32, 12, 11, 40, (2, 3), (1, 0), 3, 1),
         (9, 20, 3, 3, 33, (3, 3), (0, 0), 1, 1), (2, 64, 20, 56, 48, (3, 3), (1, 1), 2, 2), (1, 40, 1, 50, 24, (1, 5), (0, 2), 1, 1),
         (8, 128, 56, 56, 64, (5, 5), (2, 2), 2, 1)]  # the longest runs of input a block stages


def _data(case):
    B, C, H, W, O, k, p, s, g = case
    rng = np.random.RandomState(B * C + H + O)
    x = rng.randn(B, C, H, W).astype(np.float32)
    w = (rng.randn(O, C // g, *k) * 0.1).astype(np.float32)
    oh, ow = (H + 2 * p[0] - k[0]) // s + 1, (W + 2 * p[1] - k[1]) // s + 1
    return x, w, rng.randn(O).astype(np.float32), rng.randn(B, O, oh, ow).astype(np.float32)


def _run(case, x, w, b, dy, **grads):
    B, C, H, W, O, k, p, s, g = case
    geo = (p, (s, s), (1, 1))
    xd, wd, dyd = (torch.from_numpy(v).cuda() for v in (x, w, dy))
    I = torch.zeros(w.shape, dtype=torch.int32, device="cuda")
    bd = None if b is None else torch.from_numpy(b).cuda()
    y = kernels.inq_convolution(xd, wd.clone(), I, wd.clone(), I.clone(), bd, *geo, g, 4, kernels.INQ_NO_SELECTION)
    dx = kernels.convolution_backward(dyd, xd, wd, *geo, g, want=(True, False, False), **grads)[0]
    return to_np(y), to_np(dx)


def _conv64(case, x, w, b=None):
    B, C, H, W, O, k, p, s, g = case
    t = lambda v: None if v is None else torch.from_numpy(np.ascontiguousarray(v)).double()
    return TF.conv2d(t(x), t(w), t(b), stride=s, padding=p, groups=g).numpy()


def _grad64(case, w, dy):
    B, C, H, W, O, k, p, s, g = case
    t = lambda v: torch.from_numpy(np.ascontiguousarray(v)).double()
    return torch.nn.grad.conv2d_input((B, C, H, W), t(w), t(dy), stride=s, padding=p, groups=g).numpy()


def _bound(terms, n):
    # a term is good to 2^-23 (the products left out), n terms summed by 16 with six roundings of the running sum each;
    # the digit and fp32 paths, which some of the sizes take, are within it too (24 bits of a row's largest)
    return terms * 2.0 ** -24 * (6 * n / 64.0 + 24)


@pytest.mark.parametrize("case", CASES)
def test_against_float64(case):
    kernels.init(0)
    B, C, H, W, O, k, p, s, g = case
    x, w, b, dy = _data(case)
    y, dx = _run(case, x, w, b, dy)
    n = C // g * k[0] * k[1]
    bound = _bound(_conv64(case, np.abs(x), np.abs(w)), n) + 2.0 ** -23 * np.abs(_conv64(case, x, w, b)) + 2.0 ** -24 * 4
    assert (np.abs(y - _conv64(case, x, w, b)) <= bound).all()
    ref = _grad64(case, w, dy)
    bound = _bound(_grad64(case, np.abs(w), np.abs(dy)), O // g * k[0] * k[1]) + 2.0 ** -23 * np.abs(ref)
    assert (np.abs(dx - ref) <= bound).all()
    # added to what is there
    old = torch.full(x.shape, 3.0, device="cuda")
    _, dx2 = _run(case, x, w, b, dy, dx=old)
    assert (np.abs(dx2 - (ref + 3.0)) <= bound + 2.0 ** -23 * (3.0 + np.abs(ref))).all()


@pytest.mark.parametrize("signs_given", [True, False])
def test_binary_input_gradient_with_a_stride(signs_given):
    kernels.init(0)
    case = (16, 64, 28, 28, 128, (3, 3), (1, 1), 2, 1)
    x, w, _, dy = _data(case)
    alpha = np.abs(w).mean(axis=(1, 2, 3)).astype(np.float32)
    xd, wd, dyd, ad = (torch.from_numpy(v).cuda() for v in (x, w, dy, alpha))
    dx = kernels.binary_convolution_backward(dyd, xd, wd, torch.sign(wd) if signs_given else None, ad, (1, 1), (2, 2), (1, 1), 1,
                                             want=(True, False, False))[0]
    wb = np.sign(w) * alpha[:, None, None, None]
    ref = _grad64(case, wb, dy)
    assert (np.abs(to_np(dx) - ref) <= _bound(_grad64(case, np.abs(wb), np.abs(dy)), 128 * 9)).all()


def test_values_out_of_range():
    kernels.init(0)
    case = (4, 32, 28, 28, 72, (3, 3), (1, 1), 2, 1)
    x, w, b, dy = _data(case)
    y0, dx0 = _run(case, x, w, b, dy)
    x[0, 3, 5, 5], x[1, 0, 0, 0], x[2, 31, 27, 27] = np.inf, np.nan, -np.inf
    dy[0, 70, 3, 3], dy[3, 0, 13, 0] = np.nan, np.inf
    y, dx = _run(case, x, w, b, dy)
    with np.errstate(invalid="ignore"):
        ry, rdx = _conv64(case, x, w, b), _grad64(case, w, dy)
    for f in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(f(y), f(ry)) and np.array_equal(f(dx), f(rdx))
    assert np.array_equal(y[np.isfinite(ry)], y0[np.isfinite(ry)])
    assert np.array_equal(dx[np.isfinite(rdx)], dx0[np.isfinite(rdx)])
    # inputs at the far ends of fp32, and rows of weights of any size
    x, w, b, dy = _data(case)
    x[1] *= np.float32(1e-30)
    x[2] *= np.float32(1e33)
    w[7] *= np.float32(1e-33)
    y, _ = _run(case, x, w, None, dy)
    ref, terms = _conv64(case, x, w), _conv64(case, np.abs(x), np.abs(w))
    assert (np.abs(y - ref) <= _bound(terms, 288) + 2.0 ** -149).all()


@pytest.mark.parametrize("case", [(4, 32, 28, 28, 72, (3, 3), (1, 1), 2, 1), (2, 40, 27, 27, 70, (3, 3), (1, 1), 1, 1)])
@pytest.mark.parametrize("size", [1e-28, 1e-33, 1e-36, 1e-40])
def test_windows_of_tiny_values_beside_ordinary_ones(case, size):
    """A corner of every map (inputs and output gradients) far below the range of the bf16 parts: what only it reaches is
    as good as anywhere else, down to the last place of the smallest numbers."""
    kernels.init(0)
    x, w, b, dy = _data(case)
    x[:, :, :12, :11] *= np.float32(size)
    dy[:, :, :6, :7] *= np.float32(size)
    y, dx = _run(case, x, w, None, dy)
    ref, n = _conv64(case, x, w), 9 * case[1]
    assert (np.abs(y - ref) <= _bound(_conv64(case, np.abs(x), np.abs(w)), n) + 2.0 ** -23 * np.abs(ref) + 2.0 ** -149).all()
    ref = _grad64(case, w, dy)
    bound = _bound(_grad64(case, np.abs(w), np.abs(dy)), 9 * case[4]) + 2.0 ** -23 * np.abs(ref) + 2.0 ** -149
    assert (np.abs(dx - ref) <= bound).all()
