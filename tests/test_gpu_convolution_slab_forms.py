"""The forms of the binary convolution that keeps input positions in LDS (csrc/kernels/conv_slab.hip): sizes at the
edges of their tiles -- output channels one short of, at and past 64, 128 and 256, maps whose rows do and do not fit a
tile of 32 or 128 windows, a last tile of few windows, channel tiles with padding, one tap -- against float64.

Bound: x is rounded to a multiple of 2^-30 of the largest magnitude under a block's windows, so an output of K terms is
off by at most K * 2^-30 * max|x|, and by the roundings of its conversion to fp32 (two, 2^-24 of the result each).
Windows more than three binades below that largest magnitude have a scale of their own: whatever else lies in their block,
they are off by at most K * 2^-27 of their own largest value.
"""
import numpy as np
import pytest
import torch

from nnabla_amd import kernels

pytestmark = pytest.mark.gpu

# (x shape, output channels, kernel, pad, stride, group)
CASES = [
    ((2, 64, 56, 56), 64, (3, 3), (1, 1), (1, 1), 1),
    ((1, 64, 55, 57), 63, (3, 3), (1, 1), (1, 1), 1),
    ((3, 32, 13, 150), 32, (3, 3), (1, 1), (1, 1), 1),    # rows of the map longer than a tile
    ((40, 32, 28, 28), 1, (1, 1), (0, 0), (1, 1), 1),
    ((9, 128, 28, 28), 128, (3, 3), (1, 1), (1, 1), 1),
    ((4, 96, 27, 27), 65, (5, 5), (2, 2), (1, 1), 1),
    ((2, 48, 31, 17), 127, (3, 3), (1, 1), (2, 2), 1),
    ((1, 96, 9, 9), 129, (3, 3), (0, 2), (1, 1), 1),
    ((2, 256, 14, 14), 257, (1, 1), (0, 0), (1, 1), 1),
    ((40, 64, 14, 14), 512, (1, 1), (0, 0), (1, 1), 1),
    ((64, 96, 28, 28), 128, (3, 3), (1, 1), (1, 1), 2),
    ((1, 30, 5, 5), 40, (3, 3), (1, 1), (1, 1), 1),       # two channels of padding
    ((2, 16, 27, 27), 200, (3, 3), (1, 1), (1, 1), 1),    # half of the only channel tile padding
    ((2, 41, 14, 14), 70, (3, 3), (1, 1), (1, 1), 1),     # 23 channels of padding
    ((8, 250, 56, 56), 65, (3, 3), (1, 1), (1, 1), 1),    # a slab filled several times, the last time in part
    ((12, 200, 55, 57), 33, (3, 3), (1, 1), (1, 1), 1),
]


@pytest.mark.parametrize("xs,O,k,pad,stride,group", CASES)
def test_forward_and_input_gradient_against_float64(xs, O, k, pad, stride, group):
    rng = np.random.RandomState(20)
    dev = torch.device("cuda:0")
    kernels.init(0)
    x = torch.from_numpy(rng.randn(*xs).astype(np.float32))
    W = torch.from_numpy(rng.randn(O, xs[1] // group, *k).astype(np.float32))
    s64 = torch.where(W < 0, -1.0, 1.0).double()
    x64 = x.double().requires_grad_()
    y64 = torch.nn.functional.conv2d(x64, s64, None, stride, pad, 1, group)
    y, Wb = kernels.binary_connect_convolution(x.to(dev), W.to(dev), None, pad, stride, (1, 1), group)
    assert torch.equal(Wb.cpu().double(), s64)
    K = s64[0].numel()
    bound = K * 2.0 ** -30 * float(x.abs().max()) + 2.0 ** -23 * y64.abs()
    assert bool(((y.cpu().double() - y64).abs() <= bound).all())
    # unit strides: the input gradient is the same product on dy, here added to a gradient that is there already
    dy = torch.from_numpy(rng.randn(*y64.shape).astype(np.float32))
    y64.backward(dy.double())
    dx0 = torch.from_numpy(rng.randn(*xs).astype(np.float32))
    dx, _, _ = kernels.binary_convolution_backward(dy.to(dev), x.to(dev), W.to(dev), Wb, None, pad, stride, (1, 1), group,
                                                   dx=dx0.to(dev), want=(True, False, False))
    K, taps, most = (O // group) * k[0] * k[1], k[0] * k[1], float(dy.abs().max())
    want = x64.grad + dx0.double()
    slab = stride == (1, 1) and O // group >= 16
    bound = 2.0 ** -22 * (want.abs() + x64.grad.abs())
    if slab:
        bound = bound + K * 2.0 ** -30 * most
    else:  # unfolded: three digits, 2^-23 of a row's largest; every tap's product and every addition rounded to fp32
        bound = bound + K * most * (2.0 ** -23 + 2 * taps * 2.0 ** -24)
    assert bool(((dx.cpu().double() - want).abs() <= bound).all())


# contractions of one or two k tiles: hardly anything lies between a block's conversion of its inputs and its epilogue
SHORT = [((64, 16, 28, 28), 64, 1), ((64, 32, 28, 28), 64, 1), ((32, 32, 28, 28), 128, 1), ((32, 32, 28, 28), 256, 1),
         ((64, 64, 14, 14), 64, 1), ((64, 32, 27, 27), 33, 1), ((64, 32, 14, 14), 64, 3)]


@pytest.mark.parametrize("xs,O,k", SHORT)
def test_short_contractions(xs, O, k):
    """The windows' sums and their marks of a value that is not finite come from what other wavefronts converted: exact
    results (whole numbers times Sign(W)) in every one of several runs, and one marked window in each run of 32."""
    rng = np.random.RandomState(3)
    kernels.init(0)
    x = torch.from_numpy(rng.randint(-99, 100, xs).astype(np.float32))
    W = torch.from_numpy(rng.randn(O, xs[1], k, k).astype(np.float32))
    s64 = torch.where(W < 0, -1.0, 1.0).double()
    y64 = torch.nn.functional.conv2d(x.double(), s64, None, 1, k // 2)
    xd, Wd = x.cuda(), W.cuda()
    geo = ((k // 2,) * 2, (1, 1), (1, 1), 1)
    for _ in range(5):
        assert torch.equal(kernels.binary_connect_convolution(xd, Wd, None, *geo)[0].cpu().double(), y64)
    xn = x.flatten(2).clone()
    xn[:, 0, 5::32] = float("nan")
    y64 = torch.nn.functional.conv2d(xn.view(xs).double(), s64, None, 1, k // 2)
    for _ in range(5):
        y = kernels.binary_connect_convolution(xn.view(xs).cuda(), Wd, None, *geo)[0].cpu().double()
        assert torch.equal(y.isnan(), y64.isnan()) and torch.equal(y.nan_to_num(), y64.nan_to_num())


def _window_max(v, k, pad, stride):
    m = v.abs().amax(1, keepdim=True)
    return torch.nn.functional.max_pool2d(torch.nn.functional.pad(m, (pad[1], pad[1], pad[0], pad[0])), k, stride)


@pytest.mark.parametrize("xs,O,k,pad,stride,group", [c for c in CASES if c[-1] == 1])
def test_windows_of_different_magnitudes(xs, O, k, pad, stride, group):
    """Patches of the map 2^0 to 2^-70 in size: every output is as good as its own window allows."""
    rng = np.random.RandomState(21)
    kernels.init(0)

    def patches(B, C, H, W):
        e = rng.choice([0, 0, -2, -5, -12, -22, -70], (B, 1, -(-H // 5), -(-W // 6))).repeat(5, 2).repeat(6, 3)
        return torch.from_numpy((rng.randn(B, C, H, W) * 2.0 ** e[:, :, :H, :W]).astype(np.float32))
    x = patches(*xs)
    W = torch.from_numpy(rng.randn(O, xs[1], *k).astype(np.float32))
    s64 = torch.where(W < 0, -1.0, 1.0).double()
    y64 = torch.nn.functional.conv2d(x.double(), s64, None, stride, pad)
    y, Wb = kernels.binary_connect_convolution(x.cuda(), W.cuda(), None, pad, stride, (1, 1), 1)
    bound = s64[0].numel() * 2.0 ** -27 * _window_max(x, k, pad, stride) + 2.0 ** -23 * y64.abs()
    assert bool(((y.cpu().double() - y64).abs() <= bound).all())
    if stride != (1, 1) or O < 16:
        return
    # the input gradient: windows of dy * alpha, the padding that of the transposed convolution
    dy, alpha = patches(*y64.shape), torch.from_numpy(rng.rand(O).astype(np.float32) + 0.5)
    scaled = dy * alpha[None, :, None, None]
    want = torch.nn.grad.conv2d_input(xs, s64, scaled.double(), stride, pad)
    old = torch.zeros(xs)
    old[:, :, ::2] = 2.0 ** -30
    dx, _, _ = kernels.binary_convolution_backward(dy.cuda(), x.cuda(), W.cuda(), Wb, alpha.cuda(), pad, stride, (1, 1), 1,
                                                   dx=old.cuda(), want=(True, False, False))
    n, taps = O * k[0] * k[1], k[0] * k[1]
    most = _window_max(scaled, k, (k[0] - 1 - pad[0], k[1] - 1 - pad[1]), (1, 1))
    # (where the geometry is unfolded instead: three digits of every position's largest, and every addition rounded)
    bound = n * most * (2.0 ** -23 + 2 * taps * 2.0 ** -24) + 2.0 ** -22 * (want.abs() + old)
    assert bool(((dx.cpu().double() - (want + old)).abs() <= bound).all())
