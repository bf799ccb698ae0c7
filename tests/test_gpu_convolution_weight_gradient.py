"""The weight gradient on the fp16 matrix cores (csrc/kernels/conv_dw.hip) against float64, at the sizes where its tiles,
groups of eight positions, phases and splits have their edges, alone and added to a gradient that is there already.

A value is held as two fp16 numbers (22 bits at least: 2^-22 of a product per factor, and 2^-22 for the product of the
two remainders) and sums are fp32: an element is off by at most (3 * 2^-22 + n * 2^-24) * sum |x dy|, n the roundings of
the longest chain of sums (three per sixteen positions of a block).  The errors of the products are independent of each
other, so the norm of the error is far below that: 2^-23 for the products and 2^-25 * sqrt(3 n / 2) for the sums of random
terms, under 1e-6 of the norm of the gradient for n up to a few thousand.
"""
import numpy as np
import pytest
import torch

from nnabla_amd import kernels

pytestmark = pytest.mark.gpu

# (x shape, output channels, kernel, pad, stride, group)
CASES = [
    ((2, 64, 56, 56), 64, (3, 3), (1, 1), 1, 1),
    ((3, 33, 55, 57), 65, (3, 3), (1, 1), 1, 1),     # channels one past a tile, rows of 57 = 7 groups and one position
    ((5, 8, 7, 7), 16, (3, 3), (1, 1), 1, 1),        # the fewest channels; whole samples of a small map per tile
    ((37, 40, 7, 7), 24, (3, 3), (1, 1), 1, 1),      # a last tile of fewer samples
    ((1, 96, 9, 8), 63, (5, 3), (2, 1), 1, 1),       # rows of taps in two passes, the second of two rows
    ((2, 32, 13, 17), 32, (1, 3), (0, 1), 1, 1),     # one row of taps
    ((2, 40, 28, 28), 48, (3, 3), (1, 1), 2, 1),
    ((2, 31, 27, 29), 130, (3, 3), (0, 1), 2, 1),    # no padding above and below, odd extents, two strides
    ((2, 48, 27, 27), 33, (5, 5), (2, 2), 1, 1),
    ((3, 17, 14, 15), 64, (5, 5), (2, 2), 2, 1),
    ((4, 129, 14, 14), 65, (1, 1), (0, 0), 1, 1),    # 128 input channels and one
    ((3, 64, 13, 13), 48, (1, 1), (0, 0), 2, 1),
    ((2, 64, 14, 14), 64, (3, 3), (1, 1), 1, 2),     # groups
    ((70, 32, 5, 3), 32, (3, 3), (1, 1), 1, 1),      # rows shorter than a group of positions
    ((2, 16, 3, 80), 32, (3, 3), (1, 1), 1, 1),      # the longest rows
    # blocks of several tiles, the last one of fewer
    ((41, 512, 7, 7), 512, (3, 3), (1, 1), 1, 1),
    ((9, 256, 14, 14), 512, (3, 3), (1, 1), 2, 1),
    ((9, 512, 14, 14), 1024, (1, 1), (0, 0), 1, 1),
    ((7, 128, 14, 14), 256, (5, 5), (2, 2), 1, 1),
    ((4, 512, 14, 14), 512, (5, 5), (2, 2), 1, 1),   # left to the product of digit operands
]

DIGITS = CASES[-1][:3]


@pytest.mark.parametrize("xs,O,k,pad,stride,group", CASES)
def test_against_float64(xs, O, k, pad, stride, group):
    rng = np.random.RandomState(7)
    dev = torch.device("cuda:0")
    kernels.init(0)
    scale = (10.0 ** rng.uniform(-3, 3, (1, xs[1], 1, 1)))   # channels of very different magnitudes
    x = torch.from_numpy((rng.randn(*xs) * scale).astype(np.float32))
    W = torch.from_numpy(rng.randn(O, xs[1] // group, *k).astype(np.float32))

    def gradient(x64, dy64):
        w = W.double().requires_grad_()
        torch.nn.functional.conv2d(x64, w, None, stride, pad, 1, group).backward(dy64)
        return w.grad
    oh = [(xs[2 + i] + 2 * pad[i] - k[i]) // stride + 1 for i in (0, 1)]
    dy = torch.from_numpy((rng.randn(xs[0], O, *oh) * 1e-2).astype(np.float32))
    ref, most = gradient(x.double(), dy.double()), gradient(x.double().abs(), dy.double().abs())
    n = 3 * (xs[0] * oh[0] * (-(-oh[1] // 8) * 8) / 16 + 16)
    bound = (3 * 2.0 ** -22 + n * 2.0 ** -24) * most
    s = (stride, stride)
    _, dW, _ = kernels.convolution_backward(dy.to(dev), x.to(dev), W.to(dev), pad, s, (1, 1), group,
                                            want=(False, True, False))
    err = (dW.cpu().double() - ref).abs()
    assert bool((err <= bound).all())
    per_channel = (err ** 2).sum((0, 2, 3)).sqrt() / (ref ** 2).sum((0, 2, 3)).sqrt()
    # (digit operands hold 24 bits of a channel's largest value, about five times its root mean square: 5 * 2^-23 a factor)
    assert float(per_channel.max()) <= (3e-6 if (xs, O, k) == DIGITS else 1e-6)
    dW0 = torch.from_numpy(rng.randn(*W.shape).astype(np.float32)) * ref.float().abs().mean()
    _, acc, _ = kernels.binary_convolution_backward(dy.to(dev), x.to(dev), W.to(dev), None, None, pad, s, (1, 1), group,
                                                    dW=dW0.to(dev), want=(False, True, False))
    assert torch.equal(acc, dW0.to(dev) + dW)


# places where a value only meets the zeros that fill up a row, a map, a tile or the last step, besides ordinary ones
@pytest.mark.parametrize("xs,k,s,at", [((2, 32, 9, 9), 3, 1, [(4, 4)]), ((2, 32, 9, 9), 3, 1, [(0, 8), (8, 0), (8, 8)]),
                                       ((3, 40, 7, 11), 3, 2, [(6, 10), (0, 0), (5, 9)]), ((2, 16, 14, 13), 5, 1, [(13, 12)]),
                                       ((5, 24, 5, 5), 3, 1, [(0, 0), (4, 4)]), ((3, 130, 13, 7), 1, 1, [(12, 6)]),
                                       ((2, 32, 10, 12), 1, 2, [(9, 11), (8, 10)]), ((1, 20, 11, 9), 5, 2, [(10, 8), (0, 7)])])
def test_non_finite_values(xs, k, s, at):
    """As the unfolded product gives it: an infinity where it stands against a finite gradient, NaN against a zero or the
    padding or another one of the other sign, and nothing in the weights that it does not meet."""
    rng = np.random.RandomState(8)
    kernels.init(0)
    B, C, H, W_ = xs
    p, O = k // 2, 40
    x = torch.from_numpy(rng.randn(*xs).astype(np.float32))
    oh, ow = (H + 2 * p - k) // s + 1, (W_ + 2 * p - k) // s + 1
    dy = torch.from_numpy(rng.randn(B, O, oh, ow).astype(np.float32))
    run = lambda: kernels.convolution_backward(dy.cuda(), x.cuda(), torch.zeros(O, C, k, k, device="cuda"), (p, p), (s, s),
                                               (1, 1), 1, want=(False, True, False))[1].cpu()
    for i, (y_, x_) in enumerate(at):
        x[i % B, 5 + i, y_, x_] = 0.0
    dy[0, 7, 0, 0], dy[B - 1, 9, oh - 1, ow - 1], dy[0, 3] = 0.0, 0.0, 0.0
    clean = run()
    for i, (y_, x_) in enumerate(at):
        x[i % B, 5 + i, y_, x_] = float("inf") if i != 1 else float("nan")
    dy[0, 7, 0, 0] = float("-inf")
    dy[B - 1, 9, oh - 1, ow - 1] = float("nan")
    cols = torch.nn.functional.unfold(x.double(), k, padding=p, stride=s)
    want = sum(torch.nan_to_num(d, 0, 0, 0) @ torch.nan_to_num(u, 0, 0, 0).t() for d, u in zip(dy.double().flatten(2), cols))
    # which outputs, term by term: 0 * Inf and Inf - Inf are NaN
    nan, plus, minus = (torch.zeros(O, C * k * k, dtype=torch.bool) for _ in range(3))
    for d, u in zip(dy.double().flatten(2), cols):
        for m in range(oh * ow):
            if d[:, m].isfinite().all() and u[:, m].isfinite().all():
                continue
            t = d[:, m, None] * u[None, :, m]
            nan |= t.isnan()
            plus |= t == float("inf")
            minus |= t == float("-inf")
    nan |= plus & minus
    got = run().flatten(1)
    assert torch.equal(got.isnan(), nan)
    assert torch.equal(got == float("inf"), plus & ~nan) and torch.equal(got == float("-inf"), minus & ~nan)
    fin = ~(nan | plus | minus)
    assert float((got.double() - want)[fin].abs().max()) <= 1e-5 * float(want.abs().max())
    got, clean = got.view(O, C, -1), clean.view(O, C, -1)
    rows = [o for o in range(O) if o not in (7, 9)]
    channels = [c for c in range(C) if not 5 <= c < 5 + len(at)]
    assert torch.equal(got[rows][:, channels], clean[rows][:, channels])


@pytest.mark.parametrize("sign,limit", [(False, 6e-7), (True, 1e-7)])
def test_many_positions_under_many_weights(sign, limit):
    """A wavefront adds up at most 512 positions in fp32 (four roundings in each of three products per sixteen: 384), the
    rest is added in double: terms of random signs are off by 0.29 * 2^-23.5 * sqrt(384 * 384 / 2) / sqrt(384) of the norm
    for a chain and for the whole (3e-7), besides 1e-7 for the products; terms of one sign by
    0.29 * 2^-23.5 * sqrt(384 / 3) for a chain and a tenth of it for the mean of 98 (3e-8), besides the result's rounding.
    Chains of 6272 positions are off by 1.0e-6 and 3.3e-7."""
    kernels.init(0)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(5)
    x = torch.randn(64, 512, 28, 28, device="cuda", generator=gen).clamp_(min=0)
    dy = torch.randn(64, 512, 28, 28, device="cuda", generator=gen) * 1e-2
    dy = dy.abs() if sign else dy
    dW = kernels.convolution_backward(dy, x, torch.zeros(512, 512, 3, 3, device="cuda"), (1, 1), (1, 1), (1, 1), 1,
                                      want=(False, True, False))[1]
    want = torch.zeros(512, 512 * 9, dtype=torch.float64, device="cuda")
    for n in range(64):
        want += dy[n].double().flatten(1) @ torch.nn.functional.unfold(x[n:n + 1].double(), 3, padding=1)[0].t().contiguous()
    assert float((dW.double().flatten(1) - want).norm() / want.norm()) <= limit


@pytest.mark.parametrize("xs,O,k", [((32, 32, 56, 56), 32, 3), ((64, 16, 56, 56), 16, 5), ((64, 8, 56, 56), 32, 3)])
def test_few_weights_keep_their_fp32_products(xs, O, k):
    """Sums in threads over products of 24 bits: 1.4e-7 to 1.9e-7 off float64 (two fp16 numbers a value: 2.1e-7 to 3.8e-7)."""
    kernels.init(0)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(6)
    x = torch.randn(*xs, device="cuda", generator=gen).clamp_(min=0)
    dy = torch.randn(xs[0], O, *xs[2:], device="cuda", generator=gen) * 1e-2
    dW = kernels.convolution_backward(dy, x, torch.zeros(O, xs[1], k, k, device="cuda"), (k // 2,) * 2, (1, 1), (1, 1), 1,
                                      want=(False, True, False))[1]
    want = torch.zeros(O, xs[1] * k * k, dtype=torch.float64, device="cuda")
    for n in range(xs[0]):
        cols = torch.nn.functional.unfold(x[n:n + 1].double(), k, padding=k // 2)[0]
        want += dy[n].double().flatten(1) @ cols.t().contiguous()
    assert float((dW.double().flatten(1) - want).norm() / want.norm()) <= 2.0e-7


def test_partial_sums_up_to_2_gib():
    """Blocks of 1024 positions would write 3.7 GB: 227 splits of 1792 positions instead (1e-7 for the products and
    0.29 * 2^-23.5 * sqrt(672 / 2) for the chains: 4.6e-7; digit operands are 1.3e-6 off)."""
    kernels.init(0)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(9)
    x = torch.randn(128, 512, 56, 56, device="cuda", generator=gen)
    dy = torch.randn(128, 512, 56, 56, device="cuda", generator=gen)
    W = torch.empty(512, 512, 3, 3, device="cuda")
    dW = kernels.convolution_backward(dy, x, W, (1, 1), (1, 1), (1, 1), 1, want=(False, True, False))[1]
    want = torch.zeros(8, 18, dtype=torch.float64, device="cuda")
    for n in range(128):
        cols = torch.nn.functional.unfold(x[n:n + 1, ::256].double(), 3, padding=1)[0]
        want += dy[n, ::64].flatten(1).double() @ cols.t().contiguous()
    assert float((dW[::64, ::256].reshape(8, -1).double() - want).norm() / want.norm()) <= 8e-7
