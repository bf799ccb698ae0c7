"""The digit x digit product (csrc/kernels/gemm_digits.hip) around its tiles: rows and columns at and one past 32, 64 and
128, an odd number of columns (64-bit stores of column pairs), contractions of one to several k steps, split and in two
k groups, outputs of one and of two blocks per CU, one-digit operands on either side, and sums added to what is there,
against float64."""
import numpy as np
import pytest
import torch

from nnabla_amd import kernels
from util import to_np

pytestmark = pytest.mark.gpu


def _check(got, a, b, add=0.0):
    """Operands are good to 2^-23 of their row's (column's) largest, the products left out below 2^-23 of both."""
    a, b = a.double(), b.double()
    k = a.shape[1]
    big = a.abs().amax(1, keepdim=True) * b.abs().amax(0, keepdim=True)
    ref = a @ b + add
    bound = big * (k * 3 * 2.0 ** -23) + ref.abs() * 2.0 ** -22 + abs(add) * 2.0 ** -23
    assert bool(((got.double() - ref).abs() <= bound).all())


# samples (the contraction of dW), inputs, outputs: past the sizes that the one-launch product takes
@pytest.mark.parametrize("M,K,N", [(4096, 33, 65), (3000, 129, 257), (2049, 1025, 1023), (300, 2049, 2175),
                                   (1000, 2176, 2305), (257, 4097, 1100)])
def test_weight_gradient(M, K, N):
    kernels.init(0)
    gen = torch.Generator(device="cuda").manual_seed(M + K + N)
    x, dy = (torch.randn(M, n, generator=gen, device="cuda") for n in (K, N))
    W = torch.randn(K, N, generator=gen, device="cuda")
    old = torch.full((K, N), 2.0, device="cuda")
    _check(kernels.affine_backward(dy, x, W, want=(False, True, False))[1], x.T, dy)
    kernels.affine_backward(dy, x, W, dW=old, want=(False, True, False))
    _check(old, x.T, dy, 2.0)


# rows around the ends of slabs of 64, 128 and 256 rows and where the number of groups that fold their statistics changes; the
# largest value of every column, and of dy's, lies in another slab: a slab left out gives digits that do not fit
@pytest.mark.parametrize("M,K,N", [(4096, 40, 70), (4097, 1, 3), (16384, 33, 5), (16385, 7, 64), (16385, 300, 11),
                                   (70001, 5, 66), (300000, 3, 2)])
@pytest.mark.parametrize("accumulate", [False, True])
def test_statistics_of_tall_columns(M, K, N, accumulate):
    kernels.init(0)
    gen = torch.Generator(device="cuda").manual_seed(M + K + N)
    x, dy = (torch.randn(M, n, generator=gen, device="cuda") for n in (K, N))
    x[torch.linspace(0, M - 1, K + 1, device="cuda").long()[1:], torch.arange(K, device="cuda")] = 300.0
    dy[torch.linspace(0, M - 1, N, device="cuda").long().flip(0), torch.arange(N, device="cuda")] = -500.0
    W = torch.randn(K, N, generator=gen, device="cuda")
    given = dict(dW=torch.full((K, N), 2.0, device="cuda"), db=torch.full((N,), 3.0, device="cuda")) if accumulate else {}
    _, dW, db = kernels.affine_backward(dy, x, W, want=(False, True, True), **given)
    _check(dW, x.T, dy, 2.0 if accumulate else 0.0)
    # chains: at most 64 rows of a slab and thread, four threads, 19 slabs a group (300000 rows), 64 groups, what was there
    ref, bound = dy.double().sum(0) + (3.0 if accumulate else 0.0), dy.double().abs().sum(0) * (160 * 2.0 ** -24)
    assert bool(((db.double() - ref).abs() <= bound + 1e-6).all())


@pytest.mark.parametrize("K", [4097, 16384, 16385, 70001])
@pytest.mark.parametrize("odd", ["none", "last", "first", "small"])
def test_one_digit_weights_of_tall_columns(K, odd):
    """Columns of powers of two are held in one digit unless a value in any slab is none, or is seven binades smaller."""
    kernels.init(0)
    gen = torch.Generator(device="cuda").manual_seed(K)
    x, W = torch.randn(3, K, generator=gen, device="cuda"), _narrow_weights(K, 5, gen)
    if odd != "none":
        W[0 if odd == "first" else K - 1, 2] = 2.0 ** -9 if odd == "small" else 0.7
        x[:, 0 if odd == "first" else K - 1] = 1000.0
    _check(kernels.affine_digits(x, W), x, W)
    if odd == "none": # (one-digit weights drop no product: what is left is x's rounding and the result's)
        ref = x.double() @ W.double()
        bound = x.abs().amax(1, keepdim=True).double() * W.double().abs().sum(0) * 2.0 ** -23 + ref.abs() * 2.0 ** -22
        assert bool(((kernels.affine_digits(x, W).double() - ref).abs() <= bound).all())


def _narrow_weights(K, N, gen):
    return (torch.sign(torch.randn(K, N, generator=gen, device="cuda")) *
            torch.exp2(torch.randint(-5, 1, (K, N), generator=gen, device="cuda").float()))


# (past the one-launch product in both directions: split contractions, one block per CU, two blocks)
ONE_DIGIT_SIZES = [(300, 4095, 1601), (1500, 2000, 2111), (2100, 2049, 1100)]


@pytest.mark.parametrize("M,K,N", ONE_DIGIT_SIZES)
@pytest.mark.parametrize("narrow_x", [False, True])
@pytest.mark.parametrize("narrow_w", [False, True])
def test_one_digit_operands(M, K, N, narrow_x, narrow_w):
    kernels.init(0)
    gen = torch.Generator(device="cuda").manual_seed(M + K + N)
    x = torch.randn(M, K, generator=gen, device="cuda")
    W = _narrow_weights(K, N, gen) if narrow_w else torch.randn(K, N, generator=gen, device="cuda")
    b = torch.randn(N, generator=gen, device="cuda")
    if narrow_x:
        x = kernels.fixed_point_quantize(x, True, 8, 2.0 ** -4)
    y = kernels.affine_digits(x, W, b)
    _check(y - b, x, W) if not (narrow_x and narrow_w) else _exact(y, x, W, b)


@pytest.mark.parametrize("M,K,N", ONE_DIGIT_SIZES)
@pytest.mark.parametrize("narrow_dy", [False, True])
@pytest.mark.parametrize("narrow_w", [False, True])
def test_input_gradient_under_one_digit_rows(M, K, N, narrow_dy, narrow_w):
    """dx = dy . W^T: both operands scaled by rows, so one-digit rows of W multiply their top digit, and those of dy with
    them.  A tile that holds one other row takes the general form, which gives its remaining rows the same bits."""
    kernels.init(0)
    gen = torch.Generator(device="cuda").manual_seed(M + K + N + 1)
    dy = torch.randn(M, N, generator=gen, device="cuda")
    if narrow_dy:
        dy = kernels.fixed_point_quantize(dy, True, 8, 2.0 ** -4)
    W = _narrow_weights(K, N, gen) if narrow_w else torch.randn(K, N, generator=gen, device="cuda")
    x = torch.zeros(M, K, device="cuda")
    gradient = lambda g, w, out=None: kernels.affine_backward(g, x, w, dx=out, want=(True, False, False))[0]
    dx = gradient(dy, W)
    if narrow_dy and narrow_w:
        assert torch.equal(dx, (dy.double() @ W.double().T).float())  # small integers on both sides
    else:
        _check(dx, dy, W.T)
    old = torch.full((M, K), 2.0, device="cuda")
    gradient(dy, W, old)
    _check(old, dy, W.T, 2.0)
    W2, dy2 = W.clone(), dy.clone()
    for row in (5, K // 2, K - 1):
        W2[row] = torch.randn(N, generator=gen, device="cuda")
    kept = (W2 == W).all(1)
    assert kept.sum() == K - 3 and torch.equal(gradient(dy, W2)[:, kept], dx[:, kept])
    for row in (0, M // 2, M - 1):
        dy2[row] = torch.randn(N, generator=gen, device="cuda")
    kept = (dy2 == dy).all(1)
    assert kept.sum() == M - 3 and torch.equal(gradient(dy2, W)[kept], dx[kept])


def _exact(y, x, W, b):
    """Small integers on both sides: the sum is exact, rounded once, and once more with the bias."""
    ref = (x.double() @ W.double()).float() + b
    assert np.array_equal(to_np(y), to_np(ref))
