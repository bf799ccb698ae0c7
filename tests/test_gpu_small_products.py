"""Real-valued products in one launch (csrc/kernels/gemm_small.hip): extents at and one past its tiles (32 rows, 64
columns, 32 terms, eight wavefronts of k tiles), each operand order, sums added to what is there, magnitudes its bf16
parts cannot hold and non-finite values, against float64."""
import numpy as np
import pytest
import torch

from nnabla_amd import kernels
from util import to_np

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (2, 33, 65), (32, 32, 64), (33, 31, 63), (20, 250, 250), (31, 256, 129), (65, 257, 64), (100, 513, 70),
         (40, 1025, 3), (17, 3000, 100), (300, 64, 1000)]


def _case(M, K, N, scale=1.0):
    rng = np.random.RandomState(M + K + N)
    x = (rng.randn(M, K) * scale).astype(np.float32)
    W = (rng.randn(K, N) / scale).astype(np.float32)
    W.ravel()[::5] = 0.0
    return x, W, rng.randn(N).astype(np.float32), rng.randn(M, N).astype(np.float32)


def _check(got, a, b, add=0.0):
    """Terms are good to 2^-24 (three of nine partial products left out), sums of k of them by 16 in fp32 to
    (k / 16 / 8 + 4) roundings of the running sum, which is at most sum |a| |b|."""
    a, b = a.astype(np.float64), b.astype(np.float64)
    k = a.shape[1]
    bound = (np.abs(a) @ np.abs(b)) * 2.0 ** -24 * (k / 128.0 + 6) + 2.0 ** -23 * np.abs(add) + 2.0 ** -24 * np.abs(a @ b)
    assert (np.abs(to_np(got) - (a @ b + add)) <= bound).all()


@pytest.mark.parametrize("M,K,N", SIZES)
@pytest.mark.parametrize("scale", [1.0, 2.0 ** 40])
def test_against_float64(M, K, N, scale):
    kernels.init(0)
    x, W, b, dy = _case(M, K, N, scale)
    xd, Wd, bd, dyd = (torch.from_numpy(v).cuda() for v in (x, W, b, dy))
    _check(kernels.affine_digits(xd, Wd, bd), x, W, b.astype(np.float64))
    dx, dW, _ = kernels.affine_backward(dyd, xd, Wd, want=(True, True, False))
    _check(dx, dy, W.T.copy())
    _check(dW, x.T.copy(), dy)
    I = torch.zeros(K, N, dtype=torch.int32, device="cuda")
    y = kernels.inq_affine(xd, Wd.clone(), I, Wd.clone(), I.clone(), bd, 4, kernels.INQ_NO_SELECTION)
    _check(y, x, W, b.astype(np.float64))


def test_sums_added_to_what_is_there():
    kernels.init(0)
    x, W, b, dy = _case(70, 130, 66)
    x[3] = 1e-30  # a row out of the range of the bf16 parts
    xd, Wd, dyd = (torch.from_numpy(v).cuda() for v in (x, W, dy))
    dx0, dW0 = torch.full_like(xd, 2.0), torch.full_like(Wd, -3.0)
    kernels.affine_backward(dyd, xd, Wd, dx=dx0, dW=dW0, want=(True, True, False))
    _check(dx0, dy, W.T.copy(), 2.0)
    _check(dW0, x.T.copy(), dy, -3.0)


@pytest.mark.parametrize("tiny,huge", [(1e-30, 1e25), (1e-39, 1e30), (2.0 ** -51, 2.0 ** 61)])
def test_rows_and_columns_out_of_range(tiny, huge):
    kernels.init(0)
    x, W, b, _ = _case(40, 100, 70)
    x[5] *= tiny
    x[6, 50] = huge
    W[:, 9] *= tiny
    W[17, 10] = huge
    xd, Wd = torch.from_numpy(x).cuda(), torch.from_numpy(W).cuda()
    with np.errstate(over="ignore"):
        _check_rel = x.astype(np.float64) @ W.astype(np.float64)
    y = to_np(kernels.affine_digits(xd, Wd, None))
    big = (np.abs(x).astype(np.float64) @ np.abs(W).astype(np.float64))
    fin = np.abs(_check_rel) < 3e38
    # (results below 2^-126 are held to 2^-149)
    assert (np.abs(y - _check_rel)[fin] <= (big * 2.0 ** -24 * 8 + 2.0 ** -149)[fin]).all()


def test_non_finite_values():
    kernels.init(0)
    x, W, b, _ = _case(40, 100, 130)
    clean = to_np(kernels.affine_digits(torch.from_numpy(x).cuda(), torch.from_numpy(W).cuda(), torch.from_numpy(b).cuda()))
    x[3, 7], x[3, 50], x[39, 99], x[5, 0] = np.inf, np.inf, -np.inf, np.nan
    W[2, 4], W[99, 129] = np.inf, np.nan
    with np.errstate(invalid="ignore"):
        ref = x.astype(np.float64) @ W.astype(np.float64) + b
    y = to_np(kernels.affine_digits(torch.from_numpy(x).cuda(), torch.from_numpy(W).cuda(), torch.from_numpy(b).cuda()))
    for f in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(f(y), f(ref))
    rows, cols = np.isfinite(x).all(1), np.isfinite(W).all(0)
    assert np.array_equal(y[rows][:, cols], clean[rows][:, cols])


@pytest.mark.parametrize("size", [2.0 ** 56, 2.0 ** 57, 2.0 ** 60])
def test_sums_that_cancel_do_not_overflow_on_the_way(size):
    kernels.init(0)
    x = torch.full((20, 4096), size, device="cuda")
    x[:, 2048:] = -size
    x[7, 5] = 0.0
    W, b = torch.full((4096, 64), size, device="cuda"), torch.ones(64, device="cuda")
    y = kernels.affine_digits(x, W, b)
    want = torch.ones(20, 64, device="cuda")
    want[7] = -size * size
    assert torch.equal(y, want)
