"""Binary affine layers small enough for the one-launch form (csrc/kernels/binary_fused.hip) and the walk over weights
whose rows start at any multiple of four bytes (binary_prepare.hip): extents at and one past the tiles (32 rows, 64
columns, 32 terms; 512 and 1024 terms; 256 columns of the walk), against the oracle and float64."""
import numpy as np
import pytest
import torch

import oracle
from nnabla_amd import kernels
from util import bits_equal, to_np

pytestmark = pytest.mark.gpu

SMALL = [(1, 5, 1), (1, 65, 67), (32, 32, 64), (33, 31, 65), (20, 250, 250), (31, 512, 63), (65, 513, 129), (66, 1024, 64),
         (100, 1023, 3), (67, 100, 130)]
LARGE = [(20, 1025, 257), (70, 1100, 255), (33, 2047, 4), (40, 1200, 770), (65, 1030, 1021)]


def _case(M, K, N):
    rng = np.random.RandomState(M + K + N)
    x = rng.randn(M, K).astype(np.float32)
    W = (rng.randn(K, N) * 0.05).astype(np.float32)
    W.ravel()[:: 7] = 0.0
    return x, W, rng.randn(N).astype(np.float32)


def _bound(x, K, N, alpha, y64):
    # x in 24 bits of its row's largest: K * max|x| * 2^-23 / 2 per output, times alpha; conversion, alpha and bias are
    # three roundings, alpha itself is good to 2e-6 (a sum of K magnitudes)
    return K * np.abs(x).max(axis=1, keepdims=True) * 2.0 ** -23 * alpha + (3 * 2.0 ** -24 + 2e-6) * np.abs(y64) + 1e-6


@pytest.mark.parametrize("M,K,N", SMALL + LARGE)
@pytest.mark.parametrize("zero_to", [1.0, -1.0, 0.0])
def test_against_the_oracle_and_float64(M, K, N, zero_to):
    x, W, b = _case(M, K, N)
    dev = torch.device("cuda:0")
    kernels.init(0)
    xd, Wd, bd = (torch.from_numpy(v).to(dev) for v in (x, W, b))
    _, ref_Wb, ref_alpha = oracle.binary_weight_affine(x[:1], W, b, zero_to)
    y, Wb, alpha = kernels.binary_weight_affine(xd, Wd, bd, zero_to)
    assert bits_equal(to_np(Wb), ref_Wb)
    np.testing.assert_allclose(to_np(alpha), ref_alpha, rtol=2e-6)
    a64 = np.abs(W.astype(np.float64)).mean(0)
    y64 = x.astype(np.float64) @ ref_Wb.astype(np.float64)
    assert (np.abs(to_np(y) - (y64 * a64 + b)) <= _bound(x, K, N, a64, y64 * a64) + 2.0 ** -24 * np.abs(b)).all()
    yc, Wbc = kernels.binary_connect_affine(xd, Wd, None, zero_to)
    assert bits_equal(to_np(Wbc), ref_Wb)
    assert (np.abs(to_np(yc) - y64) <= _bound(x, K, N, 1.0, y64)).all()


@pytest.mark.parametrize("M,K,N", [(33, 100, 130), (40, 600, 70)])
def test_rows_with_a_non_finite_value(M, K, N):
    x, W, b = _case(M, K, N)
    clean, _, _ = kernels.binary_weight_affine(torch.from_numpy(x).cuda(), torch.from_numpy(W).cuda(),
                                               torch.from_numpy(b).cuda())
    x[3, 7], x[3, 50] = np.inf, np.inf
    x[M - 1, K - 1] = -np.inf
    x[5, 0] = np.nan
    with np.errstate(invalid="ignore"):
        ref, _, _ = oracle.binary_weight_affine(x, W, b, 1.0)
    y = to_np(kernels.binary_weight_affine(torch.from_numpy(x).cuda(), torch.from_numpy(W).cuda(),
                                           torch.from_numpy(b).cuda())[0])
    for f in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(f(y), f(ref))
    rows = np.isfinite(ref).all(axis=1)
    assert not rows[[3, 5, M - 1]].any() and rows.sum() == M - 3
    assert bits_equal(y[rows], to_np(clean)[rows])


def test_signs_in_the_place_of_the_weights():
    """Wb may be W itself (the walk reads an element before it writes it)."""
    x, W, b = _case(40, 70, 90)
    Wd = torch.from_numpy(W).cuda()
    y0, Wb, alpha0 = kernels.binary_weight_affine(torch.from_numpy(x).cuda(), Wd, torch.from_numpy(b).cuda())
    y1, Wb1, alpha1 = kernels.binary_weight_affine(torch.from_numpy(x).cuda(), Wd, torch.from_numpy(b).cuda(), Wb=Wd)
    assert Wb1.data_ptr() == Wd.data_ptr() and torch.equal(Wb1, Wb)
    assert torch.allclose(y1, y0, rtol=0, atol=2e-6 * float(y0.abs().max()))
