"""The input gradient of a small binary layer in one launch (csrc/kernels/gemm_small.hip with signs): extents at and one
past its tiles, Sign(0), with and without alpha, sums added to what is there, magnitudes that bf16 parts cannot hold and
non-finite values, against float64."""
import numpy as np
import pytest
import torch

from nnabla_amd import kernels
from util import to_np

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (2, 65, 33), (32, 64, 32), (33, 63, 31), (20, 250, 250), (65, 64, 257), (100, 70, 513), (40, 3, 1025),
         (1000, 260, 96)]


def _case(M, K, N):
    rng = np.random.RandomState(M + K + N)
    W = (rng.randn(K, N) * 0.05).astype(np.float32)
    W.ravel()[::5] = 0.0
    W.ravel()[3::11] *= -0.0
    return rng.randn(M, N).astype(np.float32), W, (rng.rand(N) + 0.1).astype(np.float32)


def _ref(dy, W, alpha, zero_to):
    s = np.where(W > 0, 1.0, np.where(W < 0, -1.0, zero_to))
    a = dy.astype(np.float64) if alpha is None else (dy * alpha).astype(np.float64)  # (rounded once, as it is there)
    return a, s.T


@pytest.mark.parametrize("M,K,N", SIZES)
@pytest.mark.parametrize("zero_to", [1.0, -1.0, 0.0])
@pytest.mark.parametrize("scaled", [False, True])
def test_against_float64(M, K, N, zero_to, scaled):
    kernels.init(0)
    dy, W, alpha = _case(M, K, N)
    a, s = _ref(dy, W, alpha if scaled else None, zero_to)
    args = [torch.from_numpy(v).cuda() for v in (dy, np.zeros((M, K), np.float32), W, np.sign(W))]
    al = torch.from_numpy(alpha).cuda() if scaled else None
    dx = kernels.binary_affine_backward(*args, al, zero_to, want=(True, False, False))[0]
    # terms exact; sums of N of them by 16 in fp32 over eight wavefronts, then in double
    bound = (np.abs(a) @ np.abs(s)) * 2.0 ** -24 * (N / 128.0 + 6) + 2.0 ** -24 * np.abs(a @ s)
    assert (np.abs(to_np(dx) - a @ s) <= bound).all()
    old = torch.full((M, K), 3.0, device="cuda")
    kernels.binary_affine_backward(*args, al, zero_to, dx=old, want=(True, False, False))
    assert (np.abs(to_np(old) - (a @ s + 3.0)) <= bound + 2.0 ** -23 * (3.0 + np.abs(a @ s))).all()


def test_extreme_and_non_finite_values():
    kernels.init(0)
    dy, W, alpha = _case(40, 70, 100)
    dy[3] *= np.float32(1e-38)
    dy[4] *= np.float32(1e36)
    dy[7, 5], dy[8, 9], dy[9, 0] = np.inf, np.nan, -np.inf
    W[5, 50], W[6, 51] = np.nan, np.inf  # Sign(NaN) = Sign(0)
    with np.errstate(invalid="ignore", over="ignore"):
        a, s = _ref(dy, W, alpha, 1.0)
        ref = a @ s
        terms = np.abs(a) @ np.abs(s)
    args = [torch.from_numpy(v).cuda() for v in (dy, np.zeros((40, 70), np.float32), W, np.sign(W), alpha)]
    dx = to_np(kernels.binary_affine_backward(*args, want=(True, False, False))[0])
    for f in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(f(dx), f(ref))
    fin = np.isfinite(ref)
    assert (np.abs(dx - ref)[fin] <= (terms * 2.0 ** -21)[fin] + 2.0 ** -149).all()


@pytest.mark.parametrize("M,K,N", [(20, 250, 250), (300, 3000, 2000)])  # in one launch, and by the bit-weight product
@pytest.mark.parametrize("zero_to", [0.0, 0.5])
def test_without_the_signs_it_is_refused_at_every_size(M, K, N, zero_to):
    """Sign(0) that is neither +1 nor -1 needs the forward's signs for dx, whichever form the size takes, and dx is not
    touched; the weights' gradient alone needs none."""
    kernels.init(0)
    dy, W, alpha = (torch.from_numpy(v).cuda() for v in _case(M, K, N))
    x, dx = torch.zeros(M, K, device="cuda"), torch.full((M, K), 3.0, device="cuda")
    with pytest.raises(kernels.KernelError):
        kernels.binary_affine_backward(dy, x, W, None, alpha, zero_to, dx=dx, want=(True, False, False))
    assert bool((dx == 3.0).all())
    kernels.binary_affine_backward(dy, x, W, None, alpha, zero_to, want=(False, True, True))
