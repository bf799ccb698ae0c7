"""Binary affine forward over a W whose rows start at any multiple of four bytes, around the number of column strips from
which neighbouring strips are dealt to one XCD, with rows of x that end inside a 128-bit load.  Sign(W) and alpha are
exact up to alpha's sum; x is rounded to 2^-23 of its row's largest, sums are exact and rounded once."""
import numpy as np
import pytest
import torch

from nnabla_amd import kernels
from util import to_np

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [1301, 1302, 1303])
@pytest.mark.parametrize("N", [1791, 1793, 2049, 2303])
def test_against_float64(K, N):
    kernels.init(0)
    M = 261
    rng = np.random.RandomState(K + N)
    x = rng.randn(M, K).astype(np.float32)
    W = rng.randn(K, N).astype(np.float32)
    b = rng.randn(N).astype(np.float32)
    y, Wb, al = kernels.binary_weight_affine(*(torch.from_numpy(v).cuda() for v in (x, W, b)))
    signs = np.where(W < 0, -1.0, 1.0)
    assert np.array_equal(to_np(Wb), signs.astype(np.float32))
    alpha = np.abs(W.astype(np.float64)).mean(0)
    assert (np.abs(to_np(al) - alpha) <= alpha * K * 2.0 ** -24).all()
    ref = x.astype(np.float64) @ signs
    bound = K * 2.0 ** -23 * np.abs(x).max(1)[:, None] + 2.0 ** -23 * np.abs(ref)
    got = (to_np(y).astype(np.float64) - b) / to_np(al)
    assert (np.abs(got - ref) <= bound + 2.0 ** -22 * (np.abs(ref) + np.abs(b) / to_np(al))).all()
