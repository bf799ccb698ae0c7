"""Up to sixteen rows through BinaryWeightAffine / BinaryConnectAffine in one walk over W (csrc/kernels/binary_small_m.hip):
every number of rows per wavefront that a size gets, numbers of columns that are no multiple of four (a row of W starts at
any multiple of four bytes, the last quad is taken apart), one strip of columns and several, Wb in the place of W, and the
folding of one to more slabs than are folded at a time, against float64."""
import numpy as np
import pytest
import torch

import oracle
from nnabla_amd import kernels
from util import bits_equal, to_np

pytestmark = pytest.mark.gpu

# rows, inputs, outputs: W large enough that the one-launch form leaves it (more than 1024 inputs), or N a multiple of four
SIZES = [(1, 1, 4), (1, 31, 8), (3, 33, 1000), (16, 100, 260), (1, 1025, 5), (2, 1030, 255), (5, 1500, 257), (9, 1027, 1023),
         (16, 2049, 66), (12, 300, 3000), (7, 4099, 514), (4, 1100, 4099), (1, 4095, 11007), (1, 5000, 12),
         # three, four and five slabs of 32 rows: the sums of up to four need no fold
         (2, 96, 8), (4, 128, 300), (4, 129, 300), (8, 160, 261)]


@pytest.mark.parametrize("M,K,N", SIZES)
def test_against_float64(M, K, N):
    kernels.init(0)
    rng = np.random.RandomState(M + K + N)
    x = rng.randn(M, K).astype(np.float32)
    W = (rng.randn(K, N) * 0.05).astype(np.float32)
    W.ravel()[::7] = 0.0
    b = rng.randn(N).astype(np.float32)
    xd, Wd, bd = (torch.from_numpy(v).cuda() for v in (x, W, b))
    y, Wb, alpha = kernels.binary_weight_affine(xd, Wd, bd)
    ref_Wb = np.where(W > 0, 1.0, np.where(W < 0, -1.0, 1.0)).astype(np.float32)
    assert bits_equal(to_np(Wb), ref_Wb)
    a64 = np.abs(W.astype(np.float64)).mean(0)
    np.testing.assert_allclose(to_np(alpha), a64, rtol=2e-6)
    # (every size here takes the walk) sums of K terms in chains of at most 64 + 4 + 128 / 4 + 8
    y64, terms = x.astype(np.float64) @ ref_Wb, np.abs(x.astype(np.float64)).sum(1, keepdims=True)
    bound = terms * 108 * 2.0 ** -24 * a64 + (3 * 2.0 ** -24 + 2e-6) * np.abs(y64 * a64) + 2.0 ** -23 * np.abs(b)
    assert (np.abs(to_np(y) - (y64 * a64 + b)) <= bound + 1e-7).all()
    yc, _ = kernels.binary_connect_affine(xd, Wd, None)
    assert (np.abs(to_np(yc) - y64) <= terms * 108 * 2.0 ** -24 + 2.0 ** -23 * np.abs(y64)).all()
    y2, Wb2, _ = kernels.binary_weight_affine(xd, Wd, bd, Wb=Wd)  # in place: W is read before it is written
    assert Wb2.data_ptr() == Wd.data_ptr() and torch.equal(Wb2, Wb)
    assert torch.allclose(y2, y, rtol=0, atol=4e-6 * float(y.abs().max()) + 1e-6)


# one to five and nine slabs of 64 rows on the matrix cores
@pytest.mark.parametrize("M,K,N", [(9, 16, 8), (18, 64, 20), (33, 80, 260), (64, 192, 2608), (17, 256, 264), (64, 272, 300),
                                   (40, 560, 12)])
def test_few_slabs_on_the_matrix_cores(M, K, N):
    kernels.init(0)
    gen = torch.Generator(device="cuda").manual_seed(M + K + N)
    x, W = torch.randn(M, K, generator=gen, device="cuda"), torch.randn(K, N, generator=gen, device="cuda")
    b = torch.randn(N, generator=gen, device="cuda")
    y, Wb, alpha = kernels.binary_weight_affine(x, W, b)
    a64, terms = W.double().abs().mean(0), x.double().abs().sum(1, keepdim=True)
    ref = (x.double() @ Wb.double()) * a64 + b
    bound = terms * (K + 16) * 2.0 ** -24 * a64 + 4e-6 * ref.abs() + 2.0 ** -23 * b.abs()
    assert torch.equal(Wb, torch.where(W < 0, -1.0, 1.0)) and bool((alpha.double() - a64).abs().le(2e-6 * a64).all())
    assert bool(((y.double() - ref).abs() <= bound + 1e-7).all())


@pytest.mark.parametrize("M,K,N", [(5, 1500, 3001), (16, 4099, 4099)])
@pytest.mark.parametrize("draw", ["normal", "relu", "uniform", "outliers"])
def test_sums_of_random_signs_are_as_near_as_those_of_digits_were(M, K, N, draw):
    """Unaligned rows of W went through exact sums of 24-bit digits before, 1.5e-7 and more off float64 (relative 2-norm) at
    such sizes.  Here a chain of n additions passes through partial sums that grow like a random walk's, each rounded by
    2^-24 / sqrt(3) of itself on average: 2^-24 sqrt(n / 6) of the result, for chains of 64 + 4 + 8 + 8."""
    kernels.init(0)
    gen = torch.Generator(device="cuda").manual_seed(M + K + N)
    x, W = torch.randn(M, K, generator=gen, device="cuda"), torch.randn(K, N, generator=gen, device="cuda")
    if draw == "relu":
        x = x.clamp(min=0)
    elif draw == "uniform":
        x = torch.rand(M, K, generator=gen, device="cuda")
    elif draw == "outliers":
        x[:, ::97] *= 100
    y, Wb = kernels.binary_connect_affine(x, W, None)
    ref = x.double() @ Wb.double()
    assert float((y.double() - ref).norm()) <= 2.0 ** -24 * (84 / 6) ** 0.5 * float(ref.norm())


def test_non_finite_values_reach_the_outputs_they_meet():
    kernels.init(0)
    rng = np.random.RandomState(5)
    x = rng.randn(3, 1100).astype(np.float32)
    W = (rng.randn(1100, 1001) * 0.05).astype(np.float32)
    x[0, 3], x[0, 900], x[2, 1099] = np.inf, np.inf, np.nan
    with np.errstate(invalid="ignore"):
        ref, _, _ = oracle.binary_weight_affine(x, W, None, 1.0)
    y = to_np(kernels.binary_weight_affine(torch.from_numpy(x).cuda(), torch.from_numpy(W).cuda())[0])
    for f in (np.isnan, np.isposinf, np.isneginf):
        assert np.array_equal(f(y), f(ref))
