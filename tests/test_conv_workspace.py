"""What the convolutions' backward asks for in scratch memory, from the shapes alone (no device is touched)."""
import pytest
import torch

from nnabla_amd import kernels


def _bytes(xs, O, k, stride=1, group=1):
    geom, _ = kernels._conv_geometry(torch.empty(xs, device="meta"), torch.empty(O, xs[1] // group, k, k, device="meta"),
                                     (k // 2,) * 2, (stride,) * 2, (1, 1), group)
    return kernels.lib().nbla_hip_convolution_backward_workspace_bytes(*geom)


@pytest.mark.parametrize("xs,O,k,stride", [((32, 64, 56, 56), 64, 3, 1), ((64, 128, 28, 28), 128, 3, 1),
                                           ((16, 64, 56, 56), 128, 5, 1)])
def test_no_room_for_an_unfolded_matrix_that_no_gradient_forms(xs, O, k, stride):
    unfolded = 4 * xs[0] * (xs[2] // stride) * (xs[3] // stride) * xs[1] * k * k
    assert _bytes(xs, O, k, stride) < unfolded // 2


@pytest.mark.parametrize("xs,O,k,stride", [((32, 512, 14, 14), 512, 5, 1), ((64, 512, 28, 28), 512, 3, 1)])
def test_the_forms_share_the_memory(xs, O, k, stride):
    """The unfolded matrix, its digits (three bytes an element) and those of the gradient, and not the other forms' on top."""
    m, kg = xs[0] * (xs[2] // stride) * (xs[3] // stride), xs[1] * k * k
    assert _bytes(xs, O, k, stride) < 1.05 * (4 * m * kg + 3 * m * kg + (4 + 3 + 3) * m * O + 64 * O * kg)
