"""ReLU and the FixedPointQuantize behind it in one launch (nbla_hip_relu_fixed_point_quantize_f32), as a call and as a
graph's forward pass takes it: the bits of the two functions one after the other, ReLU's own result included."""
import ctypes

import numpy as np
import pytest
import torch

import nnabla_amd as nn
import nnabla_amd.functions as F
from nnabla_amd import kernels
from nnabla_amd.ext_utils import get_extension_context
from nnabla_amd.function import forward_nodes
from util import bits_equal, to_np

pytestmark = pytest.mark.gpu


def _values(size):
    x = (np.random.RandomState(size).randn(size) * 3).astype(np.float32)
    x[: min(size, 8)] = np.array([np.nan, np.inf, -np.inf, -0.0, 0.0, 1e-45, -1e-45, 3e38], np.float32)[: min(size, 8)]
    return torch.from_numpy(x).cuda()


def _pair(x, mid, y, sign, n, delta):
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    kernels.check(kernels.lib().nbla_hip_relu_fixed_point_quantize_f32(
        p(x), p(mid), p(y), ctypes.c_size_t(x.numel()), int(sign), n, ctypes.c_float(delta), None))
    torch.cuda.synchronize()


@pytest.mark.parametrize("size", [1, 3, 4, 1023, 1024, 1027, 300001])
@pytest.mark.parametrize("sign,n,delta", [(True, 8, 2.0 ** -4), (False, 3, 0.3)])
@pytest.mark.parametrize("shift", [0, 1])
def test_the_bits_of_both_functions(size, sign, n, delta, shift):
    kernels.init(0)
    x = _values(size + shift)[shift:]
    mid, y = torch.empty_like(x), torch.empty_like(x)
    torch.cuda.synchronize()
    relu = torch.where(x > 0, x, torch.zeros_like(x))
    want = kernels.fixed_point_quantize(relu, sign, n, delta)
    _pair(x, mid, y, sign, n, delta)
    assert bits_equal(to_np(mid), to_np(relu)) and bits_equal(to_np(y), to_np(want))
    x2 = x.clone()
    torch.cuda.synchronize()
    _pair(x2, x2, y, sign, n, delta)  # ReLU in place
    assert bits_equal(to_np(x2), to_np(relu)) and bits_equal(to_np(y), to_np(want))
    x2 = x.clone()
    torch.cuda.synchronize()
    _pair(x2, mid, x2, sign, n, delta)  # the quantizer's result in the place of x
    assert bits_equal(to_np(mid), to_np(relu)) and bits_equal(to_np(x2), to_np(want))
    _pair(x, y, y, sign, n, delta)  # both results in one place: the quantizer's stays
    assert bits_equal(to_np(y), to_np(want))
    x2 = x.clone()
    torch.cuda.synchronize()
    _pair(x2, x2, x2, sign, n, delta)  # and that the place of x
    assert bits_equal(to_np(x2), to_np(want))


def test_no_place_for_relu_is_refused():
    kernels.init(0)
    x = _values(16)
    p = ctypes.c_void_p(x.data_ptr())
    with pytest.raises(kernels.KernelError):
        kernels.check(kernels.lib().nbla_hip_relu_fixed_point_quantize_f32(p, None, p, ctypes.c_size_t(16), 1, 8,
                                                                         ctypes.c_float(0.1), None))


@pytest.mark.parametrize("shape", [(5, 7), (64, 130)])
def test_a_graph_gives_what_its_functions_give_one_by_one(shape):
    rng = np.random.RandomState(3)
    with nn.context_scope(get_extension_context("hip")):
        x = nn.Variable(shape)
        x.d = rng.randn(*shape).astype(np.float32) * 3
        r = F.relu(x)
        q = F.fixed_point_quantize(r, True, 8, 2 ** -4)
        r2 = F.relu(q)                  # another pair, on the first one's result
        q2 = F.fixed_point_quantize(r2, False, 4, 0.25)
        z = F.add2(q2, r)               # ReLU's result is used elsewhere too
    nodes = z._function_order()
    assert forward_nodes(nodes) == 2  # both pairs ran as one launch each
    got = [v.d.copy() for v in (r, q, r2, q2, z)]
    for node in z._function_order():
        node.forward()
    for g, v in zip(got, (r, q, r2, q2, z)):
        assert bits_equal(g, v.d)
    x.d = -x.d  # new values through the same graph
    z.forward()
    assert np.array_equal(r.d, np.maximum(x.d, 0)) and not np.array_equal(r.d, got[0])


def test_where_the_pair_does_not_hold_the_functions_run_one_by_one():
    """A quantizer that writes into ReLU's own array, one that reads another variable than ReLU's result, one that comes
    later in the order, and a ReLU that no quantizer follows."""
    rng = np.random.RandomState(4)
    with nn.context_scope(get_extension_context("hip")):
        x = nn.Variable((33, 9))
        x.d = rng.randn(33, 9).astype(np.float32) * 3
        r = F.relu(x)
        q = F.fixed_point_quantize(r, True, 8, 2 ** -4, outputs=[r.data])
        assert forward_nodes(q._function_order()) == 0
        assert bits_equal(q.d, np.minimum(np.round(np.maximum(x.d, 0) * 16) / 16, np.float32(127 / 16)))
        a, b = F.relu(x), F.fixed_point_quantize(x, True, 8, 2 ** -4)
        assert forward_nodes(F.add2(a, b)._function_order()) == 0
        a = F.relu(x)
        z = F.add2(F.relu(a), F.fixed_point_quantize(a, True, 8, 2 ** -4))
        order = [n.name for n in z._function_order()]
        assert order[1] == order[0] and forward_nodes(z._function_order()) == 0
