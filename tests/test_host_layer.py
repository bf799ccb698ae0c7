"""The nbla-compatible host layer on the CPU: contexts, registries, SyncedArray head tracking, the caching allocator
and the error behaviour of the function registry.  No GPU is touched (functions are created and set up, never run)."""
import ctypes

import numpy as np
import pytest

import nnabla_amd as nn
import nnabla_amd.functions as F
from nnabla_amd import _capi
from nnabla_amd.ext_utils import get_extension_context


def test_extension_context_and_array_classes():
    ctx = get_extension_context('hip', device_id='0')
    assert ctx.backend == ['hip:float', 'cpu:float'] and ctx.array_class == 'HipCachedArray' and ctx.device_id == '0'
    half = get_extension_context('hip', type_config='half')
    assert half.backend == ['hip:half', 'hip:float', 'cpu:float']
    with pytest.raises(ValueError):
        get_extension_context('hip', type_config='int8')
    with pytest.raises(ImportError):
        get_extension_context('cuda')
    from nnabla_amd import ext_hip
    assert ext_hip.array_classes() == ['HipCachedArray', 'HipArray']


def test_context_scope_nesting():
    base = nn.get_current_context()
    ctx = get_extension_context('hip')
    with nn.context_scope(ctx):
        assert nn.get_current_context() is ctx
        with nn.context_scope(nn.Context(['cpu:float'], 'CpuArray', '0')):
            assert nn.get_current_context().array_class == 'CpuArray'
        assert nn.get_current_context() is ctx
    assert nn.get_current_context() is base


def test_variable_host_roundtrip_and_dtypes():
    x = nn.Variable((2, 3))
    assert np.array_equal(x.d, np.zeros((2, 3), np.float32))       # a fresh array reads as zeros
    x.d = np.arange(6).reshape(2, 3)
    assert x.d.dtype == np.float32 and np.array_equal(x.d, np.arange(6, dtype=np.float32).reshape(2, 3))
    assert x.head_array_class == 'CpuCachedArray'
    x.fill(2.5)
    assert np.all(x.d == 2.5)
    x.zero()
    assert np.all(x.d == 0)
    i = nn.Variable((4,))
    i.set_data([1, 0, 1, 1], np.int32)
    assert i.d.dtype == np.int32 and i.d.tolist() == [1, 0, 1, 1]
    v = nn.Variable.from_numpy_array(np.ones((2, 2), np.float32) * 3)
    r = v.reshape((4,))
    assert np.array_equal(r.d, np.full(4, 3, np.float32))
    r.d = [1, 2, 3, 4]
    assert np.array_equal(v.d, np.array([[1, 2], [3, 4]], np.float32))   # views share storage
    with pytest.raises(ValueError):
        v.reset_shape((5,))
    v.reset_shape((5,), force=True)
    assert v.shape == (5,)


def test_registry_lookup_and_fallback_errors():
    x = nn.Variable((2, 3))
    # cpu context: this build registers no cpu:float implementation (function_registry.hpp:57-72 message)
    with pytest.raises(ValueError) as ei:
        F.fixed_point_quantize(x)
    assert "could not be found in [hip:float]" in str(ei.value)
    # the hip context resolves through the ordered backend list, including the 'half' config
    for ctx in (get_extension_context('hip'), get_extension_context('hip', type_config='half')):
        with nn.context_scope(ctx):
            y = F.fixed_point_quantize(x)
        assert y.parent.name == 'FixedPointQuantize' and y.shape == (2, 3)
    with nn.context_scope(nn.Context(['cuda:float'], 'CudaArray', '0')):
        with pytest.raises(ValueError):
            F.pow2_quantize(x)


def test_quantize_flag_returns_input_untouched():
    x = nn.Variable((2, 3))
    assert F.fixed_point_quantize(x, quantize=False) is x
    assert F.pow2_quantize(x, quantize=False) is x
    q = nn.Variable((1, 1))
    assert F.min_max_quantize(x, q, q, q, q, quantize=False) is x


def test_setup_shape_inference_and_argument_checks():
    ctx = get_extension_context('hip')
    with nn.context_scope(ctx):
        x = nn.Variable((4, 3, 5, 6))
        # affine with base_axis folding and tensor weights
        w = nn.Variable((30, 7, 2))
        y = F.binary_connect_affine(x, w, nn.Variable((30, 7, 2)), base_axis=2)
        assert y.shape == (4, 3, 7, 2)
        y = F.binary_weight_affine(x, w, nn.Variable((30, 7, 2)), nn.Variable((14,)), base_axis=-2)
        assert y.shape == (4, 3, 7, 2)
        with pytest.raises(ValueError):
            F.binary_weight_affine(x, w, nn.Variable((30, 7, 2)), nn.Variable((13,)), base_axis=2)   # alpha size
        with pytest.raises(ValueError):
            F.binary_connect_affine(x, nn.Variable((31, 7)), nn.Variable((31, 7)), base_axis=2)      # K mismatch
        # convolution geometry (convolution.cpp:97-98)
        wc = nn.Variable((8, 3, 3, 2))
        y = F.binary_weight_convolution(x, wc, nn.Variable((8, 3, 3, 2)), nn.Variable((8,)), pad=(1, 0),
                                        stride=(2, 1), dilation=(1, 2))
        assert y.shape == (4, 8, 3, 4)
        y = F.inq_convolution(x, wc, nn.Variable((8, 3, 3, 2)), nn.Variable((8,)))
        assert y.shape == (4, 8, 3, 5)
        with pytest.raises(ValueError):
            F.binary_connect_convolution(x, nn.Variable((8, 2, 3, 3)), nn.Variable((8, 2, 3, 3)))     # channels
        with pytest.raises(ValueError):
            F.binary_connect_convolution(x, nn.Variable((8, 3, 9, 9)), nn.Variable((8, 3, 9, 9)))     # kernel too big
        # quantizer argument checks are raised at setup, as in the reference
        with pytest.raises(ValueError):
            F.fixed_point_quantize(x, n=1, sign=True)
        with pytest.raises(ValueError):
            F.pow2_quantize(x, n=2, sign=True, with_zero=True)
        q = nn.Variable((1, 3, 1, 1))
        assert F.min_max_quantize(x, q, nn.Variable((1, 3, 1, 1)), nn.Variable((1, 3, 1, 1)),
                                  nn.Variable((1, 3, 1, 1))).shape == x.shape
        with pytest.raises(ValueError):
            F.min_max_quantize(x, nn.Variable((1, 2, 1, 1)), nn.Variable((1, 2, 1, 1)), nn.Variable((1, 2, 1, 1)),
                               nn.Variable((1, 2, 1, 1)))
        with pytest.raises(ValueError):
            F.inq_affine(nn.Variable((2, 6)), nn.Variable((6, 4)), nn.Variable((6, 4)), selection_algorithm='best')
        with pytest.raises(ValueError):
            F.inq_affine(nn.Variable((2, 6)), nn.Variable((6, 4)), nn.Variable((6, 5)))


def test_outputs_argument_reuses_the_given_variable():
    with nn.context_scope(get_extension_context('hip')):
        x = nn.Variable((2, 3))
        out = nn.Variable((2, 3))
        y = F.fixed_point_quantize(x, outputs=[out])
        assert y is out and out.parent is not None


def test_caching_allocator_reuses_and_merges_host_blocks():
    """CachingAllocatorWithBuckets through the host backend: rounding to 512 B, 1 MiB slabs for small requests,
    reuse after free, release of whole cached blocks."""
    L = _capi.lib()
    before = L.nblac_allocator_bytes(b"cpu", b"", 1)
    vs = []
    for _ in range(3):
        v = nn.Variable((100,))          # 400 B -> one 512 B piece of a 1 MiB slab
        v.d = 1.0
        vs.append(v)
    grown = L.nblac_allocator_bytes(b"cpu", b"", 1) - before
    assert grown in (0, 1 << 20)         # at most one new slab, whatever was cached before
    big = nn.Variable((1 << 20,))        # 4 MiB -> large pool, rounded to 128 KiB
    big.d = 0.0
    assert L.nblac_allocator_bytes(b"cpu", b"", 1) - before >= 4 << 20
    level = L.nblac_allocator_bytes(b"cpu", b"", 1)
    del big
    big2 = nn.Variable((1 << 20,))
    big2.d = 0.0
    assert L.nblac_allocator_bytes(b"cpu", b"", 1) == level   # the freed block was reused, not re-allocated


def test_a_graph_hands_its_functions_over_without_new_types(monkeypatch):
    """Variable.forward gives the host library every function with its inputs and outputs in order, and makes no ctypes
    array types for it: those are gone after a garbage collection, and a new graph's first launch waited for them to be made
    again."""
    import gc
    with nn.context_scope(get_extension_context('hip')):
        x, w = nn.Variable((3, 4)), nn.Variable((4, 4))
        h = F.binary_connect_affine(F.relu(x), w, nn.Variable((4, 4)))
        for _ in range(13):
            h = F.relu(h)
        h = F.add2(h, x)
    seen = {}

    class Host(object):
        @staticmethod
        def nblac_functions_forward(n, functions, num_inputs, inputs, num_outputs, outputs, pairs):
            words = lambda p, count: list((ctypes.c_uint64 * count).from_address(p.value))
            ints = lambda p: list((ctypes.c_int32 * n).from_address(p.value))
            seen.update(functions=words(functions, n), num_inputs=ints(num_inputs), num_outputs=ints(num_outputs))
            seen.update(inputs=words(inputs, sum(seen["num_inputs"])), outputs=words(outputs, sum(seen["num_outputs"])))
            return 0

    array_types = lambda: {id(o) for o in gc.get_objects() if type(o) is type(ctypes.Array)}
    calls = []
    monkeypatch.setattr(_capi, "lib", lambda: type("Counts", (), {
        "nblac_functions_forward": staticmethod(lambda *a: calls.append(a) or 0)}))
    gc.collect()
    before = array_types()
    h.forward()
    assert array_types() <= before and len(calls) == 1
    monkeypatch.setattr(_capi, "lib", lambda: Host)
    h.forward()
    nodes = h._function_order()
    assert seen["functions"] == [n.function._h.value for n in nodes] and len(nodes) == 16
    assert seen["num_inputs"] == [len(n.inputs) for n in nodes] and seen["num_outputs"] == [len(n.outputs) for n in nodes]
    assert seen["inputs"] == [v._h.value for n in nodes for v in n.inputs]
    assert seen["outputs"] == [v._h.value for n in nodes for v in n.outputs]
