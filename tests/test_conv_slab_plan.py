"""The slab convolution's host-side sizing against a brute-force walk over every window and tap.

The kernel keeps, per block, the input positions [lo, hi] of one flattened input plane in LDS, lo / hi being the
smallest window origin and the largest origin plus the last tap's offset over the block's windows (clamped to the
plane).  The host sizes the LDS for the longest such run from the ends of each block and of the output rows inside
it only.  Here every window of every block is visited: the run must hold every tap that lies inside the input, and
the plan's capacity must equal the longest run exactly (the kernel's own clamp to the capacity then never acts).
No device is touched.
"""
import itertools

import numpy as np
import pytest

from nnabla_amd import kernels


def brute_force(in_sp, kernel, pad, stride, dil, tile_rows):
    nd = len(in_sp)
    in3 = [1] * (3 - nd) + list(in_sp)
    k3 = [1] * (3 - nd) + list(kernel)
    p3 = [0] * (3 - nd) + list(pad)
    s3 = [1] * (3 - nd) + list(stride)
    d3 = [1] * (3 - nd) + list(dil)
    out3 = [(in3[i] + 2 * p3[i] - (d3[i] * (k3[i] - 1) + 1)) // s3[i] + 1 for i in range(3)]
    plane = in3[0] * in3[1] * in3[2]
    n_out = out3[0] * out3[1] * out3[2]
    o = np.arange(n_out)
    o2, o1, o0 = o % out3[2], (o // out3[2]) % out3[1], o // (out3[2] * out3[1])
    b = [o0 * s3[0] - p3[0], o1 * s3[1] - p3[1], o2 * s3[2] - p3[2]]
    origin = (b[0] * in3[1] + b[1]) * in3[2] + b[2]
    last = ((k3[0] - 1) * d3[0] * in3[1] + (k3[1] - 1) * d3[1]) * in3[2] + (k3[2] - 1) * d3[2]
    longest, uncovered = 1, 0
    tiles = -(-n_out // tile_rows)
    for t in range(tiles):
        sel = slice(t * tile_rows, min((t + 1) * tile_rows, n_out))
        lo = int(np.clip(origin[sel].min(), 0, plane - 1))
        hi = int(np.clip(origin[sel].max() + last, 0, plane - 1))
        longest = max(longest, hi - lo + 1)
        # every tap of every window of the tile that lies inside the input
        for t0, t1, t2 in itertools.product(range(k3[0]), range(k3[1]), range(k3[2])):
            c = [b[0][sel] + t0 * d3[0], b[1][sel] + t1 * d3[1], b[2][sel] + t2 * d3[2]]
            inside = np.ones(c[0].shape, bool)
            for i in range(3):
                inside &= (c[i] >= 0) & (c[i] < in3[i])
            pos = (c[0] * in3[1] + c[1]) * in3[2] + c[2]
            uncovered += int(((pos[inside] < lo) | (pos[inside] > hi)).sum())
    return out3, tiles, longest, uncovered


def geometries():
    rng = np.random.RandomState(20240)
    fixed = [
        ((14, 14), (3, 3), (1, 1), (1, 1), (1, 1)), ((56, 56), (3, 3), (1, 1), (1, 1), (1, 1)),
        ((28, 28), (3, 3), (1, 1), (2, 2), (1, 1)), ((7, 7), (3, 3), (1, 1), (1, 1), (1, 1)),
        ((5, 70), (3, 3), (1, 1), (1, 1), (1, 1)), ((6, 6), (1, 1), (0, 0), (1, 1), (1, 1)),
        ((9, 11), (3, 2), (2, 0), (1, 2), (2, 1)), ((40,), (5,), (2,), (1,), (1,)), ((33,), (3,), (0,), (2,), (3,)),
        ((4, 6, 5), (2, 3, 2), (1, 1, 0), (1, 1, 1), (1, 1, 1)), ((3, 9, 9), (3, 3, 3), (1, 1, 1), (1, 2, 1), (1, 1, 2)),
        ((14, 14), (3, 3), (4, 4), (1, 1), (1, 1)),  # padding wider than the kernel: windows wholly outside
    ]
    for g in fixed:
        yield g
    for _ in range(300):
        nd = int(rng.randint(1, 4))
        in_sp = tuple(int(v) for v in rng.randint(1, [9, 20, 40][3 - nd:][0] + 1, size=nd))
        in_sp = tuple(max(v, 1) for v in in_sp)
        kernel = tuple(int(v) for v in rng.randint(1, 4, size=nd))
        dil = tuple(int(v) for v in rng.randint(1, 3, size=nd))
        stride = tuple(int(v) for v in rng.randint(1, 4, size=nd))
        pad = tuple(int(v) for v in rng.randint(0, 4, size=nd))
        if any(in_sp[i] + 2 * pad[i] < dil[i] * (kernel[i] - 1) + 1 for i in range(nd)):
            continue
        yield in_sp, kernel, pad, stride, dil


def test_the_plan_holds_every_tap_and_is_tight():
    planned, widths, filled_in_parts = 0, {32: 0, 64: 0, 128: 0}, 0
    for in_sp, kernel, pad, stride, dil in geometries():
        # channel counts and batches for which every tile of the kernel is the cheapest somewhere
        for outer, C, O in ((2, 32, 64), (2, 96, 64), (2, 32, 300), (64, 32, 200), (64, 96, 64), (64, 256, 128), (16, 700, 65)):
            plan = kernels.binary_convolution_slab_plan(outer, C, in_sp, O, kernel, pad, stride, dil, 1)
            if plan is None:
                continue
            planned += 1
            out3, tiles, longest, uncovered = brute_force(in_sp, kernel, pad, stride, dil, plan["tile_rows"])
            what = "in %s k %s pad %s stride %s dil %s C %d" % (in_sp, kernel, pad, stride, dil, C)
            width = min(w for w in widths if plan["tile_rows"] <= w)
            widths[width] += 1
            assert plan["tiles_per_sample"] == tiles, what
            assert uncovered == 0, what
            assert plan["cap"] == longest, what
            # all channels of a position, or at least one tile of 32 of them at a time
            held = (plan["lds_bytes"] // (plan["cap"] + 1) - 16) // 128
            assert 1 <= held and plan["lds_bytes"] <= 156 * 1024, what
            filled_in_parts += held < -(-C // 32)
    assert planned >= 300 and min(widths.values()) >= 15 and filled_in_parts >= 30


@pytest.mark.parametrize("C,in_sp,expected", [
    (8, (14, 14), False),      # too few input channels per group
    (12, (27, 27), False),     # the same: fp32 on the vector units
    (16, (27, 27), True),      # as few as it takes, to few maps, however few the windows are
    (16, (8, 8), True),
    (40, (14, 14), True),      # 40 channels padded to 64
    (256, (14, 14), True),
    (1024, (14, 14), True),    # the channels under a block do not fit the LDS: some after the other
    (1024, (56, 56), False),   # the same, and gathering is estimated the cheaper for one sample
])
def test_which_geometries_take_the_form(C, in_sp, expected):
    plan = kernels.binary_convolution_slab_plan(1, C, in_sp, 64, (3, 3), (1, 1), (1, 1), (1, 1), 1)
    assert (plan is not None) == expected


@pytest.mark.parametrize("outer,C,in_sp,O,kernel,stride,expected", [
    (1, 23, (28, 28), 16, (3, 5), 1, True),         # 15 us against 86 of the fp32 kernel
    (1, 16, (8, 8), 8, (2, 2), 1, True),            # 12 against 19: the fewest windows
    (16, 23, (56, 56), 64, (2, 2), 1, True),        # 19 against 47
    (13, 20, (160, 160), 32, (7, 1), 1, False),     # 742 against 171: few channels and maps, many windows
    (70, 20, (112, 112), 8, (4, 1), 2, False),      # 99 against 49
    (134, 16, (80, 80), 16, (3, 2), 2, False),      # 92 against 48
])
def test_few_channels_to_few_maps_take_the_faster_form(outer, C, in_sp, O, kernel, stride, expected):
    pad = tuple(k // 2 for k in kernel)
    plan = kernels.binary_convolution_slab_plan(outer, C, in_sp, O, kernel, pad, (stride, stride), (1, 1), 1)
    assert (plan is not None) == expected


def test_whole_rows_of_the_output_map_per_block():
    # 14 x 14 outputs: two rows of 14 per block, seven blocks per sample
    plan = kernels.binary_convolution_slab_plan(32, 256, (14, 14), 256, (3, 3), (1, 1), (1, 1), (1, 1), 1)
    assert plan["tile_rows"] == 28 and plan["tiles_per_sample"] == 7
    # the run: two output rows' windows span four input rows, plus the position before the first row's first window
    # (origin one column to the left) and the one after the last window's last tap
    assert plan["cap"] == 4 * 14 + 2


def test_the_layers_of_a_network_do_not_plan_anew_on_every_call():
    """Forty geometries one after the other, as a training step asks for them: from the second round on an answer is a
    look-up (planning one of these anew takes 50 us and more)."""
    import time
    geometries = [(1, 64, (224, 224), 64 + 8 * i, (3, 3), (1, 1), (1, 1), (1, 1), 1) for i in range(40)]
    answers = [kernels.binary_convolution_slab_plan(*g) for g in geometries]
    best = 1.0
    for _ in range(5):
        t = time.perf_counter()
        again = [kernels.binary_convolution_slab_plan(*g) for g in geometries]
        best = min(best, (time.perf_counter() - t) / len(geometries))
        assert again == answers
    assert best < 30e-6
