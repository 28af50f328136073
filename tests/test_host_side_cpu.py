"""Host-side logic of the compiled libraries without a GPU: every case runs in a process of its own in which tests/hip_stub.c
stands in for the HIP runtime (streams, graphs and copies keep their order, kernels do nothing)."""
import ctypes as C
import os
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


# ---- the cases, each in its own process --------------------------------------------------------------------------------------
def inverted_residual_add_needs_equal_shapes():
    """The residual of hipq_inverted_residual_run is the block's input, read with the output's geometry: an add is taken only
    where the two are the same tensor shape, at stride 1 and with equal channels.  (The shapes without an add stay accepted.)"""
    import numpy as np
    from nart_amd import hipq

    def block(ci, ch, co, hw, stride):
        plans = []
        for C_, K, R, s, g, H in ((ci, ch, 1, 1, 1, hw), (ch, ch, 3, stride, ch, hw), (ch, co, 1, 1, 1, (hw - 1) // stride + 1)):
            w = np.full((K, C_ // g, R, R), 129, np.uint8)
            plans.append(hipq.Conv2d((1, C_, H, H), w, None, R // 2, s, g, 0.05, 9, 0.002, 128, 0.05, 9))
        plans[2].special(2)
        return plans
    x, y = np.zeros(1 << 16, np.uint8), np.zeros(1 << 16, np.uint8)  # never touched
    kernels = C.c_long.in_dll(STUB, "stub_kernels")
    for ci, ch, co, stride, same in ((24, 144, 24, 1, True), (16, 96, 24, 1, False), (24, 144, 16, 1, False), (24, 144, 24, 2, False),
                                     (30, 64, 32, 1, False), (32, 64, 30, 1, False)):
        plans = block(ci, ch, co, 14, stride)
        assert hipq.inverted_residual_fusable(*plans), (ci, ch, co, stride)
        for first in (False, True):
            assert hipq.inverted_residual_fusable(*plans, add=(first, 0.09, 10)) is same, (ci, ch, co, stride, first)
            before = kernels.value
            rc = hipq.lib().hipq_inverted_residual_run(*[p.handle for p in plans], x.ctypes.data, 0, 1, int(first), 0.09, 10, 8, y.ctypes.data,
                                                       None)
            assert (rc == 0) is same and kernels.value == before + same, (ci, ch, co, stride, first)


def a_chained_add_names_its_kernels():
    """hipq_conv2d_run_add_conv is one kernel from 20 000 pixels on, or where mode 2 asks for it, and two launches below that: the
    name says which, and as many kernels are launched."""
    import numpy as np
    from nart_amd import hipq
    kernels = C.c_long.in_dll(STUB, "stub_kernels")
    x = np.zeros(64, np.uint8).ctypes.data  # never touched
    for N, HW, mode, one in ((2, 24, 1, False), (2, 24, 2, True), (7, 56, 1, True), (6, 56, 1, False)):
        wide = hipq.Conv2d((N, 64, HW, HW), np.full((256, 64, 1, 1), 129, np.uint8), None, 0, 1, 1, 0.05, 9, 0.002, 128, 0.05, 9).special(mode)
        nxt = hipq.Conv2d((N, 256, HW, HW), np.full((64, 256, 1, 1), 129, np.uint8), None, 0, 1, 1, 0.09, 10, 0.002, 128, 0.05, 9)
        assert wide.add_conv_fusable(False, 0.04, 3, 0.09, 10, nxt)
        name = wide.add_conv_kernel(nxt)
        assert name == ("conv_mfma_i8_expand+add+conv" if one else wide.kernel_add + ", " + nxt.kernel), (N, HW, mode, name)
        before = kernels.value
        hipq.check(hipq.lib().hipq_conv2d_run_add_conv(wide.handle, x, x, 0, 0.04, 3, 0.09, 10, 8, x, nxt.handle, 0, x, None))
        assert kernels.value - before == (1 if one else 2), (N, HW, mode, name)


def a_plan_launches_the_kernel_that_it_names():
    """By the built-in rule, in every mode and with a named shape, without and with a residual: the name that a plan gives is that of the
    kernel it launches, and a shape that the caller names is run."""
    import random
    import re
    import numpy as np
    from nart_amd import hipq
    last = C.c_char_p.in_dll(STUB, "stub_last_kernel")
    x = np.zeros(64, np.uint8).ctypes.data  # never touched
    names = (("resident", "conv_resident_kernel"), ("stream", "conv_mfma_stream_kernel"), ("hreg3x3", "conv_hreg_kernel"), ("wreg", "conv_wreg_kernel"),
             ("rows3x3", "conv3x3_c64_rows_kernel"), ("expand", "conv_mfma_expand_kernel"), ("stem3x3", "conv_stem3x3_kernel"),
             ("pointwise", "conv_mfma_pointwise_kernel"), ("halo", "conv_mfma_halo_kernel"), ("k2", "conv_mfma_dma_k2_kernel"), ("c4", "conv_mfma_kernel"),
             ("", "conv_mfma_dma_kernel"))

    def check(plan, what):
        for name, add in ((plan.kernel, False), (plan.kernel_add, True)):
            if add:
                rc = hipq.lib().hipq_conv2d_run_add(plan.handle, x, x, 0, 0.05, 3, 0.09, 10, 8, x, None)
            else:
                rc = hipq.lib().hipq_conv2d_run(plan.handle, x, x, None, None)
            hipq.check(rc)
            assert re.match(r"conv_mfma_i8_", name), name
            want = [k for n, k in names if n in re.split(r"[_+]", name[len("conv_mfma_i8_"):]) or n == ""][0]
            assert want in last.value.decode(), (what, name, last.value.decode())
            seen.add(want)
    rng, seen = random.Random(6), set()
    layers = [(11, 256, 13, 256, 3, 1), (1, 128, 28, 128, 3, 1), (64, 256, 14, 256, 3, 2), (8, 64, 56, 64, 3, 1), (64, 64, 56, 256, 1, 1), (1, 64, 14, 96, 3, 1), (1, 64, 32, 256, 1, 1),
              (2, 3, 64, 32, 3, 2), (2, 3, 64, 64, 7, 2), (16, 512, 14, 512, 1, 1), (1, 480, 14, 64, 1, 1), (64, 2048, 7, 512, 1, 1), (1, 32, 20, 48, 1, 1)]
    while len(layers) < 120:
        N, C_, H, K, R, s = rng.choice((1, 2, 6, 16)), rng.choice((3, 20, 64, 96, 128, 256, 480)), rng.randrange(3, 40), rng.choice((16, 64, 135, 256, 512)), rng.choice((1, 3, 5)), rng.choice((1, 1, 2))
        layers.append((N, C_, H, K, R, s))
    for N, C_, H, K, R, s in layers:
        plan = hipq.Conv2d((N, C_, H, H), np.full((K, C_, R, R), 129, np.uint8), None, R // 2, s, 1, 0.05, 9, 0.002, rng.choice((128, 128, 128, 90)), 0.05, 9)
        for mode in (1, 0, 2, 3):
            plan.special(mode)
            check(plan, (N, C_, H, K, R, s, mode))
        plan.special(1)
        for shape in ((64, 32, 4), (16, 16, 4)):
            try:
                plan.stream(*shape)
            except hipq.HipqError:
                continue
            assert "stream_%dx%d" % shape[:2] in plan.kernel and "stream_%dx%d" % shape[:2] in plan.kernel_add, (plan.kernel, plan.kernel_add)
            check(plan, (N, C_, H, K, R, s, shape))
            plan.stream()
        if C_ > 4:
            plan.resident(32, 16, 1, 4)
            assert "resident_32x16" in plan.kernel and "resident_32x16" in plan.kernel_add
            check(plan, (N, C_, H, K, R, s, "resident"))
            plan.resident()
            plan.select(3, 0)
            check(plan, (N, C_, H, K, R, s, "tile"))
        plan.close()
    assert len(seen) == len(names), seen


def inverted_residual_blocks_run_as_one_where_that_is_faster():
    """The built-in rule against blocks that were measured both ways (as one launch, and as the first layer and what is faster behind it):
    it takes the one launch where that is clearly ahead."""
    import numpy as np
    from nart_amd import hipq
    for n, ci, ch, co, h, w, one, apart in ((22, 64, 192, 16, 31, 28, 9.6, 13.0), (9, 80, 480, 16, 21, 22, 7.6, 12.8), (15, 40, 240, 24, 25, 22, 7.3, 12.5),
                                            (92, 80, 480, 16, 5, 6, 7.5, 12.3), (17, 160, 480, 160, 5, 5, 7.2, 11.2), (5, 80, 480, 24, 29, 39, 7.8, 10.0),
                                            (64, 24, 144, 24, 56, 56, 26.8, 39.5)):
        plans = []
        for C_, K, R, g in ((ci, ch, 1, 1), (ch, ch, 3, ch), (ch, co, 1, 1)):
            plans.append(hipq.Conv2d((n, C_, h, w), np.full((K, C_ // g, R, R), 129, np.uint8), None, R // 2, 1, g, 0.05, 9, 0.002, 128, 0.05, 9))
        assert hipq.inverted_residual_fusable(*plans), (n, ci, ch, co, h, w, one, apart)
        for p in plans:
            p.close()


def depthwise_pairs_run_as_one_where_that_is_faster():
    """The built-in rule against pairs of layers that were measured both ways, a tenth apart and more (a tie: 960 -> 320 channels at 7x7,
    64 images, 9.6 us and 10.2, where the network around it gains 4)."""
    import numpy as np
    from nart_amd import hipq
    for n, h, w, c, k, stride, one, apart in ((64, 7, 7, 960, 320, 1, 9.6, 10.2), (64, 7, 7, 768, 320, 1, 8.0, 9.1), (64, 7, 7, 960, 160, 1, 8.3, 10.1), (5, 5, 4, 878, 14, 1, 6.1, 8.4),
                                              (13, 17, 18, 708, 38, 2, 6.5, 8.9), (10, 47, 38, 454, 56, 1, 10.1, 13.6), (128, 7, 7, 960, 320, 1, 16.6, 14.2), (64, 10, 10, 960, 320, 1, 23.6, 14.0),
                                              (64, 7, 7, 512, 512, 1, 12.0, 8.6)):
        oh, ow = (h - 1) // stride + 1, (w - 1) // stride + 1
        depthwise = hipq.Conv2d((n, c, h, w), np.full((c, 1, 3, 3), 129, np.uint8), None, 1, stride, c, 0.05, 9, 0.002, 128, 0.05, 9)
        point = hipq.Conv2d((n, c, oh, ow), np.full((k, c, 1, 1), 129, np.uint8), None, 0, 1, 1, 0.05, 9, 0.002, 128, 0.05, 9)
        assert hipq.depthwise_point_fusable(depthwise, point) is (one < apart), (n, h, w, c, k, stride, one, apart)
        depthwise.close(), point.close()


def layers_with_channel_scales_take_the_faster_shape():
    """The built-in rule against layers with a scale per channel or a signed range that were measured in two kernels or shapes, a fifth
    apart and more: not the slower one, whatever the neighbouring sizes take."""
    import numpy as np
    from nart_amd import hipq
    for n, c, h, w, k, r, i8, pc, fast, slow in ((5, 96, 75, 67, 192, 3, True, True, 11.1, ("resident_64x192", 13.8)), (5, 96, 75, 67, 160, 3, True, True, 10.8, ("resident_64x160", 12.9)),
                                                 (13, 41, 65, 53, 32, 3, True, True, 5.2, ("resident_128x32", 8.4)), (22, 18, 41, 43, 18, 3, False, True, 5.5, ("resident_128x32", 7.8)),
                                                 (9, 23, 70, 58, 21, 3, False, True, 5.4, ("resident_128x32", 7.7)), (3, 124, 16, 17, 156, 1, False, True, 3.3, ("64x64", 4.7)),
                                                 (1, 29, 11, 9, 967, 1, True, True, 3.1, ("64x64", 4.4)), (5, 96, 75, 67, 200, 3, True, True, 12.1, ("resident_64x256", 14.2))):
        wt = np.full((k, c, r, r), 1 if i8 else 129, np.int8 if i8 else np.uint8)
        p = hipq.Conv2d((n, c, h, w), wt, None, r // 2, 1, 1, 0.02, 0 if i8 else 128, np.linspace(0.003, 0.007, k).astype(np.float32) if pc else 0.005, 0 if i8 else 128,
                        0.02, 0 if i8 else 120, obits=7 if i8 else 8, dtype=hipq.DTYPE_I8 if i8 else hipq.DTYPE_U8)
        assert p.kernel.split("_i8_")[1].replace("_signed", "").replace("_perchannel", "") != slow[0], (p.kernel, n, c, h, w, k, fast, slow)
        p.close()


def a_patch_shape_out_of_range_names_the_range():
    import numpy as np
    from nart_amd import hipq
    p = hipq.Conv2d((1, 32, 8, 8), np.full((16, 32, 1, 1), 129, np.uint8), None, 0, 1, 1, 0.05, 9, 0.002, 128, 0.05, 9)
    for shape in range(-1, 6):
        hipq.inverted_residual_select(p, shape)
    for shape in (-2, 6):
        with pytest.raises(hipq.HipqError, match="shape %d outside -1..5" % shape):
            hipq.inverted_residual_select(p, shape)


def block_tails_keep_to_patches_that_divide_an_image():
    """hipq_bottleneck_tail_run may write the sum over the residual wherever some patch shape divides the image, also where another would
    need as many overlapping patches or fewer, and takes 128 channels by rule on such images however few their pixels; where none
    divides it, patches overlap: another tensor, and 600 pixels."""
    import numpy as np
    from nart_amd import hipq
    x, y, z = 4096, 8192, 12288  # never touched
    grids = {"conv_bottleneck_tail_kernelILi2ELi%dELi%dE" % (h, w): (h, w) for h, w in ((8, 8), (4, 14), (7, 7))}
    last = C.c_char_p.in_dll(STUB, "stub_last_kernel")
    for H, W, patch, divides in ((14, 14, (7, 7), True), (21, 21, (7, 7), True), (35, 35, (7, 7), True), (49, 49, (7, 7), True), (14, 21, (7, 7), True),
                                 (14, 28, (7, 7), True), (7, 14, (7, 7), True), (42, 42, (7, 7), True), (63, 63, (7, 7), True), (28, 28, (4, 14), True),
                                 (56, 56, (8, 8), True), (8, 14, (4, 14), True), (16, 17, (8, 8), False), (13, 13, (8, 8), False), (9, 29, (8, 8), False),
                                 (25, 25, (4, 14), False), (7, 9, (7, 7), False)):
        mid = hipq.Conv2d((1, 128, H, W), np.full((128, 128, 3, 3), 129, np.uint8), None, 1, 1, 1, 0.05, 9, 0.002, 128, 0.05, 9)
        widen = hipq.Conv2d((1, 128, H, W), np.full((512, 128, 1, 1), 129, np.uint8), None, 0, 1, 1, 0.05, 9, 0.002, 128, 0.05, 9)
        rule = hipq.bottleneck_tail_fusable(mid, widen, False, 0.04, 3, 0.09, 10)
        assert rule == (divides or H * W >= 600), (H, W, rule)
        mid.special(2)

        def run(to):
            return hipq.lib().hipq_bottleneck_tail_run(mid.handle, widen.handle, x, y, 0, 0.04, 3, 0.09, 10, 8, to, None, 0, None, None)
        hipq.check(run(z))
        assert [p for k, p in grids.items() if k in last.value.decode()] == [patch], (H, W, last.value)
        assert (run(y) == 0) == divides, (H, W)


def a_pair_of_layers_is_launched_as_quickly_as_two():
    """hipq_conv2d_run_pair and its predicate choose among what the plans keep: the call takes the host little more than two launches."""
    import time
    import numpy as np
    from nart_amd import hipq
    lib = hipq.lib()
    a, b = (hipq.Conv2d((1, 128, 28, 28), np.full((256, 128, r, r), 129, np.uint8), None, r // 2, 2, 1, 0.05, 9, 0.002, 128, 0.05, 9) for r in (3, 1))

    def best(f):
        times = []
        for _ in range(40):
            t = time.perf_counter()
            for _ in range(50):
                f()
            times.append(time.perf_counter() - t)
        return min(times)
    two = best(lambda: (lib.hipq_conv2d_run(a.handle, 4096, 8192, None, None), lib.hipq_conv2d_run(b.handle, 4096, 12288, None, None)))
    pair = best(lambda: lib.hipq_conv2d_run_pair(a.handle, 4096, 0, 8192, b.handle, 4096, 0, 12288, None))
    assert lib.hipq_conv2d_pair_fusable(a.handle, b.handle) and pair < 2.2 * two, (pair, two)


def add_forms(pairs, took=None):
    """make_add_params and make_add_exact (csrc/hipq/common.h) for (alpha 0, zero point 0, alpha 1, zero point 1, alpha, zero point) of an
    add: its constants, and those of its exact form or None; took: called with the seconds that the latter took."""
    import time
    from nart_amd import hipq

    class Params(C.Structure):
        _fields_ = [(n, C.c_uint32) for n in ("m0", "m1")] + [(n, C.c_int32) for n in "s0 s1 sh z0 z1 oz hi c0 c1 cadd fast".split()]
    params, exact = hipq.lib()._ZN4hipq15make_add_paramsEfififiiPNS_9AddParamsE, hipq.lib()._ZN4hipq14make_add_exactEPNS_9AddParamsE
    params.restype = exact.restype = C.c_bool
    params.argtypes = [C.c_float, C.c_int, C.c_float, C.c_int, C.c_float, C.c_int, C.c_int, C.POINTER(Params)]
    exact.argtypes = [C.POINTER(Params)]
    out = []
    for q in pairs:
        plain = Params()
        assert params(*q, 8, C.byref(plain))
        form = Params.from_buffer_copy(plain)
        t = time.perf_counter()
        found = exact(C.byref(form))
        if took:
            took(time.perf_counter() - t)
        out.append((plain, form if found else None))
    return out


def exact_adds_are_the_operator():
    """The exact form of an add, wherever there is one, against the oracle's add over all 65 536 pairs of bytes: scales from an eighth of the
    sum's to eight times it, any zero points.  Of the adds with a 32-bit form nearly all have one where both operands' scales are below
    the sum's, otherwise none."""
    import random
    import numpy as np
    from oracle import orc
    rng = random.Random(11)
    x0, x1 = (v.astype(np.uint8).reshape(1, 1, 256, 256) for v in np.indices((256, 256)))
    a, b = x0.astype(np.uint64), x1.astype(np.uint64)
    count = {True: [0, 0], False: [0, 0]}
    for k in range(400):
        r0, r1 = (2.0 ** rng.uniform(-3, 0 if k % 4 else 3) for _ in range(2))
        if k % 8 == 1:
            r1 = r0
        alpha = float(np.float32(rng.uniform(0.01, 0.2)))
        q = (float(np.float32(alpha * r0)), rng.choice((0, 255, rng.randrange(256))), float(np.float32(alpha * r1)), rng.choice((0, 255, rng.randrange(256))),
             alpha, rng.choice((0, 255, rng.randrange(256))))
        (plain, form), = add_forms([q])
        kind = count[bool(np.float32(q[0]) / np.float32(alpha) < 1 and np.float32(q[2]) / np.float32(alpha) < 1)]
        kind[0] += plain.fast
        if form is None:
            continue
        kind[1] += 1
        assert form.sh == 0
        t = a * np.uint64(form.m0) + b * np.uint64(form.m1) + np.uint64((form.c1 & 0xffffffff) << 32 | (form.c0 & 0xffffffff))
        got = np.clip((t >> np.uint64(32)).astype(np.uint32).view(np.int32), 0, 255)
        assert np.array_equal(got, orc.add_u8(x0, x1, *q)), (q, int((got != orc.add_u8(x0, x1, *q)).sum()))
    assert count[True][1] > 0.95 * count[True][0] and count[True][0] > 250 and count[False][0] > 50 and count[False][1] == 0, count


def exact_adds_are_searched_for_once():
    """A launch asks for the exact form of its add each time: the forms of a network's adds are all remembered."""
    import random
    rng = random.Random(3)
    pairs = [(rng.uniform(0.03, 0.09), rng.randrange(256), rng.uniform(0.03, 0.09), rng.randrange(256), rng.uniform(0.09, 0.12), rng.randrange(40))
             for _ in range(48)]

    passes = []
    for _ in range(40):
        times, forms = [], []
        for q in pairs:
            (plain, form), = add_forms([q], lambda t: times.append(t))
            forms.append((plain.m0, form and (form.m0, form.m1, form.sh, form.c0, form.c1)))
        passes.append((times, forms))
    first = passes[0]
    assert all(f == first[1] for _, f in passes) and sum(f is not None for _, f in first[1]) > 40
    later = [min(t[i] for t, _ in passes[1:]) for i in range(len(pairs))]
    assert max(later) < 0.5 * sorted(first[0])[len(pairs) // 2], (max(later), sorted(first[0])[len(pairs) // 2])


def runtime():
    from nart_amd import art
    lib = os.path.join(ROOT, "nart_amd", "lib")
    return art.Runtime(os.path.join(lib, "libart.so"), [os.path.join(lib, "libart_module_hip.so")])


def fused_block_follows_the_scales_of_its_operators():
    """An inverted residual block that ran as one launch, then one operator alone gets another input scale and is prepared again -
    the add for its residual, or the first convolution: the two no longer read the block's input alike, so the block runs
    operator by operator until they do again."""
    import numpy as np
    rt = runtime()
    ws = rt.workspace("hip")
    fused = rt.libs[1].hip_module_fused_inverted
    fused.restype = C.c_long
    x = ws.tensor(np.zeros((2, 24, 15, 17), np.uint8))
    ops, cur = [], x
    for K, c, k, g, q in ((144, 24, 1, 1, dict(ialpha=0.05, izp=9, walpha=0.0018, wzp=128, oalpha=0.06, ozp=30)),
                          (144, 1, 3, 144, dict(ialpha=0.06, izp=30, walpha=0.0026, wzp=128, oalpha=0.055, ozp=40)),
                          (24, 144, 1, 1, dict(ialpha=0.055, izp=40, walpha=0.0012, wzp=128, oalpha=0.07, ozp=121))):
        ops.append(ws.conv2d(cur, ws.tensor(np.full((K, c, k, k), 130, np.uint8)), None, k // 2, 1, g, q).prepare())
        cur = ops[-1].output(0)
    ops.append(ws.add(x, cur, dict(ialpha=[0.05, 0.07], izp=[9, 121], oalpha=0.09, ozp=10)).prepare())

    def taken():
        before = fused()
        for o in ops:
            o.run()
        return fused() - before
    assert taken() == 1 and taken() == 1
    for ialpha, izp, want in ((0.04, 9, 0), (0.05, 9, 1), (0.05, 11, 0), (0.05, 9, 1)):
        ops[3].set_quant(ialpha=[ialpha, 0.07], izp=[izp, 121]).config().prepare()
        assert taken() == want, ("add", ialpha, izp)
    for ialpha, izp, want in ((0.04, 9, 0), (0.05, 9, 1), (0.05, 11, 0), (0.05, 9, 1)):
        ops[0].set_quant(ialpha=ialpha, izp=izp).config().prepare()
        assert taken() == want, ("expanding convolution", ialpha, izp)


def small_parade(rt, ws, hw=64):
    """An engine file whose pass is long enough to be recorded, and one pass over it: one() returns what that pass did."""
    import numpy as np
    from nart_amd import cases, engine
    case = cases.resnet18(N=1, hw=hw)
    p = engine.Parade(rt, engine.write_engine(case), [ws])
    x = np.zeros(case.input.shape, np.float32)
    count = {n: C.c_long.in_dll(STUB, "stub_" + n) for n in ("kernels", "captures", "graph_launches")}

    def one(read=True):
        before = {n: c.value for n, c in count.items()}
        p.inputs()[0].write(x)
        p.run()
        if read:
            p.outputs()[0].numpy()
        did = {n: c.value - before[n] for n, c in count.items()}
        return "recorded" if did["captures"] else "replayed" if did["graph_launches"] else "eager" if did["kernels"] else "nothing"
    return p, one


def a_chain_of_separable_layers_is_divided_blocks_first():
    """Depthwise and 1x1 layers in turn: a 1x1 layer that begins a whole inverted residual block belongs to that block, not to the
    depthwise layer in front of it - the division that the executor makes as well."""
    import numpy as np
    from nart_amd import hipq
    rt = runtime()
    ws = rt.workspace("hip")
    count = {n: getattr(rt.libs[1], "hip_module_fused_" + n) for n in ("inverted", "pairs")}
    for f in count.values():
        f.restype = C.c_long
    kernels = C.c_long.in_dll(STUB, "stub_kernels")
    for N, HW, widths in ((1, 14, (32, 96, 32)), (1, 14, (32, 96, 32, 64)), (1, 28, (16, 64, 24))):
        # depthwise, 1x1 to widths[1], depthwise, 1x1 to widths[2], ...
        ops, cur = [], ws.tensor(np.zeros((N, widths[0], HW, HW), np.uint8))
        plans, c = [], widths[0]
        for K in widths[1:]:
            for k, cols, g, out in ((3, 1, c, c), (1, c, 1, K)):
                w = np.full((out, cols, k, k), 130, np.uint8)
                ops.append(ws.conv2d(cur, ws.tensor(w), None, k // 2, 1, g, dict(ialpha=0.05, izp=9, walpha=0.002, wzp=128, oalpha=0.05, ozp=9)).prepare())
                plans.append(hipq.Conv2d((N, c, HW, HW), w, None, k // 2, 1, g, 0.05, 9, 0.002, 128, 0.05, 9))
                cur = ops[-1].output(0)
            c = K
        assert hipq.depthwise_point_fusable(*plans[:2]) and hipq.inverted_residual_fusable(*plans[1:4]), widths
        last_pair = len(widths) > 3 and hipq.depthwise_point_fusable(*plans[4:6])
        for again in range(2):  # the first run brings the input into the device's layout as well
            before, launches = {n: f() for n, f in count.items()}, kernels.value
            for o in ops:
                o.run()
            assert {n: f() - before[n] for n, f in count.items()} == {"inverted": 1, "pairs": int(last_pair)}, widths
            assert not again or kernels.value - launches == 2 + (0 if len(widths) == 3 else 1 if last_pair else 2), widths
        for o in ops:
            o.delete()


def blocks_are_decided_again_for_recorded_passes():
    """A bottleneck block of few pixels is one launch where its operators run one by one, three where a pass is recorded: also when the
    operators have run before the workspace's first pass, and again when they are prepared anew."""
    import numpy as np
    from nart_amd import hipq
    rt = runtime()
    ws = rt.workspace("hip")
    blocks = rt.libs[1].hip_module_fused_blocks
    blocks.restype = C.c_long
    kernels = C.c_long.in_dll(STUB, "stub_kernels")
    x = ws.tensor(np.zeros((2, 1024, 14, 14), np.uint8))
    ops, cur = [], x
    for K, c, k, q in ((256, 1024, 1, dict(ialpha=0.05, izp=9, walpha=0.0011, wzp=128, oalpha=0.06, ozp=0)),
                       (256, 256, 3, dict(ialpha=0.06, izp=0, walpha=0.0016, wzp=128, oalpha=0.055, ozp=0)),
                       (1024, 256, 1, dict(ialpha=0.055, izp=0, walpha=0.0035, wzp=128, oalpha=0.07, ozp=121))):
        ops.append(ws.conv2d(cur, ws.tensor(np.full((K, c, k, k), 130, np.uint8)), None, k // 2, 1, 1, q).prepare())
        cur = ops[-1].output(0)
    ops.append(ws.add(cur, x, dict(ialpha=[0.07, 0.05], izp=[121, 9], oalpha=0.09, ozp=0)).prepare())

    def one():
        before, launches = blocks(), kernels.value
        for o in ops:
            o.run()
        return blocks() - before, kernels.value - launches
    assert one()[0] == 1  # the first run brings the input into the device's layout as well
    assert [one() for _ in range(3)] == [(1, 1)] * 3
    p, pass_of = small_parade(rt, ws)
    assert pass_of() == "eager"
    assert [one() for _ in range(3)] == [(0, 3)] * 3, "decided before the workspace ran passes"
    for o in ops:
        o.prepare()
    assert [one() for _ in range(2)] == [(0, 3)] * 2
    p.delete()
    # the passes themselves: operator by operator, recorded and replayed, below and above the pixels from which one launch pays
    from nart_amd import cases, engine
    did = {n: C.c_long.in_dll(STUB, "stub_" + n) for n in ("captures", "graph_launches")}
    for N, want in ((2, 0), (20, 3)):
        c = cases.Case("chain", 12)
        t = c.input_u8((N, 1024, 14, 14), 0.0186, 114)
        for _ in range(3):
            b = c.conv(c.conv(t, 256, 1, ozp=0), 256, 3, ozp=0)
            t = c.add(c.conv(b, 1024, 1), t)
        for _ in range(6):  # long enough to be recorded where the blocks are one launch each
            t = c.conv(t, 64, 1)
        c.output = t
        p = engine.Parade(rt, engine.write_engine(c), [ws])
        before = {n: v.value for n, v in did.items()}
        for k in range(4):
            p.inputs()[0].write(np.zeros((N, 1024, 14, 14), np.uint8))
            n = blocks()
            p.run()
            assert blocks() - n == want, (N, k)
        assert [v.value - before[n] for n, v in did.items()] == [1, 3], N
        p.delete()


def launched(o):
    """How many kernels an operator's run() launches."""
    kernels = C.c_long.in_dll(STUB, "stub_kernels")
    before = kernels.value
    o.run()
    return kernels.value - before


def operators_run_one_by_one_launch_themselves():
    """Two convolutions of one tensor run as one launch inside a pass only: on a workspace that has run passes, whatever is run between
    them and however often each has run, each run() launches its own kernel and reads what the tensor holds then."""
    import numpy as np
    rt = runtime()
    ws = rt.workspace("hip")
    p, pass_of = small_parade(rt, ws)
    assert pass_of() == "eager"
    x = ws.tensor(np.zeros((1, 64, 14, 14), np.uint8))
    q = dict(ialpha=0.05, izp=9, walpha=0.002, wzp=128, oalpha=0.05, ozp=9)
    a, b = (ws.conv2d(x, ws.tensor(np.full((128, 64, r, r), 130, np.uint8)), None, r // 2, 2, 1, q).prepare() for r in (3, 1))
    for o in (a, b, a, b, a, a, b, b, a, b, a, b):
        x.write(np.ones((1, 64, 14, 14), np.uint8))  # one kernel brings it in
        assert launched(o) == 2 and launched(o) == 1
        if o is b:
            pass_of()


def shared(data, pairs):
    """The engine file `data` with tensors that share one memory, (from, to) by their indices."""
    import struct
    return data[:-4] + struct.pack("<i", len(pairs)) + b"".join(struct.pack("<ii", *p) for p in pairs)


def two_parades_of_one_input_launch_their_own_layers():
    """Two parades of a workspace whose input is one memory, each with a convolution of it that could run with the other's: a pass computes
    the layers of its own parade, recorded or not, in whatever order the passes come."""
    import numpy as np
    from nart_amd import cases, engine
    rt = runtime()
    ws = rt.workspace("hip")
    parades = []
    for r in (3, 1):
        c = cases.Case("chain", 3)
        t = c.conv(c.input_u8((1, 64, 14, 14), 0.05, 9), 128, r, stride=2)
        for _ in range(9):
            t = c.conv(t, 64, 1)
        c.output = t
        parades.append(engine.Parade(rt, engine.write_engine(c), [ws], prepare=False))
    inputs = [p.inputs()[0] for p in parades]
    rt.core.tensor_share.argtypes = [C.c_void_p, C.c_void_p]
    rt.core.tensor_share(inputs[0].ptr, inputs[1].ptr)
    for p in parades:
        rt.core.parade_prepare(p.ptr)
    kernels, replays = (C.c_long.in_dll(STUB, "stub_" + n) for n in ("kernels", "graph_launches"))
    x = np.zeros((1, 64, 14, 14), np.uint8)
    eager = []
    for p in parades:
        before = kernels.value
        p.run()
        eager.append(kernels.value - before)
    assert eager == [11, 10]  # the first one's pass brings the input in
    for k, order in enumerate(((0, 0, 1), (1, 0, 1), (0, 1, 0))):
        for i in order:
            inputs[0].write(x)
            before, n = kernels.value, replays.value
            parades[i].run()
            assert replays.value == n + 1
            launches = kernels.value - before
            assert launches in (0, 1, 10, 11), (k, i, launches)  # replayed, replayed behind an upload, recorded
    assert rt.libs[1].hip_module_chained_convs() == 0


def layers_run_together_only_where_their_memories_allow():
    """A convolution runs with a later one of the same tensor - unless an operator between the two writes that tensor's memory, or one
    ahead of the second has to do with the memory that it writes (tensors of an engine file may share memories)."""
    import numpy as np
    from nart_amd import cases, engine
    rt = runtime()
    ws = rt.workspace("hip")
    for share, pairs in ((None, 1), ("written between", 0), ("read between", 0), ("read before", 0)):
        c = cases.Case("chain", 3)
        x0 = c.input_u8((1, 16, 14, 14), 0.05, 9)
        x, v, t = c.conv(x0, 64, 3), c.conv(x0, 64, 1), c.conv(x0, 128, 3, stride=2)
        if share == "read before":
            z = c.conv(t, 128, 1)
        a = c.conv(x, 128, 3, stride=2)
        u = c.add(x, v) if share == "written between" else x
        if share == "read between":
            z = c.conv(t, 128, 1)
        b = c.conv(u, 128, 1, stride=2)
        if share in (None, "written between"):
            z = c.conv(t, 128, 1)
        y = c.add(c.add(c.conv(a, 128, 1), b), z)
        for _ in range(6):
            y = c.conv(y, 64, 1)
        c.output = y
        names = [c.input.name] + [n.attrs[k] for n in c.nodes if n.kind == "conv" for k in ("w", "b")]
        index = {}
        for n in c.nodes:
            index[n.output] = len(names)
            names.append(n.output)
        data = engine.write_engine(c)
        if share == "written between":
            data = shared(data, [(index[x.name], index[u.name])])
        elif share:
            data = shared(data, [(index[t.name], index[b.name])])
        p = engine.Parade(rt, data, [ws])
        for k in range(4):
            p.inputs()[0].write(np.zeros(x0.shape, np.uint8))
            before = rt.libs[1].hip_module_chained_convs()
            p.run()
            assert rt.libs[1].hip_module_chained_convs() - before == (pairs if k else 0), (share, k)
        p.delete()


def layers_computed_ahead_follow_their_tensors():
    """The kernel of a stem and its pooling computes the convolution that reads the pooled tensor as well, whose run() then has nothing to
    do - unless the pooled tensor, its own output or its scales have changed since."""
    import numpy as np
    rt = runtime()
    ws = rt.workspace("hip")
    x = ws.tensor(np.zeros((2, 3, 64, 96), np.uint8))
    conv = ws.conv2d(x, ws.tensor(np.full((64, 3, 7, 7), 130, np.uint8)), None, 3, 2, 1,
                     dict(ialpha=0.031, izp=77, walpha=0.0042, wzp=128, oalpha=0.09, ozp=0)).prepare()
    pool = ws.pool(conv.output(0), 3, 1, 2, 0, False, dict(ialpha=0.09, izp=0, oalpha=0.09, ozp=0)).prepare()
    q = dict(ialpha=0.09, izp=0, walpha=0.004, wzp=128, oalpha=0.07, ozp=0)
    layer = ws.conv2d(pool.output(0), ws.tensor(np.full((64, 64, 1, 1), 130, np.uint8)), None, 0, 1, 1, q).prepare()

    def ahead():
        before = rt.libs[1].hip_module_chained_convs()
        conv.run()
        pool.run()
        return rt.libs[1].hip_module_chained_convs() - before
    for change, kernels in ((None, 0), ("input", 2), ("output", 1), ("scales", 1), (None, 0)):
        assert ahead() == 1
        if change == "input":
            pool.output(0).write(np.ones((2, 64, 16, 24), np.uint8))  # one kernel brings it in
        elif change == "output":
            layer.output(0).write(np.ones((2, 64, 16, 24), np.uint8))
        elif change == "scales":
            layer.set_quant(**dict(q, oalpha=0.08)).config().prepare()
        assert launched(layer) == kernels, change
        assert launched(layer) == 1, change


def a_pass_that_cannot_be_recorded_runs_its_operators():
    """On the null stream, which cannot be captured, and where the runtime refuses the graph: every pass runs operator by
    operator, and no error stays behind for the next launch to find."""
    rt = runtime()
    ws = rt.workspace("hip")
    rt.libs[1].hip_workspace_set_stream.argtypes = [C.c_void_p, C.c_void_p]
    rt.libs[1].hip_workspace_set_stream(ws.ptr, None)
    p, one = small_parade(rt, ws)
    assert [one() for _ in range(5)] == ["eager"] * 5 and STUB.stub_error() == 0
    p.delete()
    ws.delete()
    fail = C.c_long.in_dll(STUB, "stub_fail_instantiate")
    fail.value = 1
    ws = rt.workspace("hip")
    p, one = small_parade(rt, ws)
    for i in range(4):
        assert one() == ("recorded" if i == 1 else "eager") and STUB.stub_error() == 0, i  # pass 1: tried, refused, then run
    p.delete()


def records_are_taken_again_after_many_changes():
    """A program that prepares its parade again before every third pass, or creates parades beside it, gets fewer and fewer
    attempts to record; once it leaves the parade alone its passes are recorded and replayed again."""
    rt = runtime()
    ws = rt.workspace("hip")
    p, one = small_parade(rt, ws)
    did = []
    for _ in range(40):
        rt.core.parade_prepare(p.ptr)
        did += [one(), one(), one()]
    assert did[:3] == ["eager", "recorded", "replayed"] and did.count("recorded") <= 3
    settled = [one() for _ in range(600)]
    assert settled.count("recorded") == 1 and settled[-300:] == ["replayed"] * 300
    rt.core.parade_prepare(p.ptr)  # a record that has served long: the next is taken at once
    assert [one() for _ in range(3)] == ["eager", "recorded", "replayed"]
    for _ in range(20):
        small_parade(rt, ws)[0].delete()
        one()
    assert [one() for _ in range(600)][-300:] == ["replayed"] * 300
    p.delete()
    ws.delete()


def an_output_that_nobody_reads_is_not_copied_back():
    """A recorded pass ends with the copy of an output that the host has read.  Once the host stops reading it, the record is taken
    again without the copy; when the host reads on, the output still comes, and a later record has the copy again."""
    rt = runtime()
    ws = rt.workspace("hip")
    stream_of = rt.libs[1].hip_workspace_stream
    stream_of.argtypes, stream_of.restype = [C.c_void_p], C.c_void_p
    STUB.stub_pending.argtypes, STUB.stub_pending.restype = [C.c_void_p], C.c_long
    p, one = small_parade(rt, ws)

    def nodes(read):  # operations that one pass queues
        rt.libs[1].hip_workspace_synchronize(C.c_void_p(C.addressof(ws.ptr.contents)))
        one(read=False)
        n = STUB.stub_pending(stream_of(ws.ptr))
        if read:
            p.outputs()[0].numpy()
        return n
    for _ in range(3):
        with_copy = nodes(read=True)
    assert one() == "replayed"
    without = [nodes(read=False) for _ in range(40)][-10:]
    assert without == [with_copy - 1] * 10 and one(read=False) == "replayed"
    for _ in range(10):
        nodes(read=True)
    rt.core.parade_prepare(p.ptr)
    assert [nodes(read=True) for _ in range(10)][-1] == with_copy
    # an output that was read once in an earlier life of the parade is not copied by the records of the next
    for _ in range(2):
        rt.core.parade_prepare(p.ptr)
        counts = [nodes(read=False) for _ in range(40)]
    assert counts[-1] == with_copy - 1 and with_copy not in counts[2:]
    p.delete()
    ws.delete()


def a_write_waits_for_the_copy_back_that_fills_the_same_mirror():
    """A replayed pass has queued the copy of its output into the host mirror; the program then writes an array of its own into that
    tensor (hip_mem_write) and reads it: it gets its array, not what the copy brings later."""
    import numpy as np
    from nart_amd import cases, engine
    rt = runtime()
    ws = rt.workspace("hip")
    # ten convolutions, then floats: their copy into the mirror is one of the runtime's own copies
    c = cases.Case("chain", 3)
    t = c.input_u8((1, 16, 8, 8), 0.05, 9)
    for _ in range(10):
        t = c.conv(t, 16, 3)
    c.output = c.dequantize(t)
    p = engine.Parade(rt, engine.write_engine(c), [ws])
    out = p.outputs()[0]
    write = rt.libs[1].hip_mem_write
    write.argtypes, write.restype = [C.c_void_p, C.c_void_p, C.c_size_t], C.c_bool
    replays = C.c_long.in_dll(STUB, "stub_graph_launches")
    for i in range(4):
        p.inputs()[0].write(np.zeros((1, 16, 8, 8), np.uint8))
        p.run()
        if i < 3:
            out.numpy()
    assert replays.value >= 2
    mine = np.arange(out.numpy().size, dtype=np.float32).reshape(out.shape)
    p.run()
    assert write(out.ptr.contents.mem, mine.ctypes.data, mine.nbytes)
    rt.libs[1].hip_workspace_synchronize(C.c_void_p(C.addressof(ws.ptr.contents)))
    assert np.array_equal(out.numpy(), mine)
    p.delete()
    ws.delete()


def a_write_waits_for_every_stream_that_reads_the_array():
    """One float input, quantize operators on two workspaces: the one prepared last reads the quantized bytes in pinned memory, the
    other the values.  The next array is written only when both streams have read the one before - also when one of the
    workspaces replays a recorded pass."""
    import numpy as np
    rt = runtime()
    write = rt.libs[1].hip_mem_write
    write.argtypes, write.restype = [C.c_void_p, C.c_void_p, C.c_size_t], C.c_bool
    stream_of = rt.libs[1].hip_workspace_stream
    stream_of.argtypes, stream_of.restype = [C.c_void_p], C.c_void_p
    STUB.stub_pending.argtypes, STUB.stub_pending.restype = [C.c_void_p], C.c_long
    for n in (8, 2048):  # read by the kernels directly; above 4 MB of bytes (16 MB of values) brought to the device first
        a = np.ones((1, 3, n, 1024 if n > 8 else n), np.float32)
        two = [rt.workspace("hip"), rt.workspace("hip")]
        streams = [stream_of(w.ptr) for w in two]
        for order in ((0, 1), (1, 0)):
            x = two[0].tensor(a)
            ops = [w.quantize(x, 0.1, 3).prepare() for w in two]
            for _ in range(3):
                assert write(x.ptr.contents.mem, a.ctypes.data, a.nbytes)
                for k in order:
                    ops[k].run()
                assert max(STUB.stub_pending(s) for s in streams) > 0
                assert write(x.ptr.contents.mem, a.ctypes.data, a.nbytes)
                pending = [STUB.stub_pending(s) for s in streams]  # above the line: the new array's own copies, on one stream
                assert pending == [0, 0] if n == 8 else 0 in pending, (n, order, pending)
                for o in ops:
                    o.run()
            for o in ops:
                o.delete()
    # a recorded pass on the first workspace, the values read by an operator on the second
    from nart_amd import cases, engine
    c = cases.Case("chain", 3)
    t = c.quantize(c.input_f32((1, 16, 8, 8)), 0.05, 9)
    for _ in range(10):
        t = c.conv(t, 16, 3)
    c.output = t
    a = np.ones((1, 16, 8, 8), np.float32)
    p = engine.Parade(rt, engine.write_engine(c), [two[0]])
    x = p.inputs()[0]
    replays, captures = (C.c_long.in_dll(STUB, "stub_" + k) for k in ("graph_launches", "captures"))
    quantize = two[1].quantize(x, 0.07, 5).prepare()
    for i in range(6):
        assert write(x.ptr.contents.mem, a.ctypes.data, a.nbytes)
        quantize.run()
        p.run()
        assert write(x.ptr.contents.mem, a.ctypes.data, a.nbytes)
        assert [STUB.stub_pending(s) for s in streams] == [0, 0], i
        p.run()
    assert captures.value >= 1 and replays.value >= 3


def operators_of_two_workspaces_wait_for_each_other():
    """One workspace's operator reads what another's writes: it is queued when that has finished, and the writer runs again when the
    reader has finished - operator by operator, and as recorded passes whose input or output the other workspace uses."""
    import numpy as np
    from nart_amd import cases, engine
    rt = runtime()
    stream_of = rt.libs[1].hip_workspace_stream
    stream_of.argtypes, stream_of.restype = [C.c_void_p], C.c_void_p
    STUB.stub_pending.argtypes, STUB.stub_pending.restype = [C.c_void_p], C.c_long
    two = [rt.workspace("hip"), rt.workspace("hip")]
    first, second = [stream_of(w.ptr) for w in two]
    q = dict(ialpha=0.1, izp=3, oalpha=0.2, ozp=4)
    writer = two[0].relu(two[0].tensor(np.ones((1, 16, 8, 8), np.uint8)), q).prepare()
    reader = two[1].relu(writer.output(0), q).prepare()
    for _ in range(3):
        writer.run()
        assert STUB.stub_pending(second) == 0 and STUB.stub_pending(first) > 0
        reader.run()
        assert STUB.stub_pending(first) == 0 and STUB.stub_pending(second) > 0
    c = cases.Case("chain", 3)
    t = c.input_u8((1, 16, 8, 8), 0.05, 9)
    for _ in range(10):
        t = c.conv(t, 16, 3)
    c.output = t
    p = engine.Parade(rt, engine.write_engine(c), [two[0]])
    reader = two[1].relu(p.outputs()[0], q).prepare()
    replays = C.c_long.in_dll(STUB, "stub_graph_launches")
    x = p.inputs()[0]
    beside = two[1].relu(x, q).prepare()
    x.write(np.ones((1, 16, 8, 8), np.uint8))
    rt.libs[1].hip_workspace_synchronize(C.c_void_p(C.addressof(two[1].ptr.contents)))
    for i in range(6):
        p.run()
        assert STUB.stub_pending(second) == 0 and STUB.stub_pending(first) > 0, i
        (reader if i % 2 else beside).run()
        assert STUB.stub_pending(first) == 0 and STUB.stub_pending(second) > 0, i
    x.write(np.ones((1, 16, 8, 8), np.uint8))  # waits for whoever reads the pinned side; the pass brings the values in again
    beside.run()
    p.run()
    assert STUB.stub_pending(second) == 0
    assert replays.value >= 4


CASES = [depthwise_pairs_run_as_one_where_that_is_faster, inverted_residual_add_needs_equal_shapes,
         inverted_residual_blocks_run_as_one_where_that_is_faster, a_pair_of_layers_is_launched_as_quickly_as_two,
         exact_adds_are_the_operator, exact_adds_are_searched_for_once, block_tails_keep_to_patches_that_divide_an_image,
         layers_with_channel_scales_take_the_faster_shape, a_patch_shape_out_of_range_names_the_range, a_chained_add_names_its_kernels,
         a_plan_launches_the_kernel_that_it_names, fused_block_follows_the_scales_of_its_operators,
         a_chain_of_separable_layers_is_divided_blocks_first, blocks_are_decided_again_for_recorded_passes,
         operators_run_one_by_one_launch_themselves, two_parades_of_one_input_launch_their_own_layers,
         layers_run_together_only_where_their_memories_allow, layers_computed_ahead_follow_their_tensors,
         a_pass_that_cannot_be_recorded_runs_its_operators, records_are_taken_again_after_many_changes,
         an_output_that_nobody_reads_is_not_copied_back, a_write_waits_for_the_copy_back_that_fills_the_same_mirror,
         a_write_waits_for_every_stream_that_reads_the_array, operators_of_two_workspaces_wait_for_each_other]


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("hip") / "hip_stub.so")
    subprocess.check_call(["gcc", "-O1", "-std=gnu11", "-Wall", "-Werror", "-fPIC", "-shared", os.path.join(ROOT, "tests", "hip_stub.c"), "-o", so])
    return so


@pytest.mark.parametrize("case", CASES, ids=lambda c: c.__name__)
def test_host_side(case, stub):
    r = subprocess.run([sys.executable, os.path.abspath(__file__), stub, case.__name__], cwd=ROOT, stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT, text=True, timeout=120)
    assert r.returncode == 0, r.stdout[-4000:]


if __name__ == "__main__":
    sys.path.insert(0, ROOT)
    STUB = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
    globals()[sys.argv[2]]()
