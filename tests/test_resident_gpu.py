"""conv_resident_kernel (pixels in LDS, weights in registers) in every shape that is built, against the CPU oracle: accumulators, bytes,
the fused add, a ReLU and the fused dequantize are exact (integer arithmetic, single rounded float products)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import orc  # noqa: E402  (checker only)
from nart_amd import hipq  # noqa: E402

SHAPES = [(1, 1, 1, 8), (1, 1, 1, 4), (2, 1, 1, 8), (2, 1, 1, 4), (2, 2, 1, 8), (2, 2, 1, 4), (2, 2, 2, 4), (2, 2, 2, 2), (4, 1, 1, 8), (4, 2, 1, 8),
          (4, 2, 1, 4), (4, 4, 1, 4), (4, 4, 2, 4), (4, 4, 2, 2), (8, 2, 1, 2), (1, 1, 2, 1), (1, 1, 4, 1), (2, 1, 4, 1), (2, 2, 2, 1), (2, 2, 4, 1),
          (4, 1, 4, 1), (4, 2, 4, 1), (4, 4, 2, 1), (4, 4, 4, 1), (8, 2, 2, 1), (8, 2, 4, 1)]
CASES = [  # N, C, H, W, K, R, pad, stride, data type, scale per channel, weight zero point
    (1, 512, 7, 7, 512, 3, 1, 1, "u8", False, 128),   # one image shorter than the widest tile, more slabs than waves
    (3, 64, 9, 17, 72, 3, 1, 2, "u8", False, 128),    # tiles across rows and images, a slab is a whole tap
    (5, 128, 3, 2, 20, 3, 1, 1, "u8", False, 128),    # images smaller than the kernel, several to a tile
    (2, 256, 8, 9, 48, 1, 0, 1, "u8", False, 128),    # 1x1
    (2, 64, 9, 11, 33, 1, 0, 2, "u8", False, 128),    # 1x1 with a stride: the region has pixels that nobody reads
    (33, 1280, 1, 1, 100, 1, 0, 1, "u8", False, 128),  # fully connected
    (2, 36, 13, 11, 24, 5, 2, 1, "u8", False, 128),   # pieces of a slab in different taps, 25 taps
    (9, 16, 5, 4, 130, 3, 0, 1, "u8", False, 128),    # one piece per tap, no padding
    (2, 20, 6, 7, 17, 5, 2, 3, "u8", False, 101),     # the weight zero point's sums
    (1, 96, 14, 13, 200, 3, 1, 1, "i8", True, 0),
    (2, 112, 7, 9, 40, 3, 1, 2, "i8", False, 0),
    (2, 48, 10, 9, 70, 3, 1, 1, "u8", True, 128),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(map(str, c)))
def test_resident_kernel_matches_the_oracle_in_every_shape(case):
    N, C, H, W, K, R, pad, st, dtype, per_channel, wzp = case
    rng = np.random.default_rng(abs(hash(case[:8])) % (1 << 31))
    x = rng.integers(0, 256, (N, C, H, W), dtype=np.uint8)
    w = rng.integers(*((0, 256) if wzp in (0, 128) else (wzp - 90, wzp + 91)), (K, C, R, R), dtype=np.uint8)  # around their zero point
    b = rng.integers(-30000, 30000, K).astype(np.int32)
    ia, izp, ozp = 0.02, 77, 120
    wa = (0.004 * rng.uniform(0.5, 1.5, K)).astype(np.float32) if per_channel else 0.004
    oa = float(np.float32(ia * 0.004 * np.sqrt(C * R * R) * 40.0))
    if dtype == "i8":
        xs, ws = x.view(np.int8), w.view(np.int8)
        want, want_acc = orc.conv2d_i8(xs, ws, b, pad, st, 1, ia, 0.004, oa, 7, return_acc=True)
        if per_channel:
            want = orc.requant_per_channel_i8(want_acc, ia, wa, oa, 7)
        plan = hipq.Conv2d(x.shape, ws, b, pad, st, 1, ia, 0, wa, 0, oa, 0, obits=7, dtype=hipq.DTYPE_I8)
        want = want.view(np.uint8)
    else:
        want, want_acc = orc.conv2d_u8(x, w, b, pad, st, 1, ia, izp, 0.004, wzp, oa, ozp, return_acc=True)
        if per_channel:
            want = orc.conv2d_u8_per_channel(x, w, b, pad, st, 1, ia, izp, wa, wzp, oa, ozp)
        plan = hipq.Conv2d(x.shape, w, b, pad, st, 1, ia, izp, wa, wzp, oa, ozp)
    assert len(np.unique(want)) > 8
    xd = hipq.to_device_nhwc(x)
    res = rng.integers(0, 256, want.shape, dtype=np.uint8)
    rd = hipq.to_device_nhwc(res)
    ran = 0
    for mb, nb, nwc, ks in SHAPES:
        try:
            plan.resident(16 * mb, 16 * nb, nwc, ks)
        except hipq.HipqError:
            assert C >= 1024  # the region of a fully-connected layer's rows does not fit LDS
            continue
        print("resident", case, (mb, nb, nwc, ks), plan.kernel, flush=True)
        assert plan.kernel.startswith("conv_mfma_i8_resident_%dx%d" % (16 * mb, 16 * nb * nwc)), plan.kernel
        got = hipq.from_device_nhwc(plan(xd, torch.full_like(plan.empty_output(), 99)), K)
        assert np.array_equal(got, want), (mb, nb, nwc, ks, int((got != want).sum()), np.argwhere(got != want)[:6].tolist())
        acc = torch.zeros((N, plan.OH, plan.OW, plan.desc.out_cs), dtype=torch.int32, device="cuda")
        got = hipq.from_device_nhwc(plan(xd, acc=acc), K)
        assert np.array_equal(acc.cpu().numpy()[..., :K].transpose(0, 3, 1, 2), want_acc) and np.array_equal(got, want), (mb, nb, nwc, ks, "acc")
        if dtype == "u8":
            first = bool(ran & 1)
            ra = float(np.float32(oa * (300.0 if ran % 5 == 4 else 1.4)))  # the general form of the add too
            sa = float(np.float32(max(oa, ra) * 1.3))
            y = plan.run_add(xd, rd, first, ra, 9, sa, 20, plan.empty_output())
            added = orc.add_u8(res, want, ra, 9, oa, ozp, sa, 20) if first else orc.add_u8(want, res, oa, ozp, ra, 9, sa, 20)
            assert np.array_equal(hipq.from_device_nhwc(y, K), added), (mb, nb, nwc, ks, "add", first)
            assert np.array_equal(hipq.from_device_nhwc(plan.run_relu(xd), K), np.maximum(want, ozp)), (mb, nb, nwc, ks, "relu")
            if plan.dequant_fusable(oa, ozp):
                f = torch.full((N, K), 7.0, dtype=torch.float32, device="cuda")
                plan.run_dequant(xd, f)
                exact = np.ascontiguousarray(orc.dequantize_u8(want.reshape(N, K), oa, ozp))
                assert np.array_equal(f.cpu().numpy().view(np.uint32), exact.view(np.uint32)), (mb, nb, nwc, ks, "floats")
        ran += 1
    assert ran >= 8
    with pytest.raises(hipq.HipqError):
        plan.resident(48, 16, 1, 8)
    plan.resident()
    assert np.array_equal(hipq.from_device_nhwc(plan(xd), K), want), plan.kernel


RECTANGULAR = [  # N, C, H, W, K, (R, S), (pad_h, pad_w), (stride_h, stride_w), data type, weight zero point
    (2, 64, 13, 9, 72, (1, 7), (0, 3), (1, 1), "u8", 128),    # a slab is a whole tap
    (3, 128, 11, 16, 40, (7, 1), (3, 0), (1, 2), "u8", 128),
    (2, 64, 9, 14, 130, (3, 5), (0, 2), (2, 1), "u8", 128),
    (4, 256, 7, 10, 24, (1, 1), (0, 0), (1, 3), "u8", 128),   # 1x1 with a stride in one direction
    (5, 48, 8, 5, 33, (5, 3), (2, 1), (1, 3), "u8", 128),     # pieces of a slab in different taps
    (2, 16, 12, 30, 20, (1, 29), (0, 14), (1, 1), "u8", 128),  # as many taps as the masks hold, in one row
    (1, 32, 31, 6, 20, (29, 1), (14, 0), (2, 1), "u8", 128),  # in one column
    (2, 80, 10, 7, 50, (4, 2), (1, 0), (3, 1), "i8", 0),      # windows of an even height
    (2, 20, 9, 12, 17, (2, 5), (0, 1), (2, 3), "u8", 90),     # the weight zero point's sums
]


@pytest.mark.parametrize("case", RECTANGULAR, ids=lambda c: "-".join(map(str, c)).replace(" ", ""))
def test_windows_pads_and_strides_that_differ_by_direction(case):
    N, C, H, W, K, (R, S), pad, st, dtype, wzp = case
    rng = np.random.default_rng(N * 1000 + C + R)
    x = rng.integers(0, 256, (N, C, H, W), dtype=np.uint8)
    w = rng.integers(*((0, 256) if wzp in (0, 128) else (wzp - 90, wzp + 91)), (K, C, R, S), dtype=np.uint8)
    b = rng.integers(-30000, 30000, K).astype(np.int32)
    oa = float(np.float32(0.02 * 0.004 * np.sqrt(C * R * S) * 40.0))
    if dtype == "i8":
        xs, ws = x.view(np.int8), w.view(np.int8)
        want, want_acc = orc.conv2d_i8(xs, ws, b, pad, st, 1, 0.02, 0.004, oa, 7, return_acc=True)
        want = want.view(np.uint8)
        plan = hipq.Conv2d(x.shape, ws, b, pad, st, 1, 0.02, 0, 0.004, 0, oa, 0, obits=7, dtype=hipq.DTYPE_I8)
    else:
        want, want_acc = orc.conv2d_u8(x, w, b, pad, st, 1, 0.02, 77, 0.004, wzp, oa, 120, return_acc=True)
        plan = hipq.Conv2d(x.shape, w, b, pad, st, 1, 0.02, 77, 0.004, wzp, oa, 120)
    assert len(np.unique(want)) > 8
    xd = hipq.to_device_nhwc(x)
    for mb, nb, nwc, ks in SHAPES:
        plan.resident(16 * mb, 16 * nb, nwc, ks)
        print("resident", case, (mb, nb, nwc, ks), plan.kernel, flush=True)
        got = hipq.from_device_nhwc(plan(xd, torch.full_like(plan.empty_output(), 99)), K)
        assert np.array_equal(got, want), (mb, nb, nwc, ks, int((got != want).sum()), np.argwhere(got != want)[:6].tolist())
        acc = torch.zeros((N, plan.OH, plan.OW, plan.desc.out_cs), dtype=torch.int32, device="cuda")
        plan(xd, acc=acc)
        assert np.array_equal(acc.cpu().numpy()[..., :K].transpose(0, 3, 1, 2), want_acc), (mb, nb, nwc, ks, "acc")


@pytest.mark.parametrize("case", [(1, 64, 56, 56, 128, 3, 1, 2, 128), (1, 256, 14, 14, 256, 3, 1, 1, 128), (11, 2048, 7, 7, 512, 1, 0, 1, 128),
                                  (2, 242, 27, 31, 130, 5, 2, 2, 128), (4, 100, 40, 40, 120, 3, 1, 1, 101)], ids=lambda c: "-".join(map(str, c)))
def test_the_built_in_rule_takes_the_kernel(case):
    N, C, H, W, K, R, pad, st, wzp = case
    rng = np.random.default_rng(C)
    x = rng.integers(0, 256, (N, C, H, W), dtype=np.uint8)
    w = rng.integers(wzp - 90, wzp + 91, (K, C, R, R), dtype=np.uint8)
    b = rng.integers(-30000, 30000, K).astype(np.int32)
    q = (0.02, 77, 0.004, wzp, float(np.float32(0.02 * 0.004 * np.sqrt(C * R * R) * 40.0)), 120)
    plan = hipq.Conv2d(x.shape, w, b, pad, st, 1, *q)
    assert plan.kernel.startswith("conv_mfma_i8_resident_"), plan.kernel
    want = orc.conv2d_u8(x, w, b, pad, st, 1, *q)
    assert np.array_equal(hipq.from_device_nhwc(plan(hipq.to_device_nhwc(x)), K), want)


def test_layers_outside_the_kernels_range_stay_where_they_were():
    """More taps than a mask holds, pads of half the window and more: refused by name, and computed by another kernel."""
    rng = np.random.default_rng(5)
    for R, S, pad, st in ((7, 7, 3, 1), (5, 6, 0, 1), (3, 3, 2, 1), (2, 2, 1, 1), (1, 1, 1, 1)):
        x = rng.integers(0, 256, (2, 32, 12, 13), dtype=np.uint8)
        w = rng.integers(0, 256, (24, 32, R, S), dtype=np.uint8)
        q = (0.02, 77, 0.004, 128, float(np.float32(0.02 * 0.004 * np.sqrt(32 * R * S) * 40.0)), 120)
        plan = hipq.Conv2d(x.shape, w, None, pad, st, 1, *q)
        assert "_resident_" not in plan.kernel
        with pytest.raises(hipq.HipqError):
            plan.resident(32, 16, 1, 4)
        assert np.array_equal(hipq.from_device_nhwc(plan(hipq.to_device_nhwc(x)), 24), orc.conv2d_u8(x, w, None, pad, st, 1, *q)), (R, S, pad)


WIDE = [c for c in CASES if c[10] in (0, 128)] + [
    (3, 96, 13, 21, 200, 3, 1, 1, "i8", True, 0),    # a step lies in one tap, a slab does not
    (2, 32, 40, 37, 40, 3, 1, 2, "u8", False, 128),   # a step is a whole tap
    (1, 272, 9, 9, 260, 3, 0, 1, "u8", True, 128),    # an odd number of pieces a tap, an odd number of steps
    (2, 48, 17, 15, 112, 5, 2, 1, "i8", False, 0),
]


@pytest.mark.parametrize("case", WIDE, ids=lambda c: "-".join(map(str, c)))
def test_resident_kernel_with_32x32_tiles_matches_the_oracle(case):
    """Every tile of a wave and several numbers of waves; what the form does not compute - accumulators, an add outside the 32-bit form, an
    add with scales per channel - another kernel does."""
    N, C, H, W, K, R, pad, st, dtype, per_channel, wzp = case
    rng = np.random.default_rng(C + K)
    x = rng.integers(0, 256, (N, C, H, W), dtype=np.uint8)
    w = rng.integers(0, 256, (K, C, R, R), dtype=np.uint8)
    b = rng.integers(-30000, 30000, K).astype(np.int32)
    ia, izp, ozp = 0.02, 77, 120
    wa = (0.004 * rng.uniform(0.5, 1.5, K)).astype(np.float32) if per_channel else 0.004
    oa = float(np.float32(ia * 0.004 * np.sqrt(C * R * R) * 40.0))  # some values saturate on either side
    if dtype == "i8":
        xs, ws = x.view(np.int8), w.view(np.int8)
        want, want_acc = orc.conv2d_i8(xs, ws, b, pad, st, 1, ia, 0.004, oa, 7, return_acc=True)
        if per_channel:
            want = orc.requant_per_channel_i8(want_acc, ia, wa, oa, 7)
        plan = hipq.Conv2d(x.shape, ws, b, pad, st, 1, ia, 0, wa, 0, oa, 0, obits=7, dtype=hipq.DTYPE_I8)
        want = want.view(np.uint8)
    else:
        want, want_acc = orc.conv2d_u8(x, w, b, pad, st, 1, ia, izp, 0.004, wzp, oa, ozp, return_acc=True)
        if per_channel:
            want = orc.conv2d_u8_per_channel(x, w, b, pad, st, 1, ia, izp, wa, wzp, oa, ozp)
        plan = hipq.Conv2d(x.shape, w, b, pad, st, 1, ia, izp, wa, wzp, oa, ozp)
    xd = hipq.to_device_nhwc(x)
    res = rng.integers(0, 256, want.shape, dtype=np.uint8)
    rd = hipq.to_device_nhwc(res)
    ran = 0
    for mb, nb in ((8, 4), (8, 2), (4, 4), (4, 2)):
        for waves in (1, 3, 8):
            try:
                plan.resident(16 * mb, 16 * nb, waves, 0)
            except hipq.HipqError:
                assert C >= 512  # the region does not fit LDS
                continue
            print("wide", case, (mb, nb, waves), plan.kernel, flush=True)
            assert plan.kernel.startswith("conv_mfma_i8_resident_%dx%d" % (16 * mb, 16 * nb * waves)), plan.kernel
            got = hipq.from_device_nhwc(plan(xd, torch.full_like(plan.empty_output(), 99)), K)
            assert np.array_equal(got, want), (mb, nb, waves, int((got != want).sum()), np.argwhere(got != want)[:6].tolist())
            if dtype == "u8":
                assert np.array_equal(hipq.from_device_nhwc(plan.run_relu(xd), K), np.maximum(want, ozp)), (mb, nb, waves, "relu")
                ra = float(np.float32(oa * (300.0 if ran % 3 == 2 else 1.4)))  # the general form of the add too
                sa = float(np.float32(max(oa, ra) * 1.3))
                first = bool(ran & 1)
                y = plan.run_add(xd, rd, first, ra, 9, sa, 20, plan.empty_output())
                added = orc.add_u8(res, want, ra, 9, oa, ozp, sa, 20) if first else orc.add_u8(want, res, oa, ozp, ra, 9, sa, 20)
                assert np.array_equal(hipq.from_device_nhwc(y, K), added), (mb, nb, waves, "add", first)
            ran += 1
    if ran:
        acc = torch.zeros((N, plan.OH, plan.OW, plan.desc.out_cs), dtype=torch.int32, device="cuda")
        got = hipq.from_device_nhwc(plan(xd, acc=acc), K)
        assert np.array_equal(acc.cpu().numpy()[..., :K].transpose(0, 3, 1, 2), want_acc) and np.array_equal(got, want), "acc"
    assert ran or C >= 512


def test_32x32_tiles_keep_out_of_what_they_do_not_compute():
    """A weight zero point, eight signed bits (whose low byte wraps), channels that are no multiple of 16 to store, an odd tile."""
    rng = np.random.default_rng(9)
    x = rng.integers(0, 256, (2, 64, 20, 20), dtype=np.uint8)
    w = rng.integers(0, 256, (64, 64, 3, 3), dtype=np.uint8)

    def refused(plan, *shape):
        with pytest.raises(hipq.HipqError):
            plan.resident(*(shape or (64, 32, 2, 0)))
    refused(hipq.Conv2d(x.shape, w, None, 1, 1, 1, 0.02, 77, 0.004, 101, 0.5, 120))
    refused(hipq.Conv2d(x.shape, w.view(np.int8), None, 1, 1, 1, 0.02, 0, 0.004, 0, 0.5, 0, obits=8, dtype=hipq.DTYPE_I8))
    refused(hipq.Conv2d(x.shape, w[:3], None, 1, 1, 1, 0.02, 77, 0.004, 128, 0.5, 120))
    for shape in ((96, 32, 2, 0), (64, 48, 2, 0), (64, 32, 9, 0), (32, 32, 2, 0)):
        refused(hipq.Conv2d(x.shape, w, None, 1, 1, 1, 0.02, 77, 0.004, 128, 0.5, 120), *shape)


@pytest.mark.parametrize("case, wide", [((5, 96, 75, 67, 200, 3, "i8"), True), ((26, 46, 101, 103, 83, 3, "u8"), True), ((1, 64, 14, 14, 128, 5, "u8"), False)],
                         ids=["ragged_i8", "large", "small"])
def test_the_rule_takes_32x32_tiles_where_there_is_work(case, wide):
    N, C, H, W, K, R, dtype = case
    i8 = dtype == "i8"
    plan = hipq.Conv2d((N, C, H, W), np.ones((K, C, R, R), np.int8 if i8 else np.uint8), None, R // 2, 1, 1, 0.02, 0 if i8 else 128,
                       np.full(K, 0.005, np.float32) if i8 else 0.005, 0 if i8 else 128, 0.1, 0 if i8 else 120, obits=7 if i8 else 8,
                       dtype=hipq.DTYPE_I8 if i8 else hipq.DTYPE_U8)
    pixels, channels = (int(v) for v in plan.kernel.split("_resident_")[1].split("_")[0].split("x")) if "_resident_" in plan.kernel else (0, 0)
    print(plan.kernel)
    built = {(16 * mb, 16 * nb * nwc) for mb, nb, nwc, ks in SHAPES}
    assert (pixels in (64, 128) and (pixels, channels) not in built) == wide, plan.kernel


PAIRS = [  # N, (C, H, W, K, R, stride) of both layers: a block's first layer and its shortcut, and layers of other inputs
    (1, (64, 56, 56, 128, 3, 2), (64, 56, 56, 128, 1, 2)),
    (2, (512, 7, 7, 512, 3, 1), (256, 14, 14, 512, 1, 2)),
    (3, (128, 13, 11, 72, 3, 2), (128, 13, 11, 40, 1, 2)),   # ragged in pixels and channels
    (16, (64, 40, 40, 128, 3, 2), (64, 40, 40, 128, 1, 2)),  # many tiles of both
    (1, (64, 5, 5, 16, 1, 1), (1024, 3, 3, 264, 3, 1)),      # one tile beside many slabs, the smaller layer first
    (5, (64, 9, 7, 200, 5, 1), (192, 1, 1, 33, 1, 1)),       # 25 taps; fully connected
]


@pytest.mark.parametrize("case", PAIRS, ids=lambda c: "-".join("x".join(map(str, v)) if isinstance(v, tuple) else str(v) for v in c))
def test_two_layers_in_one_launch_match_the_oracle(case):
    N, *layers = case
    rng = np.random.default_rng(77 + N + layers[0][0])
    plans, xs, wants = [], [], []
    for C, H, W, K, R, st in layers:
        x = rng.integers(0, 256, (N, C, H, W), dtype=np.uint8)
        w = rng.integers(0, 256, (K, C, R, R), dtype=np.uint8)
        b = rng.integers(-30000, 30000, K).astype(np.int32)
        q = (0.02, int(rng.integers(0, 256)), 0.004, 128, float(np.float32(0.02 * 0.004 * np.sqrt(C * R * R) * 150.0)), int(rng.integers(60, 160)))
        plans.append(hipq.Conv2d(x.shape, w, b, R // 2, st, 1, *q))
        xs.append(hipq.to_device_nhwc(x))
        wants.append((orc.conv2d_u8(x, w, b, R // 2, st, 1, *q), q[5]))
    plans[0].special(2)
    for relus in ((False, False), (True, False), (False, True)):
        assert hipq.pair_fusable(*plans)
        ys = [p.empty_output().fill_(7) for p in plans]
        hipq.run_pair(plans[0], xs[0], ys[0], plans[1], xs[1], ys[1], *relus)
        torch.cuda.synchronize()
        for y, (want, ozp), relu, layer in zip(ys, wants, relus, layers):
            want = np.maximum(want, ozp).astype(np.uint8) if relu else want
            bad = hipq.from_device_nhwc(y, layer[3]) != want
            assert not bad.any(), (layer, relu, int(bad.sum()), np.argwhere(bad)[:8].tolist())
            assert len(np.unique(want)) > 8


def test_what_does_not_run_as_a_pair():
    """int8 tensors, weight zero points, scales per channel, channels that are no multiple of 64, more work than the rule allows, and a layer
    that writes what the other reads."""
    def layer(N=1, C=64, H=14, K=64, dtype=hipq.DTYPE_U8, wzp=128, wa=0.004):
        i8 = dtype == hipq.DTYPE_I8
        w = np.ones((K, C, 3, 3), np.int8 if i8 else np.uint8)
        return hipq.Conv2d((N, C, H, H), w, None, 1, 1, 1, 0.02, 0 if i8 else 120, wa, 0 if i8 else wzp, 0.1, 0 if i8 else 120, obits=7 if i8 else 8, dtype=dtype)
    good = layer()
    assert hipq.pair_fusable(good, layer()) and not hipq.pair_fusable(layer(64, 256, 28, 256), good)
    for other in (layer(dtype=hipq.DTYPE_I8), layer(wzp=101), layer(wa=np.full(64, 0.004, np.float32)), layer(C=48)):
        assert not hipq.pair_fusable(good, other) and not hipq.pair_fusable(other, good)
    x, y = torch.zeros((1, 14, 14, 64), dtype=torch.uint8, device="cuda"), good.empty_output()
    with pytest.raises(hipq.HipqError, match="do not run in one launch"):
        hipq.run_pair(good, x, y, layer(wzp=101), x, torch.zeros_like(y))
    with pytest.raises(hipq.HipqError, match="neither layer"):
        hipq.run_pair(good, x, y, layer(), y, torch.zeros_like(y))
