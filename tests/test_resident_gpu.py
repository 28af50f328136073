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
