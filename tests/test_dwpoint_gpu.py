"""A depthwise 3x3 layer and the 1x1 layer behind it as one kernel, against the reference's arithmetic (pytest.mark.gpu)."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import orc  # noqa: E402  (checker only)
from nart_amd import hipq  # noqa: E402

# channels, output channels, (N, H, W), stride: one slice and one tile; a half slice and partial tiles; more slices than waves; images
# that a patch just fills, that it overhangs on two sides, and smaller than one; work-groups with idle waves (5 images); six, seven and as
# many waves as slices in a work-group
CASES = [(32, 16, (5, 8, 8), 1), (32, 16, (5, 15, 16), 2), (80, 72, (3, 13, 11), 1), (80, 72, (3, 13, 11), 2), (560, 160, (2, 7, 7), 1),
         (576, 320, (1, 7, 7), 1), (560, 160, (2, 14, 14), 2), (20, 20, (1, 3, 2), 1), (24, 200, (1, 3, 2), 2),
         (192, 40, (2, 9, 10), 2), (224, 40, (1, 6, 9), 1), (512, 48, (1, 9, 9), 2)]
SHAPES = ["4x8_n1", "4x8_n2", "4x8_n3", "4x8_n5", "8x8_n1", "8x8_n2", "8x8_n3", "narrow4x8_n1", "narrow4x8_n2", "narrow8x8_n1", "narrow8x8_n2"]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "%dto%d_%dx%dx%d_s%d" % (c[0], c[1], *c[2], c[3]))
def test_every_shape(case):
    """Every division of the work gives the oracle's bytes: without and with the ReLU clamp between the layers, and with an add, the
    residual on either side."""
    ci, co, (N, H, W), st = case
    rng = np.random.default_rng(ci + co + H)
    x = rng.integers(0, 256, (N, ci, H, W), dtype=np.uint8)
    t, a, z, plans, outs = x, 0.03, 77, [], []
    for k, (C, K, R, s, group) in enumerate(((ci, ci, 3, st, ci), (ci, co, 1, 1, 1))):
        w = rng.integers(1, 256, (K, C // group, R, R), dtype=np.uint8)
        sigma = 74.0 * 74.0 * math.sqrt(w[0].size) * (0.7 if k else 1.0)
        b = rng.integers(-int(sigma), int(sigma) + 1, K).astype(np.int32)
        oa = float(np.float32(0.03 * rng.uniform(0.75, 1.35)))
        q = (a, z, float(np.float32(oa * 45.0 / (a * sigma))), 128, oa, 30 if k == 0 else 120)
        plans.append(hipq.Conv2d(t.shape, w, b, R // 2, s, group, *q))
        outs.append((w, b, R // 2, s, group, q))
        t = orc.conv2d_u8(t, w, b, R // 2, s, group, *q)
        a, z = q[4], q[5]
    want = {}
    for relu in (False, True):
        t = orc.conv2d_u8(x, *outs[0][:5], *outs[0][5])
        if relu:
            t = np.maximum(t, outs[0][5][5]).astype(np.uint8)
        want[relu] = orc.conv2d_u8(t, *outs[1][:5], *outs[1][5])
        assert len(np.unique(want[relu])) > min(8, want[relu].size // 2)
    r = rng.integers(0, 256, want[True].shape, dtype=np.uint8)
    plans[1].special(2)
    assert hipq.depthwise_point_fusable(*plans)
    xd, rd = hipq.to_device_nhwc(x), hipq.to_device_nhwc(r)
    for i, shape in enumerate(SHAPES):
        if (st == 2 and "8x8" in shape) or (ci > 32 and "narrow" in shape):
            continue  # not built
        hipq.depthwise_point_select(plans[1], i)
        name = hipq.depthwise_point_kernel(*plans)
        assert name == "conv_dwpoint_s%d_%s" % (st, shape)
        print(case, name, flush=True)
        for relu in (False, True):
            y = hipq.depthwise_point_run(*plans, xd, torch.full_like(plans[1].empty_output(), 99), relu=relu)
            got = hipq.from_device_nhwc(y, co)
            assert np.array_equal(got, want[relu]), (name, relu, int((got != want[relu]).sum()), np.argwhere(got != want[relu])[:8].tolist())
        for first in (False, True):
            s = (r, want[True], 0.041, 90, a, z) if first else (want[True], r, a, z, 0.041, 90)
            y = hipq.depthwise_point_run(*plans, xd, torch.full_like(rd, 99), rd, (first, 0.041, 90, 0.05, 100), relu=True)
            assert np.array_equal(hipq.from_device_nhwc(y, co), orc.add_u8(*s, 0.05, 100)), (name, "add", first)


def test_refusals():
    """What the kernel does not compute is refused, not computed wrongly."""
    w3, w1 = np.full((32, 1, 3, 3), 130, np.uint8), np.full((16, 32, 1, 1), 131, np.uint8)
    b3, b1 = np.zeros(32, np.int32), np.zeros(16, np.int32)
    d = hipq.Conv2d((1, 32, 8, 8), w3, b3, 1, 1, 32, 0.03, 77, 0.01, 128, 0.03, 30)
    for pq in ((0.04, 30, 0.01, 128, 0.03, 120), (0.03, 31, 0.01, 128, 0.03, 120), (0.03, 30, 0.01, 127, 0.03, 120)):
        p = hipq.Conv2d((1, 32, 8, 8), w1, b1, 0, 1, 1, *pq)
        p.special(2)
        assert not hipq.depthwise_point_fusable(d, p), pq
        with pytest.raises(RuntimeError):
            hipq.depthwise_point_run(d, p, torch.zeros((1, 8, 8, 32), dtype=torch.uint8, device="cuda"), p.empty_output())
