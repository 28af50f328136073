"""GPU parity of hipq_bottleneck_run - an identity bottleneck block (1x1, 3x3, 1x1, residual add) in one launch - against
the CPU oracle's four operators, bit for bit, through the C ABI."""
import math
import sys
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from oracle import orc  # noqa: E402  (checker only)
from nart_amd import hipq  # noqa: E402


def make_block(rng, N, CW, H, W, ozps=(0, 0, None)):
    """Seeded tensors and quantisation parameters of one identity block: widths CW -> CW/4 -> CW/4 -> CW."""
    CM = CW // 4
    xa, xz = 0.05, int(rng.integers(0, 256))
    x = rng.integers(0, 256, (N, CW, H, W), dtype=np.uint8)
    layers = []
    ia, iz = xa, xz
    for (K, C, k), oz in zip(((CM, CW, 1), (CM, CM, 3), (CW, CM, 1)), ozps):
        w = rng.integers(1, 256, (K, C, k, k), dtype=np.uint8)
        sigma = 74.0 * 74.0 * math.sqrt(C * k * k)
        b = rng.integers(-int(sigma), int(sigma) + 1, K).astype(np.int32)
        oa = float(np.float32(ia * rng.uniform(0.75, 1.35)))
        wa = float(np.float32(oa * 40.0 / (ia * sigma)))
        oz = int(rng.integers(96, 160)) if oz is None else oz
        layers.append(dict(w=w, b=b, pad=k // 2, q=(ia, iz, wa, 128, oa, oz)))
        ia, iz = oa, oz
    sa = float(np.float32(math.hypot(ia, xa) * 1.1))
    return x, (xa, xz), layers, (sa, int(rng.integers(0, 40)))


def oracle_block(x, xq, layers, sq, res_first):
    t = x
    for L in layers:
        t = orc.conv2d_u8(t, L["w"], L["b"], L["pad"], 1, 1, *L["q"])
    q3 = layers[2]["q"]
    if res_first:
        return orc.add_u8(x, t, xq[0], xq[1], q3[4], q3[5], sq[0], sq[1])
    return orc.add_u8(t, x, q3[4], q3[5], xq[0], xq[1], sq[0], sq[1])


def plans_of(x, layers, stride=1):
    """stride: of the first layer (a 3x3 / pad 1 layer when it is 2)."""
    shape = x.shape
    plans = []
    for L in layers:
        st = stride if not plans else 1
        p = hipq.Conv2d(shape, L["w"], L["b"], L["pad"], st, 1, *L["q"])
        plans.append(p)
        if len(plans) == 1:
            p.special(2)  # the block kernel wherever it applies, not only where the built-in rule uses it
        shape = (shape[0], L["w"].shape[0], (shape[2] - 1) // st + 1, (shape[3] - 1) // st + 1)
    return plans


CASES = [  # N, CW, H, W
    (2, 1024, 14, 14), (1, 512, 28, 28), (1, 256, 28, 35), (3, 1024, 7, 7), (2, 512, 14, 7), (1, 256, 7, 14), (1, 1024, 21, 14),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "x".join(map(str, c)))
def test_bottleneck_block(case):
    N, CW, H, W = case
    rng = np.random.default_rng(1000 + CW + H)
    for res_first, ozps in ((False, (0, 0, None)), (True, (7, 200, None))):
        x, xq, layers, sq = make_block(rng, N, CW, H, W, ozps)
        plans = plans_of(x, layers)
        print("block case", case, res_first, [p.kernel for p in plans], flush=True)
        assert hipq.bottleneck_fusable(*plans, res_first, sq[0], sq[1]), hipq.lib().hipq_last_error()
        want = oracle_block(x, xq, layers, sq, res_first)
        xd = hipq.to_device_nhwc(x)
        y = torch.zeros_like(xd)
        hipq.bottleneck_run(*plans, xd, res_first, sq[0], sq[1], y)
        torch.cuda.synchronize()
        got = hipq.from_device_nhwc(y, CW)
        bad = got != want
        assert not bad.any(), (case, res_first, int(bad.sum()), np.argwhere(bad)[:8].tolist())
        # the three existing entry points give the same bytes
        t1 = plans[0](xd)
        t2 = plans[1](t1)
        y2 = torch.zeros_like(xd)
        plans[2].run_add(t2, xd, res_first, xq[0], xq[1], sq[0], sq[1], y2)
        torch.cuda.synchronize()
        assert torch.equal(y, y2)
        # the same with the next stage's first layer (CW -> CW / 2) computed in the kernel as well
        CN = CW // 2
        wn = rng.integers(1, 256, (CN, CW, 1, 1), dtype=np.uint8)
        sigma = 74.0 * 74.0 * math.sqrt(CW)
        bn = rng.integers(-int(sigma), int(sigma) + 1, CN).astype(np.int32)
        oan = float(np.float32(sq[0] * rng.uniform(0.75, 1.35)))
        qn = (sq[0], sq[1], float(np.float32(oan * 40.0 / (sq[0] * sigma))), 128, oan, int(rng.integers(20, 60)))
        pn = hipq.Conv2d((N, CW, H, W), wn, bn, 0, 1, 1, *qn, relu=res_first)
        assert hipq.bottleneck_conv_fusable(*plans, res_first, sq[0], sq[1], pn), hipq.lib().hipq_last_error()
        y3, yn = torch.zeros_like(xd), torch.zeros((N, H, W, CN), dtype=torch.uint8, device="cuda")
        hipq.bottleneck_run_conv(*plans, xd, res_first, sq[0], sq[1], y3, pn, yn)
        torch.cuda.synchronize()
        assert torch.equal(y3, y)
        wantn = orc.conv2d_u8(want, wn, bn, 0, 1, 1, *qn)
        if res_first:
            wantn = np.maximum(wantn, qn[5]).astype(np.uint8)
        gotn = hipq.from_device_nhwc(yn, CN)
        bad = gotn != wantn
        assert not bad.any(), (case, "next layer", int(bad.sum()), np.argwhere(bad)[:8].tolist())
        assert len(np.unique(wantn)) > 8


TAIL_CASES = [  # N, CW, H, W: patches of 8 x 8, 4 x 14 and 7 x 7 pixels; 64, 128 and 256 middle channels
    (1, 256, 16, 24), (2, 512, 8, 28), (2, 256, 14, 21), (1, 1024, 8, 8), (1, 512, 56, 8), (3, 256, 4, 14), (1, 1024, 7, 7),
]


def make_tail(rng, N, CW, H, W, relu_next, wide_next=False, in_hw=None):
    """The block from its 3x3 layer on: t1 [N, CM, H, W] -> 3x3 -> 1x1 to CW -> add(., residual) -> 1x1 back to CM (to
    2 CM with wide_next: the first layer of the next stage).  in_hw: the size of t1 where the 3x3 layer has stride 2 and
    H x W is its output."""
    CM = CW // 4
    CN = 2 * CM if wide_next else CM
    t1 = rng.integers(0, 256, (N, CM) + tuple(in_hw or (H, W)), dtype=np.uint8)
    res = rng.integers(0, 256, (N, CW, H, W), dtype=np.uint8)
    ia, iz = 0.04, int(rng.integers(0, 256))
    layers = []
    for (K, C, k), oz in zip(((CM, CM, 3), (CW, CM, 1)), (int(rng.integers(0, 30)), None)):
        w = rng.integers(1, 256, (K, C, k, k), dtype=np.uint8)
        sigma = 74.0 * 74.0 * math.sqrt(C * k * k)
        b = rng.integers(-int(sigma), int(sigma) + 1, K).astype(np.int32)
        oa = float(np.float32(ia * rng.uniform(0.75, 1.35)))
        wa = float(np.float32(oa * 40.0 / (ia * sigma)))
        oz = int(rng.integers(96, 160)) if oz is None else oz
        layers.append(dict(w=w, b=b, pad=k // 2, q=(ia, iz, wa, 128, oa, oz)))
        ia, iz = oa, oz
    ra, rz = float(np.float32(ia * rng.uniform(0.6, 1.6))), int(rng.integers(0, 256))
    sa, sz = float(np.float32(math.hypot(ia, ra) * 1.1)), int(rng.integers(0, 40))
    w = rng.integers(1, 256, (CN, CW, 1, 1), dtype=np.uint8)
    sigma = 74.0 * 74.0 * math.sqrt(CW)
    b = rng.integers(-int(sigma), int(sigma) + 1, CN).astype(np.int32)
    oa = float(np.float32(sa * rng.uniform(0.75, 1.35)))
    nxt = dict(w=w, b=b, pad=0, q=(sa, sz, float(np.float32(oa * 40.0 / (sa * sigma))), 128, oa, int(rng.integers(20, 60))), relu=relu_next)
    return t1, res, layers, (ra, rz), (sa, sz), nxt


@pytest.mark.parametrize("case", TAIL_CASES, ids=lambda c: "x".join(map(str, c)))
def test_bottleneck_tail(case):
    """hipq_bottleneck_tail_run == 3x3 convolution, widening convolution, add with any residual and - chained - the next
    1x1 convolution run one by one by the oracle: both operand orders of the add, with and without the chained layer, a
    ReLU on the chained layer, a chained layer of twice the channels, every patch shape and channel count."""
    N, CW, H, W = case
    CM = CW // 4
    rng = np.random.default_rng(2000 + CW + H)
    for res_first, chain, relu_next, wide in ((False, True, False, False), (True, True, True, False), (True, False, False, False),
                                              (False, True, True, True)):
        t1, res, layers, rq, sq, nx = make_tail(rng, N, CW, H, W, relu_next, wide)
        plans = plans_of(t1, layers)
        pn = hipq.Conv2d((N, CW, H, W), nx["w"], nx["b"], 0, 1, 1, *nx["q"])
        print("tail case", case, res_first, chain, relu_next, [p.kernel for p in plans], flush=True)
        assert hipq.bottleneck_tail_fusable(plans[0], plans[1], res_first, rq[0], rq[1], sq[0], sq[1], pn if chain else None)
        t = orc.conv2d_u8(t1, layers[0]["w"], layers[0]["b"], 1, 1, 1, *layers[0]["q"])
        c = orc.conv2d_u8(t, layers[1]["w"], layers[1]["b"], 0, 1, 1, *layers[1]["q"])
        q3 = layers[1]["q"]
        want = orc.add_u8(res, c, rq[0], rq[1], q3[4], q3[5], sq[0], sq[1]) if res_first else orc.add_u8(c, res, q3[4], q3[5], rq[0], rq[1], sq[0], sq[1])
        xd, rd = hipq.to_device_nhwc(t1), hipq.to_device_nhwc(res)
        y = torch.zeros_like(rd)
        yn = torch.zeros((N, H, W, nx["w"].shape[0]), dtype=torch.uint8, device="cuda") if chain else None
        hipq.bottleneck_tail_run(plans[0], plans[1], xd, rd, res_first, rq[0], rq[1], sq[0], sq[1], y, pn if chain else None, yn,
                                 next_relu=relu_next)
        torch.cuda.synchronize()
        got = hipq.from_device_nhwc(y, CW)
        bad = got != want
        assert not bad.any(), (case, res_first, chain, int(bad.sum()), np.argwhere(bad)[:8].tolist())
        if chain:
            wantn = orc.conv2d_u8(want, nx["w"], nx["b"], 0, 1, 1, *nx["q"])
            if relu_next:
                wantn = np.maximum(wantn, nx["q"][5]).astype(np.uint8)
            gotn = hipq.from_device_nhwc(yn, nx["w"].shape[0])
            bad = gotn != wantn
            assert not bad.any(), (case, "next layer", relu_next, int(bad.sum()), np.argwhere(bad)[:8].tolist())


@pytest.mark.parametrize("case", [(2, 512, 28, 28, 56, 56), (1, 512, 8, 16, 15, 32), (2, 512, 7, 14, 13, 27), (1, 512, 4, 14, 8, 28)],
                         ids=lambda c: "x".join(map(str, c)))
def test_bottleneck_tail_with_a_strided_3x3_layer(case):
    """The first block of a stage: the 3x3 layer has stride 2 (even and odd input sizes, every patch shape), the residual is
    any tensor of the output's size (the projection shortcut), with and without the chained layer."""
    N, CW, H, W, IH, IW = case
    CM = CW // 4
    rng = np.random.default_rng(2500 + H + IW)
    for res_first, chain, wide in ((False, True, False), (True, False, False), (True, True, True)):
        t1, res, layers, rq, sq, nx = make_tail(rng, N, CW, H, W, False, wide, (IH, IW))
        plans = plans_of(t1, layers, stride=2)
        pn = hipq.Conv2d((N, CW, H, W), nx["w"], nx["b"], 0, 1, 1, *nx["q"])
        print("strided tail case", case, res_first, chain, wide, [p.kernel for p in plans], flush=True)
        assert hipq.bottleneck_tail_fusable(plans[0], plans[1], res_first, rq[0], rq[1], sq[0], sq[1], pn if chain else None)
        t = orc.conv2d_u8(t1, layers[0]["w"], layers[0]["b"], 1, 2, 1, *layers[0]["q"])
        assert t.shape[2:] == (H, W)
        c = orc.conv2d_u8(t, layers[1]["w"], layers[1]["b"], 0, 1, 1, *layers[1]["q"])
        q3 = layers[1]["q"]
        want = orc.add_u8(res, c, rq[0], rq[1], q3[4], q3[5], sq[0], sq[1]) if res_first else orc.add_u8(c, res, q3[4], q3[5], rq[0], rq[1], sq[0], sq[1])
        xd, rd = hipq.to_device_nhwc(t1), hipq.to_device_nhwc(res)
        y = torch.zeros_like(rd)
        yn = torch.zeros((N, H, W, nx["w"].shape[0]), dtype=torch.uint8, device="cuda") if chain else None
        hipq.bottleneck_tail_run(plans[0], plans[1], xd, rd, res_first, rq[0], rq[1], sq[0], sq[1], y, pn if chain else None, yn)
        torch.cuda.synchronize()
        got = hipq.from_device_nhwc(y, CW)
        bad = got != want
        assert not bad.any(), (case, res_first, chain, int(bad.sum()), np.argwhere(bad)[:8].tolist())
        if chain:
            wantn = orc.conv2d_u8(want, nx["w"], nx["b"], 0, 1, 1, *nx["q"])
            gotn = hipq.from_device_nhwc(yn, nx["w"].shape[0])
            bad = gotn != wantn
            assert not bad.any(), (case, "next layer", int(bad.sum()), np.argwhere(bad)[:8].tolist())
    # 64 or 256 middle channels with a strided 3x3 layer go through the separate entry points
    t1, res, layers, rq, sq, nx = make_tail(rng, 1, 256, 8, 8, False, False, (16, 16))
    plans = plans_of(t1, layers, stride=2)
    assert not hipq.bottleneck_tail_fusable(plans[0], plans[1], False, rq[0], rq[1], sq[0], sq[1])


# the sum's scale over the root of the operands' squares, the residual's over the convolution's: sums in 64 bits, sums in 32 (one ratio of 1 or
# more, of which the exact form has no multiplier), scales far apart, equal ones
ADD_SCALES = [(1.1, 0.83), (1.1, 1.57), (0.66, 0.9), (0.5, 1.0), (1.0, 1.0), (2.0, 1.0), (1.3, 1 / 90), (1.3, 60.0), (3.7, 0.4)]


@pytest.mark.parametrize("scales", ADD_SCALES, ids=lambda s: "%.2f-%.2f" % s)
@pytest.mark.parametrize("case", [(1, 256, 16, 16, 1), (1, 512, 14, 28, 1), (1, 512, 7, 14, 2), (1, 1024, 7, 7, 1)], ids=lambda c: "x".join(map(str, c)))
def test_sums_of_any_pair_of_scales(case, scales):
    N, CW, H, W, st = case
    rng = np.random.default_rng(CW + H + int(scales[0] * 100))
    t1, res, layers, rq, sq, nx = make_tail(rng, N, CW, H, W, False, False, (2 * H, 2 * W) if st == 2 else None)
    q3 = layers[1]["q"]
    ra = float(np.float32(q3[4] * scales[1]))
    sa, sz = float(np.float32(math.hypot(q3[4], ra) * scales[0])), sq[1]
    plans = plans_of(t1, layers, stride=st)
    pn = hipq.Conv2d((N, CW, H, W), nx["w"], nx["b"], 0, 1, 1, sa, sz, *nx["q"][2:])
    t = orc.conv2d_u8(t1, layers[0]["w"], layers[0]["b"], 1, st, 1, *layers[0]["q"])
    c = orc.conv2d_u8(t, layers[1]["w"], layers[1]["b"], 0, 1, 1, *q3)
    xd, rd = hipq.to_device_nhwc(t1), hipq.to_device_nhwc(res)
    for res_first, chain in ((False, False), (True, True)):
        print("scales", case, scales, res_first, chain, flush=True)
        if not hipq.bottleneck_tail_fusable(plans[0], plans[1], res_first, ra, rq[1], sa, sz, pn if chain else None):
            assert max(ra, q3[4]) < sa / 8 or max(ra, q3[4]) > 30 * min(ra, q3[4])  # shifts beyond the fast form's
            continue
        want = orc.add_u8(res, c, ra, rq[1], q3[4], q3[5], sa, sz) if res_first else orc.add_u8(c, res, q3[4], q3[5], ra, rq[1], sa, sz)
        y = torch.zeros_like(rd)
        yn = torch.zeros((N, H, W, nx["w"].shape[0]), dtype=torch.uint8, device="cuda") if chain else None
        hipq.bottleneck_tail_run(plans[0], plans[1], xd, rd, res_first, ra, rq[1], sa, sz, y, pn if chain else None, yn)
        got = hipq.from_device_nhwc(y, CW)
        assert np.array_equal(got, want), (case, scales, res_first, chain, int((got != want).sum()))


def test_bottleneck_refusals():
    """What the one-launch forms do not serve is refused by the predicates and fails loudly in the run entry points."""
    rng = np.random.default_rng(7)
    x, xq, layers, sq = make_block(rng, 1, 256, 10, 14)  # a height that is no multiple of 7
    plans = plans_of(x, layers)
    assert not hipq.bottleneck_fusable(*plans, False, sq[0], sq[1])
    xd = hipq.to_device_nhwc(x)
    with pytest.raises(hipq.HipqError, match="do not run as one kernel"):
        hipq.bottleneck_run(*plans, xd, False, sq[0], sq[1], torch.zeros_like(xd))
    x, xq, layers, sq = make_block(rng, 1, 256, 14, 14)
    plans = plans_of(x, layers)
    xd = hipq.to_device_nhwc(x)
    with pytest.raises(hipq.HipqError, match="cannot overwrite"):
        hipq.bottleneck_run(*plans, xd, False, sq[0], sq[1], xd)
    assert not hipq.bottleneck_fusable(*plans, False, sq[0], sq[1], obits=7)
    # the tail form: a stride-2 3x3 layer, and a chained layer that reads the sum with another zero point
    t1, res, tl, rq, sq2, nx = make_tail(rng, 1, 256, 16, 16, False)
    p2s = hipq.Conv2d(t1.shape, tl[0]["w"], tl[0]["b"], 1, 2, 1, *tl[0]["q"]).special(2)
    p3 = hipq.Conv2d((1, 64, 8, 8), tl[1]["w"], tl[1]["b"], 0, 1, 1, *tl[1]["q"])
    assert not hipq.bottleneck_tail_fusable(p2s, p3, False, rq[0], rq[1], sq2[0], sq2[1])
    plans = plans_of(t1, tl)
    q = list(nx["q"])
    q[1] = (q[1] + 1) % 256
    pn = hipq.Conv2d((1, 256, 16, 16), nx["w"], nx["b"], 0, 1, 1, *q)
    assert hipq.bottleneck_tail_fusable(plans[0], plans[1], False, rq[0], rq[1], sq2[0], sq2[1])
    assert not hipq.bottleneck_tail_fusable(plans[0], plans[1], False, rq[0], rq[1], sq2[0], sq2[1], pn)
    xd, rd = hipq.to_device_nhwc(t1), hipq.to_device_nhwc(res)
    with pytest.raises(hipq.HipqError, match="do not run as one kernel"):
        hipq.bottleneck_tail_run(plans[0], plans[1], xd, rd, False, rq[0], rq[1], sq2[0], sq2[1], torch.zeros_like(rd), pn, torch.zeros_like(xd))


def time_tail(N, CW, HW, reps=50):
    rng = np.random.default_rng(6)
    t1, res, layers, rq, sq, nx = make_tail(rng, N, CW, HW, HW, False)
    plans = plans_of(t1, layers)
    pn = hipq.Conv2d((N, CW, HW, HW), nx["w"], nx["b"], 0, 1, 1, *nx["q"])
    xd, rd = hipq.to_device_nhwc(t1), hipq.to_device_nhwc(res)
    y, yn, t = torch.zeros_like(rd), torch.zeros_like(xd), torch.zeros_like(xd)
    fusable = plans[1].add_conv_fusable(False, rq[0], rq[1], sq[0], sq[1], pn)

    def fused():
        hipq.bottleneck_tail_run(plans[0], plans[1], xd, rd, False, rq[0], rq[1], sq[0], sq[1], y, pn, yn)

    def separate():
        plans[0](xd, t)
        if fusable:
            plans[1].run_add_conv(t, rd, False, rq[0], rq[1], sq[0], sq[1], y, pn, yn)
        else:
            plans[1].run_add(t, rd, False, rq[0], rq[1], sq[0], sq[1], y)
            pn(y, yn)

    out = {}
    for name, fn in (("fused", fused), ("separate", separate)):
        fn()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            for _ in range(10):
                fn()
        for _ in range(3):
            g.replay()
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(reps):
            g.replay()
        e1.record()
        torch.cuda.synchronize()
        out[name] = e0.elapsed_time(e1) / reps / 10 * 1e3
    print("tail N=%d CW=%d %dx%d: fused %.1f us, separate (%s, %s) %.1f us" % (
        N, CW, HW, HW, out["fused"], plans[0].kernel, "expand+add+conv" if fusable else "add, conv", out["separate"]), flush=True)


WREG_CASES = [  # N, C, H, W, K, kernel, stride: 1x1 and 3x3 layers of the 14x14 and 7x7 stages
    (2, 1024, 14, 14, 256, 1, 1), (1, 2048, 7, 7, 512, 1, 1), (3, 512, 7, 7, 2048, 1, 1), (2, 512, 28, 28, 1024, 1, 2),
    (1, 256, 9, 13, 128, 1, 1), (2, 1024, 14, 14, 2048, 1, 2), (2, 512, 7, 7, 512, 3, 1), (1, 256, 28, 28, 256, 3, 2),
    (2, 128, 14, 21, 128, 3, 1), (1, 512, 14, 14, 512, 3, 2), (1, 128, 56, 28, 128, 3, 2), (2, 256, 14, 14, 256, 3, 1),
]


@pytest.mark.parametrize("case", WREG_CASES, ids=lambda c: "x".join(map(str, c)))
def test_register_fed_convolution(case):
    """conv_wreg_kernel (special(3)) against the oracle's convolution and, for 1x1 layers, convolution + add."""
    N, C, H, W, K, k, st = case
    rng = np.random.default_rng(3000 + C + K + k)
    x = rng.integers(0, 256, (N, C, H, W), dtype=np.uint8)
    w = rng.integers(1, 256, (K, C, k, k), dtype=np.uint8)
    sigma = 74.0 * 74.0 * math.sqrt(C * k * k)
    b = rng.integers(-int(sigma), int(sigma) + 1, K).astype(np.int32)
    for relu in (False, True):
        ia, iz = 0.03, int(rng.integers(0, 256))
        oa = float(np.float32(ia * rng.uniform(0.75, 1.35)))
        q = (ia, iz, float(np.float32(oa * 40.0 / (ia * sigma))), 128, oa, int(rng.integers(0, 200)))
        plan = hipq.Conv2d(x.shape, w, b, k // 2, st, 1, *q, relu=relu).special(3)
        print("register-fed case", case, relu, plan.kernel, flush=True)
        assert plan.kernel == "conv_mfma_i8_wreg", plan.kernel
        want = orc.conv2d_u8(x, w, b, k // 2, st, 1, *q)
        if relu:
            want = np.maximum(want, q[5]).astype(np.uint8)
        xd = hipq.to_device_nhwc(x)
        y = plan(xd)
        torch.cuda.synchronize()
        got = hipq.from_device_nhwc(y, K)
        bad = got != want
        assert not bad.any(), (case, relu, int(bad.sum()), np.argwhere(bad)[:8].tolist())
        if k == 1 and not relu:
            for res_first in (False, True):
                res = rng.integers(0, 256, want.shape, dtype=np.uint8)
                ra, rz = float(np.float32(oa * rng.uniform(0.6, 1.6))), int(rng.integers(0, 256))
                sa, sz = float(np.float32(math.hypot(oa, ra) * 1.1)), int(rng.integers(0, 40))
                assert plan.kernel_add == "conv_mfma_i8_wreg+add", plan.kernel_add
                wanta = orc.add_u8(res, want, ra, rz, q[4], q[5], sa, sz) if res_first else orc.add_u8(want, res, q[4], q[5], ra, rz, sa, sz)
                ya = torch.zeros_like(y)
                plan.run_add(xd, hipq.to_device_nhwc(res), res_first, ra, rz, sa, sz, ya)
                torch.cuda.synchronize()
                gota = hipq.from_device_nhwc(ya, K)
                assert np.array_equal(gota, wanta), (case, "add", res_first, int((gota != wanta).sum()))


HREG_CASES = [  # N, C, H, W, K
    (11, 256, 13, 13, 256), (3, 128, 17, 29, 200), (2, 512, 17, 19, 200), (1, 64, 70, 71, 48), (5, 64, 101, 9, 144), (25, 64, 40, 40, 64),
    (900, 512, 1, 1, 256), (20, 256, 2, 40, 128), (64, 256, 14, 14, 256), (40, 128, 25, 26, 128), (1, 128, 90, 91, 128),
]


@pytest.mark.parametrize("case", HREG_CASES, ids=lambda c: "x".join(map(str, c)))
def test_register_fed_convolution_on_any_image(case):
    """conv_hreg_kernel against the oracle's convolution and convolution + add: tiles of 32, 64 and 128 pixels that end inside an
    image, a row or behind the last pixel, images of one pixel, one or two rows, taps that must not leak across borders,
    channel groups that are partly outside the output, both operand orders of the add, a ReLU."""
    N, C, H, W, K = case
    rng = np.random.default_rng(sum(case))
    x = rng.integers(0, 256, (N, C, H, W), dtype=np.uint8)
    w = rng.integers(0, 256, (K, C, 3, 3), dtype=np.uint8)
    sigma = 74.0 * 74.0 * math.sqrt(C * 9)
    b = rng.integers(-int(sigma), int(sigma) + 1, K).astype(np.int32)
    ia, oa = 0.03, float(np.float32(0.03 * rng.uniform(0.75, 1.35)))
    q = (ia, int(rng.integers(0, 256)), float(np.float32(oa * 40.0 / (ia * sigma))), 128, oa, int(rng.integers(0, 200)))
    relu = bool(sum(case) & 1)
    plan = hipq.Conv2d(x.shape, w, b, 1, 1, 1, *q, relu=relu)
    print("any image", case, relu, plan.kernel, flush=True)
    assert "hreg3x3" in plan.kernel and "hreg3x3" in plan.kernel_add, (plan.kernel, plan.kernel_add)
    want = orc.conv2d_u8(x, w, b, 1, 1, 1, *q)
    if relu:
        want = np.maximum(want, q[5]).astype(np.uint8)
    xd = hipq.to_device_nhwc(x)
    got = hipq.from_device_nhwc(plan(xd), K)
    assert np.array_equal(got, want), (case, int((got != want).sum()), np.argwhere(got != want)[:8].tolist())
    res = rng.integers(0, 256, want.shape, dtype=np.uint8)
    ra, rz = float(np.float32(oa * rng.uniform(0.6, 1.6))), int(rng.integers(0, 256))
    sa, sz = float(np.float32(math.hypot(oa, ra) * 1.1)), int(rng.integers(0, 40))
    for res_first in (False, True):
        wanta = orc.add_u8(res, want, ra, rz, q[4], q[5], sa, sz) if res_first else orc.add_u8(want, res, q[4], q[5], ra, rz, sa, sz)
        ya = plan.run_add(xd, hipq.to_device_nhwc(res), res_first, ra, rz, sa, sz, plan.empty_output())
        gota = hipq.from_device_nhwc(ya, K)
        assert np.array_equal(gota, wanta), (case, "add", res_first, int((gota != wanta).sum()))


@pytest.mark.parametrize("case", [(3, 256, 25, 25, 256), (5, 128, 37, 29, 128), (12, 512, 9, 11, 512)], ids=lambda c: "x".join(map(str, c)))
def test_register_fed_stride_2_on_ragged_images(case):
    """conv_wreg_kernel's 7x7 output patches on images whose output is no multiple of 7."""
    N, C, H, W, K = case
    rng = np.random.default_rng(sum(case))
    x = rng.integers(0, 256, (N, C, H, W), dtype=np.uint8)
    w = rng.integers(0, 256, (K, C, 3, 3), dtype=np.uint8)
    b = rng.integers(-50000, 50000, K).astype(np.int32)
    q = (0.03, int(rng.integers(0, 256)), 0.004, 128, float(np.float32(0.03 * 0.004 * 74.0 * 74.0 * math.sqrt(C * 9) / 40.0)), 17)
    plan = hipq.Conv2d(x.shape, w, b, 1, 2, 1, *q).special(3)
    assert plan.kernel == "conv_mfma_i8_wreg", plan.kernel
    want = orc.conv2d_u8(x, w, b, 1, 2, 1, *q)
    y = torch.full_like(plan.empty_output(), 99)
    got = hipq.from_device_nhwc(plan(hipq.to_device_nhwc(x), y), K)
    assert np.array_equal(got, want), (case, int((got != want).sum()))


ADD2_CASES = [  # N, C (widening layer's input channels), output H, W, K, the shortcut's stride
    (2, 256, 14, 14, 1024, 2), (3, 512, 7, 7, 2048, 2), (1, 256, 9, 13, 384, 1), (2, 512, 14, 7, 1024, 1),
]


@pytest.mark.parametrize("case", ADD2_CASES, ids=lambda c: "x".join(map(str, c)))
def test_widening_convolution_shortcut_and_add(case):
    """hipq_conv2d_run_add2: the widening 1x1 convolution of a block, its projection shortcut (1x1, stride 1 or 2, from the
    block's input) and the add, against the oracle's three operators; both operand orders."""
    N, C, H, W, K, st = case
    rng = np.random.default_rng(4000 + C + K + st)
    x = rng.integers(0, 256, (N, C, H, W), dtype=np.uint8)
    xs = rng.integers(0, 256, (N, 2 * C, H * st - (st - 1), W * st - (st - 1)), dtype=np.uint8)

    def layer(Cin):
        w = rng.integers(1, 256, (K, Cin, 1, 1), dtype=np.uint8)
        sigma = 74.0 * 74.0 * math.sqrt(Cin)
        b = rng.integers(-int(sigma), int(sigma) + 1, K).astype(np.int32)
        ia, iz = float(np.float32(rng.uniform(0.02, 0.06))), int(rng.integers(0, 256))
        oa = float(np.float32(ia * rng.uniform(0.75, 1.35)))
        return w, b, (ia, iz, float(np.float32(oa * 40.0 / (ia * sigma))), 128, oa, int(rng.integers(96, 160)))
    w, b, q = layer(C)
    ws_, bs, qs = layer(2 * C)
    pm = hipq.Conv2d(x.shape, w, b, 0, 1, 1, *q).special(2)
    ps = hipq.Conv2d(xs.shape, ws_, bs, 0, st, 1, *qs)
    want_m = orc.conv2d_u8(x, w, b, 0, 1, 1, *q)
    want_s = orc.conv2d_u8(xs, ws_, bs, 0, st, 1, *qs)
    assert want_m.shape == want_s.shape
    xd, xsd = hipq.to_device_nhwc(x), hipq.to_device_nhwc(xs)
    for sc_first in (False, True):
        sa, sz = float(np.float32(math.hypot(q[4], qs[4]) * 1.1)), int(rng.integers(0, 40))
        print("add2 case", case, sc_first, pm.kernel, ps.kernel, flush=True)
        assert hipq.add2_fusable(pm, ps, sc_first, sa, sz)
        want = orc.add_u8(want_s, want_m, qs[4], qs[5], q[4], q[5], sa, sz) if sc_first else orc.add_u8(want_m, want_s, q[4], q[5], qs[4], qs[5], sa, sz)
        y = pm.empty_output()
        hipq.run_add2(pm, xd, ps, xsd, sc_first, sa, sz, y)
        torch.cuda.synchronize()
        got = hipq.from_device_nhwc(y, K)
        bad = got != want
        assert not bad.any(), (case, sc_first, int(bad.sum()), np.argwhere(bad)[:8].tolist())
    # a shortcut with other output channels is refused
    w3 = rng.integers(1, 256, (K + 128, 2 * C, 1, 1), dtype=np.uint8)
    p3 = hipq.Conv2d(xs.shape, w3, None, 0, st, 1, *qs)
    assert not hipq.add2_fusable(pm, p3, False, 0.1, 0)
    with pytest.raises(hipq.HipqError, match="do not run as one kernel"):
        hipq.run_add2(pm, xd, p3, xsd, False, 0.1, 0, pm.empty_output())


def time_layers():
    """Every convolution of the 28x28-and-smaller stages of ResNet-50 at batch 64: the built-in kernel against special(3)."""
    rng = np.random.default_rng(9)
    layers = [  # C, H, K, k, stride, with add
        (256, 56, 128, 1, 1, False), (128, 56, 128, 3, 2, False), (256, 56, 512, 1, 2, False), (512, 28, 128, 1, 1, False),
        (512, 28, 256, 1, 1, False), (256, 28, 256, 3, 2, False), (512, 28, 1024, 1, 2, False), (256, 14, 1024, 1, 1, True),
        (1024, 14, 256, 1, 1, False), (256, 14, 256, 3, 1, False), (1024, 14, 512, 1, 1, False), (512, 14, 512, 3, 2, False),
        (1024, 14, 2048, 1, 2, False), (512, 7, 2048, 1, 1, True), (2048, 7, 512, 1, 1, False), (512, 7, 512, 3, 1, False),
    ]
    for C, HW, K, k, st, add in layers:
        N = 64
        x = torch.randint(0, 256, (N, HW, HW, C), dtype=torch.uint8, device="cuda")
        w = rng.integers(1, 256, (K, C, k, k), dtype=np.uint8)
        sigma = 74.0 * 74.0 * math.sqrt(C * k * k)
        b = rng.integers(-int(sigma), int(sigma) + 1, K).astype(np.int32)
        q = (0.03, 120, float(np.float32(40.0 / sigma)), 128, 0.03, 0 if not add else 128)
        out = {}
        for mode in (1, 3):
            plan = hipq.Conv2d((N, C, HW, HW), w, b, k // 2, st, 1, *q).special(mode)
            y = plan.empty_output()
            res = torch.randint(0, 256, y.shape, dtype=torch.uint8, device="cuda")
            fn = (lambda: plan.run_add(x, res, False, 0.04, 100, 0.06, 0, y)) if add else (lambda: plan(x, y))
            fn()
            torch.cuda.synchronize()
            g = torch.cuda.CUDAGraph()
            with torch.cuda.graph(g):
                for _ in range(10):
                    fn()
            for _ in range(3):
                g.replay()
            torch.cuda.synchronize()
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(20):
                g.replay()
            e1.record()
            torch.cuda.synchronize()
            out[mode] = (e0.elapsed_time(e1) / 200 * 1e3, plan.kernel_add if add else plan.kernel)
        print("layer C=%4d %2dx%2d K=%4d k=%d s=%d add=%d: %-34s %6.1f us | %-22s %6.1f us" % (
            C, HW, HW, K, k, st, add, out[1][1], out[1][0], out[3][1], out[3][0]), flush=True)


def time_block(N, CW, HW, reps=50):
    rng = np.random.default_rng(5)
    x, xq, layers, sq = make_block(rng, N, CW, HW, HW)
    plans = plans_of(x, layers)
    xd = hipq.to_device_nhwc(x)
    y = torch.zeros_like(xd)
    t1, t2 = plans[0].empty_output(), plans[1].empty_output()

    def fused():
        hipq.bottleneck_run(*plans, xd, False, sq[0], sq[1], y)

    def separate():
        plans[0](xd, t1)
        plans[1](t1, t2)
        plans[2].run_add(t2, xd, False, xq[0], xq[1], sq[0], sq[1], y)

    out = {}
    for name, fn in (("fused", fused), ("separate", separate)):
        fn()
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            for _ in range(10):
                fn()
        for _ in range(3):
            g.replay()
        torch.cuda.synchronize()
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record()
        for _ in range(reps):
            g.replay()
        e1.record()
        torch.cuda.synchronize()
        out[name] = e0.elapsed_time(e1) / reps / 10 * 1e3
    print("block N=%d CW=%d %dx%d: fused %.1f us, separate (%s) %.1f us" % (
        N, CW, HW, HW, out["fused"], " + ".join([plans[0].kernel, plans[1].kernel, plans[2].kernel_add]), out["separate"]), flush=True)


if __name__ == "__main__":
    for N, CW, HW in ((64, 1024, 14), (64, 512, 28), (64, 256, 56)):
        time_block(N, CW, HW)
    for N, CW, HW in ((64, 1024, 14), (64, 512, 28), (64, 256, 56)):
        time_tail(N, CW, HW)
    time_layers()


INVRES_CASES = [  # N, CIN, HIDDEN, COUT, H, W, stride
    (1, 16, 96, 24, 20, 33, 2), (1, 24, 144, 24, 14, 9, 1), (2, 32, 192, 64, 7, 7, 2), (3, 64, 384, 64, 5, 6, 1), (1, 160, 960, 160, 7, 7, 1),
    (2, 96, 576, 96, 14, 14, 1), (2, 96, 80, 160, 3, 50, 2), (1, 48, 40, 72, 1, 1, 1), (1, 30, 33, 10, 2, 1, 2), (4, 128, 256, 40, 17, 19, 1),
    (40, 24, 144, 24, 33, 31, 1), (40, 24, 144, 32, 33, 31, 1), (64, 16, 96, 24, 56, 56, 2), (64, 40, 100, 60, 29, 28, 2),
    (64, 64, 384, 96, 14, 14, 1), (30, 32, 64, 32, 31, 34, 1), (12, 96, 200, 130, 40, 40, 1),
]


@pytest.mark.parametrize("case", INVRES_CASES, ids=lambda c: "x".join(map(str, c)))
def test_inverted_residual_block(case):
    """conv_invres_kernel against the oracle's convolutions and add: patches of 2x4, 4x8 and 8x8 outputs and one wave per patch, all
    partly outside the image, images of one pixel, slices and tiles that are partly empty, both strides, ReLUs in the plan and at
    the launch, with and without the add in both operand orders."""
    N, CI, CH, CO, H, W, st = case
    rng = np.random.default_rng(sum(case))
    x = rng.integers(0, 256, (N, CI, H, W), dtype=np.uint8)
    late = bool(sum(case) & 1)  # the ReLUs as flags of the launch instead of the plans
    t, a, z, plans, cur = x, 0.03, int(rng.integers(0, 256)), [], None
    qx = (a, z)
    for k, (C, K, R, s, group) in enumerate(((CI, CH, 1, 1, 1), (CH, CH, 3, st, CH), (CH, CO, 1, 1, 1))):
        w = rng.integers(1, 256, (K, C // group, R, R), dtype=np.uint8)
        sigma = 74.0 * 74.0 * math.sqrt(w[0].size) * (0.7 if k else 1.0)
        b = rng.integers(-int(sigma), int(sigma) + 1, K).astype(np.int32)
        oa = float(np.float32(0.03 * rng.uniform(0.75, 1.35)))
        q = (a, z, float(np.float32(oa * 45.0 / (a * sigma))), 128, oa, int(rng.integers(0, 60)) if k < 2 else int(rng.integers(90, 160)))
        plans.append(hipq.Conv2d(t.shape, w, b, R // 2, s, group, *q, relu=k < 2 and not late))
        t = orc.conv2d_u8(t, w, b, R // 2, s, group, *q)
        if k < 2:
            t = np.maximum(t, q[5]).astype(np.uint8)
        a, z = q[4], q[5]
    plans[2].special(2)
    xd = hipq.to_device_nhwc(x)
    relus = 3 if late else 0
    assert hipq.inverted_residual_fusable(*plans), case
    print("inverted residual", case, late, flush=True)
    got = hipq.from_device_nhwc(hipq.inverted_residual_run(*plans, xd, torch.full_like(plans[2].empty_output(), 99), relus=relus), CO)
    assert len(np.unique(t)) > min(8, t.size // 2)
    assert np.array_equal(got, t), (case, int((got != t).sum()), np.argwhere(got != t)[:8].tolist())
    if CI != CO or st != 1:
        return
    sa, sz = float(np.float32(math.hypot(a, qx[0]) * 1.1)), int(rng.integers(0, 60))
    for first in (False, True):
        want = orc.add_u8(x, t, *qx, a, z, sa, sz) if first else orc.add_u8(t, x, a, z, *qx, sa, sz)
        y = hipq.inverted_residual_run(*plans, xd, torch.full_like(plans[2].empty_output(), 99), (first, sa, sz), relus)
        got = hipq.from_device_nhwc(y, CO)
        assert np.array_equal(got, want), (case, "add", first, int((got != want).sum()))


INVRES_CHANNELS = [(1, 1, 16, 24), (1, 2, 24, 40), (2, 2, 40, 60), (2, 3, 64, 72), (3, 3, 96, 96), (3, 5, 80, 130), (5, 5, 160, 160)]
# every kernel that is built: k-steps, channel tiles, their channel counts; stride; shape
INVRES_SHAPES = [(nk, ct, ci, co, st, sh) for nk, ct, ci, co in INVRES_CHANNELS for st in (1, 2) for sh in range(4)
                 if not (sh == 3 and (nk > 2 or ct > 2)) and not (sh == 2 and (st == 2 or ct > 3))]


@pytest.mark.parametrize("case", INVRES_SHAPES, ids=lambda c: "s%d_%s_k%d_n%d" % (c[4], ("2x4", "4x8", "8x8", "own")[c[5]], c[0], c[1]))
def test_inverted_residual_every_kernel(case):
    """Each of the 39 instantiations of conv_invres_kernel by name, on an image whose patches overhang on two sides (13 x 11) and one
    smaller than a patch, three slices of which the last is partial, against the oracle's convolutions; where input and output
    have equal channels, the add as well."""
    nk, ct, ci, co, st, sh = case
    assert len(INVRES_SHAPES) == 39
    ch = 80
    for N, H, W in ((3, 13, 11), (1, 3, 2)):
        rng = np.random.default_rng(ci + co + st + H)
        x = rng.integers(0, 256, (N, ci, H, W), dtype=np.uint8)
        t, a, z, plans = x, 0.03, 77, []
        for k, (C, K, R, s, group) in enumerate(((ci, ch, 1, 1, 1), (ch, ch, 3, st, ch), (ch, co, 1, 1, 1))):
            w = rng.integers(1, 256, (K, C // group, R, R), dtype=np.uint8)
            sigma = 74.0 * 74.0 * math.sqrt(w[0].size) * (0.7 if k else 1.0)
            b = rng.integers(-int(sigma), int(sigma) + 1, K).astype(np.int32)
            oa = float(np.float32(0.03 * rng.uniform(0.75, 1.35)))
            q = (a, z, float(np.float32(oa * 45.0 / (a * sigma))), 128, oa, 30 if k < 2 else 120)
            plans.append(hipq.Conv2d(t.shape, w, b, R // 2, s, group, *q, relu=k < 2))
            t = orc.conv2d_u8(t, w, b, R // 2, s, group, *q)
            if k < 2:
                t = np.maximum(t, q[5]).astype(np.uint8)
            a, z = q[4], q[5]
        plans[2].special(2)
        hipq.inverted_residual_select(plans[2], sh)
        name = hipq.inverted_residual_kernel(*plans)
        assert name == "conv_invres_s%d_%s_k%d_n%d" % (st, ("2x4", "4x8", "8x8", "own")[sh], nk, ct), name
        print(name, (N, H, W), flush=True)
        xd = hipq.to_device_nhwc(x)
        got = hipq.from_device_nhwc(hipq.inverted_residual_run(*plans, xd, torch.full_like(plans[2].empty_output(), 99)), co)
        assert np.array_equal(got, t), (name, int((got != t).sum()), np.argwhere(got != t)[:8].tolist())
        if ci == co and st == 1:
            want = orc.add_u8(t, x, a, z, 0.03, 77, 0.05, 20)
            y = hipq.inverted_residual_run(*plans, xd, torch.full_like(plans[2].empty_output(), 99), (False, 0.05, 20))
            assert np.array_equal(hipq.from_device_nhwc(y, co), want), (name, "add")


@pytest.mark.parametrize("hw", [(13, 11), (4, 8), (3, 2)], ids=lambda v: "%dx%d" % v)
@pytest.mark.parametrize("case", [(1, 1, 24, 24), (1, 2, 24, 40), (2, 2, 40, 60)], ids=lambda c: "k%d_n%d" % c[:2])
def test_inverted_residual_half_patch_per_wave(case, hw):
    """A patch of 4x8 outputs per wave: overhanging on two sides, exactly one, smaller than one; 5 images, so that the last
    work-group has idle waves; three slices, the last partial; with the add where the channels allow it."""
    nk, ct, ci, co = case
    rng = np.random.default_rng(ci + co + hw[0])
    x = rng.integers(0, 256, (5, ci, *hw), dtype=np.uint8)
    t, a, z, plans = x, 0.03, 77, []
    for k, (C, K, R, group) in enumerate(((ci, 80, 1, 1), (80, 80, 3, 80), (80, co, 1, 1))):
        w = rng.integers(1, 256, (K, C // group, R, R), dtype=np.uint8)
        sigma = 74.0 * 74.0 * math.sqrt(w[0].size) * (0.7 if k else 1.0)
        b = rng.integers(-int(sigma), int(sigma) + 1, K).astype(np.int32)
        oa = float(np.float32(0.03 * rng.uniform(0.75, 1.35)))
        q = (a, z, float(np.float32(oa * 45.0 / (a * sigma))), 128, oa, 30 if k < 2 else 120)
        plans.append(hipq.Conv2d(t.shape, w, b, R // 2, 1, group, *q, relu=k < 2))
        t = orc.conv2d_u8(t, w, b, R // 2, 1, group, *q)
        if k < 2:
            t = np.maximum(t, q[5]).astype(np.uint8)
        a, z = q[4], q[5]
    plans[2].special(2)
    hipq.inverted_residual_select(plans[2], 4)
    name = hipq.inverted_residual_kernel(*plans)
    assert name == "conv_invres_s1_own4x8_k%d_n%d" % (nk, ct), name
    print(name, hw, flush=True)
    xd = hipq.to_device_nhwc(x)
    got = hipq.from_device_nhwc(hipq.inverted_residual_run(*plans, xd, torch.full_like(plans[2].empty_output(), 99)), co)
    assert np.array_equal(got, t), (name, int((got != t).sum()))
    if ci == co:
        want = orc.add_u8(t, x, a, z, 0.03, 77, 0.05, 20)
        y = hipq.inverted_residual_run(*plans, xd, torch.full_like(plans[2].empty_output(), 99), (False, 0.05, 20))
        assert np.array_equal(hipq.from_device_nhwc(y, co), want), (name, "add")


# channels, hidden channels, image, shape: 7x7 patches that overhang on both sides, fit exactly, are larger than the image; the most hidden
# channels that a shape takes, most of them without room in LDS for the last layer's weights; more output tiles than waves
INVRES_SPLITS = [(ci, 80, co, hw, 5) for ci, co in ((24, 24), (24, 40), (40, 60), (64, 72), (96, 96)) for hw in ((13, 11), (7, 14), (3, 2))]
INVRES_SPLITS += [(16, 1152, 16, (9, 5), 2), (96, 1152, 96, (5, 4), 5), (96, 32, 96, (9, 5), 2), (160, 2048, 160, (3, 9), 1), (160, 2000, 24, (3, 5), 0)]


@pytest.mark.parametrize("case", INVRES_SPLITS, ids=lambda c: "%d_%d_%d_%s_%d" % (c[:3] + ("%dx%d" % c[3],) + c[4:]))
def test_inverted_residual_splits_of_the_hidden_channels(case):
    ci, ch, co, hw, sh = case
    rng = np.random.default_rng(ci + ch + co + hw[0])
    x = rng.integers(0, 256, (2, ci, *hw), dtype=np.uint8)
    t, a, z, plans = x, 0.03, 77, []
    for k, (C, K, R, group) in enumerate(((ci, ch, 1, 1), (ch, ch, 3, ch), (ch, co, 1, 1))):
        w = rng.integers(1, 256, (K, C // group, R, R), dtype=np.uint8)
        sigma = 74.0 * 74.0 * math.sqrt(w[0].size) * (0.7 if k else 1.0)
        b = rng.integers(-int(sigma), int(sigma) + 1, K).astype(np.int32)
        oa = float(np.float32(0.03 * rng.uniform(0.75, 1.35)))
        q = (a, z, float(np.float32(oa * 45.0 / (a * sigma))), 128, oa, 30 if k < 2 else 120)
        plans.append(hipq.Conv2d(t.shape, w, b, R // 2, 1, group, *q, relu=k < 2))
        t = orc.conv2d_u8(t, w, b, R // 2, 1, group, *q)
        if k < 2:
            t = np.maximum(t, q[5]).astype(np.uint8)
        a, z = q[4], q[5]
    plans[2].special(2)
    hipq.inverted_residual_select(plans[2], sh)
    name = hipq.inverted_residual_kernel(*plans)
    assert name.startswith("conv_invres_s1_%s_k" % ("2x4", "4x8", "8x8", "own", "own4x8", "7x7")[sh]), name
    print(name, case, flush=True)
    xd = hipq.to_device_nhwc(x)
    got = hipq.from_device_nhwc(hipq.inverted_residual_run(*plans, xd, torch.full_like(plans[2].empty_output(), 99)), co)
    assert np.array_equal(got, t), (name, int((got != t).sum()))
    if ci == co:
        want = orc.add_u8(t, x, a, z, 0.03, 77, 0.05, 20)
        y = hipq.inverted_residual_run(*plans, xd, torch.full_like(plans[2].empty_output(), 99), (False, 0.05, 20))
        assert np.array_equal(hipq.from_device_nhwc(y, co), want), (name, "add")


@pytest.mark.parametrize("n, pays", [(1, False), (16, False), (20, True), (64, True)])
def test_whole_blocks_pay_from_some_pixels_on(n, pays):
    """The executor leaves the three layers apart below 20 images of 14x14, where a block's weights take one work-group longer than
    three launches; the kernel itself stays applicable, and asked for (special 2) it pays at any size."""
    w = np.full((256, 1024, 1, 1), 129, np.uint8)
    p = hipq.Conv2d((n, 1024, 14, 14), w, np.zeros(256, np.int32), 0, 1, 1, 0.05, 9, 0.001, 128, 0.06, 0)
    assert hipq.bottleneck_pays(p) == pays
    assert hipq.bottleneck_pays(p.special(2))


RAGGED_TAILS = [  # N, CW, H, W: the last patch of a row or column overlaps its neighbour by all but one, by one, or not at all
    (2, 256, 9, 15), (1, 256, 25, 25), (1, 512, 13, 29), (3, 512, 5, 15), (2, 512, 25, 25), (1, 1024, 9, 8), (1, 256, 7, 8), (1, 512, 15, 8),
]


@pytest.mark.parametrize("case", RAGGED_TAILS, ids=lambda c: "x".join(map(str, c)))
def test_bottleneck_tail_on_ragged_images(case):
    """Images that no patch divides: the pixels that two patches share are computed by both and lie where one of them would put them."""
    test_bottleneck_tail(case)


@pytest.mark.parametrize("case", [(2, 512, 13, 13, 25, 26), (1, 512, 9, 17, 18, 33), (1, 512, 25, 25, 50, 49)], ids=lambda c: "x".join(map(str, c)))
def test_strided_bottleneck_tail_on_ragged_images(case):
    test_bottleneck_tail_with_a_strided_3x3_layer(case)


@pytest.mark.parametrize("case", [(2, 1024, 13, 13), (1, 1024, 8, 8), (1, 1024, 7, 9), (1, 1024, 16, 10)], ids=lambda c: "x".join(map(str, c)))
def test_bottleneck_block_on_ragged_images(case):
    test_bottleneck_block(case)


def test_overlapping_patches_do_not_overwrite_their_residual():
    """A patch reads its residual before it writes the sum, its neighbour's shared pixels perhaps after: y must be another tensor there
    (and may be the residual where patches are disjoint)."""
    rng = np.random.default_rng(11)
    for CW, H, W, ok in ((256, 16, 16, True), (256, 16, 17, False), (512, 14, 14, True), (512, 21, 21, True), (256, 14, 21, True),
                         (512, 7, 14, True), (1024, 14, 14, True), (256, 42, 42, True), (512, 13, 13, False)):
        t1, res, layers, rq, sq, nx = make_tail(rng, 1, CW, H, W, False)
        plans = plans_of(t1, layers)
        xd, rd, want = hipq.to_device_nhwc(t1), hipq.to_device_nhwc(res), torch.zeros_like(hipq.to_device_nhwc(res))
        hipq.bottleneck_tail_run(plans[0], plans[1], xd, rd, False, rq[0], rq[1], sq[0], sq[1], want)
        t = orc.conv2d_u8(t1, layers[0]["w"], layers[0]["b"], 1, 1, 1, *layers[0]["q"])
        c = orc.conv2d_u8(t, layers[1]["w"], layers[1]["b"], 0, 1, 1, *layers[1]["q"])
        assert np.array_equal(hipq.from_device_nhwc(want, CW), orc.add_u8(c, res, *layers[1]["q"][4:6], *rq, *sq)), (CW, H, W)
        if ok:
            hipq.bottleneck_tail_run(plans[0], plans[1], xd, rd, False, rq[0], rq[1], sq[0], sq[1], rd)
            torch.cuda.synchronize()
            assert torch.equal(rd, want)
        else:
            with pytest.raises(hipq.HipqError, match="cannot overwrite the residual"):
                hipq.bottleneck_tail_run(plans[0], plans[1], xd, rd, False, rq[0], rq[1], sq[0], sq[1], rd)


@pytest.mark.parametrize("n, hw, block, tail", [(11, 13, False, True), (64, 13, True, True), (64, 10, False, True), (1, 20, False, False), (2, 20, False, True),
                                                (1, 14, True, True), (1, 21, True, True)])
def test_rules_on_ragged_images(n, hw, block, tail):
    """Where the one-launch forms are chosen on images that their patches do not divide: whole blocks by the two fitted costs, tails of 128
    channels with a wider next layer from 600 pixels on."""
    rng = np.random.default_rng(n)
    x, xq, layers, sq = make_block(rng, 1, 1024, 7, 7)
    shapes = ((n, 1024, hw, hw), (n, 256, hw, hw), (n, 256, hw, hw))
    plans = [hipq.Conv2d(s, L["w"], L["b"], L["pad"], 1, 1, *L["q"]) for s, L in zip(shapes, layers)]
    assert hipq.bottleneck_fusable(*plans, False, sq[0], sq[1]) == block
    t1, res, tl, rq, sq2, nx = make_tail(rng, 1, 512, 7, 7, False, True)
    p2 = hipq.Conv2d((n, 128, hw, hw), tl[0]["w"], tl[0]["b"], 1, 1, 1, *tl[0]["q"])
    p3 = hipq.Conv2d((n, 128, hw, hw), tl[1]["w"], tl[1]["b"], 0, 1, 1, *tl[1]["q"])
    pn = hipq.Conv2d((n, 512, hw, hw), nx["w"], nx["b"], 0, 1, 1, *nx["q"])
    assert hipq.bottleneck_tail_fusable(p2, p3, False, rq[0], rq[1], sq2[0], sq2[1], pn) == tail
