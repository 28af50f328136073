"""What the speed of this package is measured on: passes through its public entry points, as programs use them.

Six kinds of work, each over the range of sizes that its users have:

  layer   one convolution or fully-connected layer (hipq.Conv2d) on tensors that are on the GPU
  ends    the float ends of a network: images to bytes (quantize), a score map back to floats (dequantize)
  joins   the operators between the convolutions of a branching network: add, n-ary eltwise, relu, pooling, concat, softmax
  net     one forward pass of a network whose tensors are on the GPU (runner.HipqExecutor, a captured pass replayed)
  engine  one forward pass of an engine file on the `hip` workspace from host arrays to host arrays (art_compat.Parade.run,
          the usage of NART's own Python package)

Everything the package computes is integer arithmetic or a single rounded float operation: every output is exact.
"""
import numpy as np
import torch

from nart_amd import art_compat, cases, engine, hipq
from nart_amd.runner import HipqExecutor

NETS = {"resnet18": cases.resnet18, "resnet50": cases.resnet50, "mobilenetv2": cases.mobilenet_v2}
CLASSES = 1000


def listed():
    return [
        # the single convolution, where a call's own cost is everything
        dict(name="layer_conv3x3_n1", kind="layer", n=1, c=64, h=56, w=56, k=64, r=3, stride=1, depthwise=False, dtype="u8",
             wzp=128, per_channel=False),
        # a layer of a detection backbone on an odd image, int8 symmetric with a weight scale per channel
        dict(name="layer_conv3x3_i8_ragged", kind="layer", n=5, c=96, h=75, w=67, k=200, r=3, stride=1, depthwise=False, dtype="i8",
             wzp=0, per_channel=True),
        # the fully-connected layer at batch 128
        dict(name="layer_fc_m128", kind="layer", n=128, c=4096, h=1, w=1, k=4096, r=1, stride=1, depthwise=False, dtype="u8",
             wzp=128, per_channel=False),
        # a batch of images in, a 21-class score map at a quarter of the resolution out (segmentation)
        dict(name="ends_n64", kind="ends", n=64, c=3, h=224, w=224, classes=21, down=4, dtype="u8"),
        # the joins of an inception-like block at 35 x 35
        dict(name="joins_n8", kind="joins", n=8, c=192, c2=100, h=35, w=35, classes=81),
        # BASELINE configuration 2 at batch 1: latency
        dict(name="net_resnet18_n1", kind="net", net="resnet18", n=1, hw=224),
        # BASELINE configurations 4 and 3: throughput at batch 64
        dict(name="net_resnet50_n64", kind="net", net="resnet50", n=64, hw=224),
        dict(name="net_mobilenetv2_n64", kind="net", net="mobilenetv2", n=64, hw=224),
        # a batch of what has just come in, at another resolution (100, 50, 25 and 13 pixels inside)
        dict(name="net_resnet50_n11_hw200", kind="net", net="resnet50", n=11, hw=200),
        # one image from host memory to scores in host memory
        dict(name="engine_resnet18_n1", kind="engine", net="resnet18", n=1, hw=224),
        # the smallest network's file at a small batch and a smaller resolution
        dict(name="engine_mobilenetv2_n6_hw160", kind="engine", net="mobilenetv2", n=6, hw=160),
        # BASELINE configuration 4 from host memory: the largest
        dict(name="engine_resnet50_n64", kind="engine", net="resnet50", n=64, hw=224),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return min(hi, max(lo, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    kind = rng.choice(("layer", "layer", "ends", "joins", "net", "net", "engine", "engine"))
    if kind == "layer":
        dtype = rng.choice(("u8", "u8", "u8", "i8"))
        quant = dict(dtype=dtype, wzp=0 if dtype == "i8" else rng.choice((128, 128, 128, rng.randrange(100, 156))),
                     per_channel=rng.random() < 0.25)
        if rng.random() < 0.3:  # fully connected
            c = _log(rng, 256, 8192)
            return dict(kind="layer", n=_log(rng, 1, 512), c=c, h=1, w=1, k=_log(rng, 10, min(8192, (16 << 20) // c)), r=1, stride=1,
                        depthwise=False, **quant)
        h = _log(rng, 5, 150)
        w = max(5, int(h * rng.uniform(0.7, 1.4)))
        n = _log(rng, 1, 64)
        most = max(16, min(1024, (24 << 20) // (n * h * w)))  # channels: at most 24 MB a tensor
        c = _log(rng, 16, most)
        depthwise = rng.random() < 0.2
        return dict(kind="layer", n=n, c=c, h=h, w=w, k=c if depthwise else _log(rng, 16, most), r=3 if depthwise else rng.choice((1, 1, 3, 3, 5)),
                    stride=rng.choice((1, 1, 2)), depthwise=depthwise, **quant)
    if kind == "ends":
        n, hw = _log(rng, 1, 64), _log(rng, 96, 300)
        return dict(kind="ends", n=n, c=rng.choice((1, 3, 3, 4, 16)) if n <= 16 else 3, h=hw, w=max(64, int(hw * rng.uniform(0.8, 1.25))),
                    classes=_log(rng, 2, 128 if n <= 16 else 32), down=rng.choice((4, 8)), dtype=rng.choice(("u8", "u8", "i8")))
    if kind == "joins":
        h = _log(rng, 7, 112)
        n = _log(rng, 1, 64)
        most = max(24, min(1024, (16 << 20) // (n * h * h)))
        return dict(kind="joins", n=n, c=_log(rng, 16, most), c2=_log(rng, 16, most), h=h, w=max(7, int(h * rng.uniform(0.7, 1.3))),
                    classes=_log(rng, 2, most))
    net = rng.choice(sorted(NETS))
    hw = 32 * rng.randrange(2, 10) if rng.random() < 0.5 else rng.randrange(64, 300)
    most = min(64, 64 * 224 * 224 // (hw * hw))
    return dict(kind=kind, net=net, n=_log(rng, 1, most), hw=hw)


# ---- inputs ---------------------------------------------------------------------------------------------------------
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _bytes(gen, *shape):
    return torch.randint(0, 256, shape, dtype=torch.uint8, device="cuda", generator=gen)


def _layer(case, seed, gen):
    n, c, h, w, k, r = (case[f] for f in ("n", "c", "h", "w", "k", "r"))
    rng = np.random.default_rng(seed)
    group = c if case["depthwise"] else 1
    i8 = case["dtype"] == "i8"
    wt = rng.integers(-127, 128, (k, c // group, r, r), dtype=np.int8) if i8 else rng.integers(0, 256, (k, c // group, r, r), dtype=np.uint8)
    spread = 74.0 * 74.0 * np.sqrt(c // group * r * r)  # of an accumulator over bytes uniform around their zero points
    bias = rng.integers(-int(spread), int(spread) + 1, k).astype(np.int32)
    ialpha, walpha = 0.02, 0.005
    oalpha = float(np.float32(ialpha * walpha * spread / 40.0))
    if case["per_channel"]:
        walpha = (walpha * rng.uniform(0.5, 1.5, k)).astype(np.float32)
    plan = hipq.Conv2d((n, c, h, w), wt, bias, r // 2, case["stride"], group, ialpha, 0 if i8 else 128, walpha, case["wzp"], oalpha,
                       0 if i8 else 120, obits=7 if i8 else 8, dtype=hipq.DTYPE_I8 if i8 else hipq.DTYPE_U8)
    y = plan.empty_output()
    return dict(plan=plan, x=_bytes(gen, n, h, w, hipq.channel_stride(c)), y=y, out=y[..., :k])


def _ends(case, seed, gen):
    n, c, h, w, k = (case[f] for f in ("n", "c", "h", "w", "classes"))
    hs, ws = h // case["down"], w // case["down"]
    return dict(i8=case["dtype"] == "i8", x=torch.randn((n, c, h, w), device="cuda", generator=gen) * 1.2,
                q=torch.zeros((n, h, w, hipq.channel_stride(c)), dtype=torch.uint8, device="cuda"), c=c,
                s=_bytes(gen, n, hs, ws, hipq.channel_stride(k)), f=torch.empty((n, k, hs, ws), device="cuda"))


def _joins(case, seed, gen):
    n, c, c2, h, w, k = (case[f] for f in ("n", "c", "c2", "h", "w", "classes"))
    cs, cs2, ks = hipq.channel_stride(c), hipq.channel_stride(c2), hipq.channel_stride(k)
    oh, ow = hipq.conv_out_dim(h, 1, 3, 2), hipq.conv_out_dim(w, 1, 3, 2)

    def empty(*shape):
        return torch.zeros(shape, dtype=torch.uint8, device="cuda")
    return dict(a=_bytes(gen, n, h, w, cs), b=_bytes(gen, n, h, w, cs), d=_bytes(gen, n, h, w, cs), e=_bytes(gen, n, h, w, cs2),
                logits=_bytes(gen, n, h, w, ks), c=c, c2=c2, k=k, total=empty(n, h, w, cs), top=empty(n, h, w, cs), act=empty(n, h, w, cs),
                cat=empty(n, h, w, hipq.channel_stride(c + c2)), small=empty(n, oh, ow, cs), mean=empty(n, h, w, cs), vec=empty(n, 1, 1, cs),
                prob=empty(n, h, w, ks))


def _input(case, net, gen):
    shape = net.input.shape
    if net.input.dtype == "f32":
        return torch.randn(shape, device="cuda", generator=gen).mul_(1.2).cpu().numpy()
    return _bytes(gen, *shape).cpu().numpy()


def _net(case, seed, gen):
    net = NETS[case["net"]](N=case["n"], hw=case["hw"], seed=seed)
    ex = HipqExecutor(net, fuse_add=True)
    ex.set_input(_input(case, net, gen))
    ex.capture()
    y = ex.buf[net.output.name]
    return dict(ex=ex, out=y if net.output.dtype == "f32" else y[..., :CLASSES])


def _engine(case, seed, gen):
    net = NETS[case["net"]](N=case["n"], hw=case["hw"], seed=seed)
    parade = art_compat.Parade(engine.write_engine(net), art_compat.create_context_for_target("hip"))
    inputs, outputs = art_compat.get_empty_io(parade)
    inputs[net.input.name][:] = _input(case, net, gen)
    return dict(parade=parade, inputs=inputs, outputs=outputs, out=outputs[net.output.name])


def prepare(case, seed):
    make = {"layer": _layer, "ends": _ends, "joins": _joins, "net": _net, "engine": _engine}[case["kind"]]
    return dict(make(case, seed, _generator(seed)), kind=case["kind"])


# ---- one pass -------------------------------------------------------------------------------------------------------
def _run_ends(s):
    if s["i8"]:
        hipq.quantize_i8(s["x"], s["q"], 0.03)
        hipq.dequantize_i8(s["s"], s["f"], 0.11)
    else:
        hipq.quantize_u8(s["x"], s["q"], 0.0186, 114)
        hipq.dequantize_u8(s["s"], s["f"], 0.11, 97)
    return s["q"][..., :s["c"]], s["f"]


def _run_joins(s):
    c, c2, k = s["c"], s["c2"], s["k"]
    hipq.add_u8(s["a"], s["b"], s["total"], 0.02, 121, 0.03, 130, 0.038, 119)
    hipq.eltwise_u8([s["a"], s["b"], s["d"]], s["top"], [0.02, 0.03, 0.025], [121, 130, 128], 0.03, 125, operation=2)
    hipq.relu_u8(s["total"], s["act"], 0.038, 119, 0.02, 0)
    hipq.concat_u8([s["act"], s["e"]], [c, c2], s["cat"], [0.02, 0.024], [0, 3], 0.022, 2)
    hipq.pool_u8(s["top"], s["small"], c, 3, 1, 2, 0, 0.03, 125, 0.03, 125)
    hipq.pool_u8(s["act"], s["mean"], c, 3, 1, 1, 1, 0.02, 0, 0.015, 4)
    hipq.pool_u8(s["act"], s["vec"], c, s["act"].shape[1:3], 0, 1, 1, 0.02, 0, 0.01, 0)
    hipq.softmax_u8(s["logits"], s["prob"], k, 0.06, 128, 1.0 / 256, 0)
    return {"total": s["total"][..., :c], "top": s["top"][..., :c], "act": s["act"][..., :c], "cat": s["cat"][..., :c + c2],
            "small": s["small"][..., :c], "mean": s["mean"][..., :c], "vec": s["vec"][..., :c], "prob": s["prob"][..., :k]}


def run(state):
    kind = state["kind"]
    if kind == "layer":
        state["plan"](state["x"], state["y"])
        return state["out"]
    if kind == "net":
        state["ex"].replay()
        return state["out"]
    if kind == "engine":
        state["parade"].run(state["inputs"], state["outputs"])
        return state["out"]
    return _run_ends(state) if kind == "ends" else _run_joins(state)


# ---- what a pass cannot do without ------------------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    if kind == "layer":
        n, c, h, w, k, r = (case[f] for f in ("n", "c", "h", "w", "k", "r"))
        pixels = n * hipq.conv_out_dim(h, r // 2, r, case["stride"]) * hipq.conv_out_dim(w, r // 2, r, case["stride"])
        per_output = r * r * (1 if case["depthwise"] else c)
        return {"bytes": n * c * h * w + pixels * k + k * per_output + 4 * k, "flops": 2 * pixels * k * per_output}
    if kind == "ends":
        n, c, h, w = (case[f] for f in ("n", "c", "h", "w"))
        return {"bytes": 5 * n * c * h * w + 5 * n * case["classes"] * (h // case["down"]) * (w // case["down"]), "flops": 0}
    if kind == "joins":
        n, c, c2, h, w, k = (case[f] for f in ("n", "c", "c2", "h", "w", "classes"))
        small = hipq.conv_out_dim(h, 1, 3, 2) * hipq.conv_out_dim(w, 1, 3, 2)
        # in: three tensors of c channels, one of c2, the logits; out: the eight results
        return {"bytes": n * (h * w * (3 * c + c2 + k) + h * w * (4 * c + c + c2 + k) + small * c + c), "flops": 0}
    net = NETS[case["net"]](N=case["n"], hw=case["hw"])
    size = {"f32": 4, "u8": 1}
    ends = sum(int(np.prod(t.shape)) * size[t.dtype] for t in (net.input, net.output))
    return {"bytes": ends + sum(v.nbytes for v in net.weights.values()), "flops": net.conv_ops()}


def tolerance(case):
    return "exact"
