"""The reference's Python usage (python/nart/art/__init__.py:20-27), run unchanged against nart_amd.art_compat: an
engine file and its JSON configuration on disk, create_context_from_json / load_parade / get_empty_io / Parade.run,
the output compared with the CPU oracle bit for bit."""
import json
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

from nart_amd import art_compat as art  # noqa: E402  (the one line a NART user changes)
from nart_amd import cases, engine  # noqa: E402
from oracle import casecpu, orc  # noqa: E402  (checkers only)


def _write(tmp_path, case):
    fp = os.path.join(tmp_path, case.name + ".bin")
    with open(fp, "wb") as f:
        f.write(engine.write_engine(case))
    with open(fp + ".json", "w") as f:
        json.dump({"workspaces": {"hip": {}}, "input_workspace": "hip"}, f)
    return fp


def test_readme_usage_on_resnet18(tmp_path):
    case = cases.resnet18(N=2, hw=96)
    fp = _write(str(tmp_path), case)
    rng = np.random.default_rng(5)
    x = rng.integers(0, 256, case.input.shape, dtype=np.uint8)
    want = casecpu.run_case(case, x)[case.output.name].reshape(2, -1)  # the runtime infers [N, K] for an inner product (art/src/op.c)

    ctx = art.create_context_from_json(fp + ".json")
    assert ctx.loaded_workspaces == ["hip"]
    parade = art.load_parade(fp, ctx)
    inputs, outputs = art.get_empty_io(parade)
    assert list(inputs) == [case.input.name] and list(outputs) == [case.output.name]
    inputs[case.input.name][:] = x
    assert parade.run(inputs, outputs) is True
    got = outputs[case.output.name]
    assert got.dtype == want.dtype and got.shape == want.shape and np.array_equal(got, want)

    # the rest of the surface (module.cpp:302-400)
    assert parade.input_shapes() == {case.input.name: list(case.input.shape)}
    assert parade.output_shapes() == {case.output.name: list(want.shape)}
    assert parade.input_dtypes() == {case.input.name: "uint8"} and parade.output_dtypes() == {case.output.name: str(want.dtype)}
    assert parade.get_tensor_dtype(case.input.name) == "uint8" and parade.get_tensor_dtype("no such tensor") is None
    assert parade.get_tensor_shape(case.output.name) == list(want.shape) and parade.get_tensor_shape("nope") is None
    assert parade.get_input_names() == [case.input.name] and parade.get_output_names() == [case.output.name]
    assert parade.get_raw_tensor_data(case.input.name) != 0 and parade.get_raw_tensor_data("nope") == 0

    # wrong arguments raise what the reference raises
    with pytest.raises(ValueError, match="input shape not match"):
        parade.run({case.input.name: x[:1]}, outputs)
    with pytest.raises(ValueError, match="input dtype not match"):
        parade.run({case.input.name: x.astype(np.float32)}, outputs)
    with pytest.raises(ValueError, match="input dim size not match"):
        parade.run({case.input.name: x.reshape(-1)}, outputs)
    with pytest.raises(ValueError, match="output dtype not match"):
        parade.run(inputs, {case.output.name: got.astype(np.float64)})

    # reshape to another batch (module.cpp:381-400), then run again
    shape = list(case.input.shape)
    shape[0] = 3
    assert parade.reshape({case.input.name: shape}) is True
    assert parade.reshape({case.input.name: shape[:3]}) is False  # rank mismatch
    inputs3, outputs3 = art.get_empty_io(parade)
    x3 = rng.integers(0, 256, shape, dtype=np.uint8)
    inputs3[case.input.name][:] = x3
    parade.run(inputs3, outputs3)
    want3 = casecpu.run_case(cases.resnet18(N=3, hw=96), x3)[case.output.name].reshape(3, -1)
    assert np.array_equal(outputs3[case.output.name], want3)
    # forward() alone re-runs on what the input memory holds
    parade.forward()


def test_float_network_ends_and_missing_modules(tmp_path):
    case = cases.resnet50(N=1, hw=64)  # fp32 input -> quantize ... dequantize -> fp32 output
    fp = _write(str(tmp_path), case)
    rng = np.random.default_rng(6)
    x = (rng.standard_normal(case.input.shape) * 1.2).astype(np.float32)
    want = casecpu.run_case(case, x)[case.output.name].reshape(1, -1)
    # a module that does not exist is skipped with a message, like the reference (module.cpp:104-110)
    ctx = art.RuntimeContext(["no_such_module", "hip"], "hip")
    assert ctx.loaded_workspaces == ["hip"]
    parade = art.load_parade(fp, ctx)
    inputs, outputs = art.get_empty_io(parade)
    assert inputs[case.input.name].dtype == np.float32
    inputs[case.input.name][:] = x
    parade.run(inputs, outputs)
    assert np.array_equal(outputs[case.output.name].view(np.uint32), want.view(np.uint32))
    ctx2 = art.create_context_for_target("hip")
    assert ctx2.loaded_workspaces == ["hip"]


def bottleneck_chain(N, blocks=3):
    """Identity bottleneck blocks of 256 middle channels on 14x14 images: one launch each, or three in a recorded pass on few images."""
    c = cases.Case("bottleneck_chain_n%d" % N, 12)
    t = c.input_u8((N, 1024, 14, 14), 0.0186, 114)
    for _ in range(blocks):
        b = c.conv(c.conv(t, 256, 1, ozp=0), 256, 3, ozp=0)
        t = c.add(c.conv(b, 1024, 1), t)
    c.output = t
    return c


@pytest.mark.parametrize("build", [lambda: cases.resnet18(N=2, hw=96), lambda: cases.mobilenet_v2(N=1, hw=70), lambda: cases.resnet50(N=2, hw=64),
                                   lambda: bottleneck_chain(2)])
def test_recorded_passes_follow_their_inputs(tmp_path, build):
    """The first pass runs operator by operator, the second is recorded, later ones replay the record: every one on new
    inputs, with other GPU work and synchronisations between, with and without a new input, before and after a reshape."""
    case = build()
    ctx = art.create_context_for_target("hip")
    parade = art.Parade(engine.write_engine(case), ctx)
    inputs, outputs = art.get_empty_io(parade)
    name, out = case.input.name, case.output.name
    noise = torch.zeros(1 << 20, device="cuda")
    for k in range(6):
        print("pass", k, case.name, flush=True)
        x = casecpu.random_input(case, k)
        want = casecpu.run_case(case, x)[out].reshape(outputs[out].shape)
        parade.run({name: x}, outputs)
        assert np.array_equal(outputs[out].view(np.uint8), want.view(np.uint8)), k
        noise.add_(1.0)
        if k % 2:
            torch.cuda.synchronize()
        if k in (0, 3):  # the same input again, and what the input memory holds
            parade.forward()
            assert np.array_equal(parade._outputs[out].numpy().view(np.uint8), want.view(np.uint8)), k
            assert np.array_equal(parade._inputs[name].numpy().view(np.uint8), x.view(np.uint8))
        if k == 4:
            assert parade.reshape({name: list(case.input.shape)}) is True


@pytest.mark.parametrize("shape", [(1, 3, 5, 7), (3, 3, 70, 67), (2, 3, 431, 433), (5, 3, 640, 641)])
def test_arrays_of_every_size_reach_the_device(shape):
    """Parade.run's way of an array to the GPU: below and above the sizes at which helper threads copy, the copy engine is used
    and the copies are cut; values quantized on the way in, values that are not (a misaligned array) and bytes."""
    rng = np.random.default_rng(shape[2])
    for kind in ("f32", "misaligned", "u8"):
        c = cases.Case("write", 0)
        if kind == "u8":
            c.dequantize(c.input_u8(shape, 0.25, 7))
        else:
            c.dequantize(c.quantize(c.input_f32(shape), 0.0186, 114))
        parade = art.Parade(engine.write_engine(c), art.create_context_for_target("hip"))
        _, outputs = art.get_empty_io(parade)
        for k in range(3):
            print(shape, kind, k, flush=True)
            if kind == "u8":
                x = rng.integers(0, 256, shape, dtype=np.uint8)
                q, alpha, zp = x, 0.25, 7
            else:
                x = (rng.standard_normal(shape) * 2.0).astype(np.float32)
                x.reshape(-1)[:8] = [np.nan, np.inf, -np.inf, 0.0, 0.0093, -2.1204, 2.6226, 1e30]
                x.reshape(-1)[-8:] = np.float32(0.0186) * (np.arange(8, dtype=np.float32) + 0.5)
                if kind == "misaligned":
                    raw = np.zeros(x.nbytes + 1, np.uint8)
                    raw[1:] = x.reshape(-1).view(np.uint8)
                    x = raw[1:].view(np.float32).reshape(shape)
                q, alpha, zp = orc.quantize_u8(np.array(x), 0.0186, 114), 0.0186, 114
            parade.run({c.input.name: x}, outputs)
            want = orc.dequantize_u8(q, alpha, zp)
            assert np.array_equal(outputs[c.output.name].view(np.uint32), want.reshape(outputs[c.output.name].shape).view(np.uint32)), (kind, k)
            assert np.array_equal(parade._inputs[c.input.name].numpy().view(np.uint8), np.array(x).view(np.uint8))


@pytest.mark.parametrize("n", [1, 3])
def test_first_layer_and_shortcut_run_as_one_launch_in_recorded_passes(n, tmp_path):
    """ResNet-18's three strided stages begin with two convolutions of one tensor: from the second pass on one launch computes both, in the
    pass that is recorded and in every replay, and new inputs give the oracle's bytes each time."""
    import ctypes
    case = cases.resnet18(N=n, hw=64, seed=3)
    fp = _write(str(tmp_path), case)
    parade = art.load_parade(fp, art.create_context_from_json(fp + ".json"))
    inputs, outputs = art.get_empty_io(parade)
    chained = ctypes.CDLL(os.path.join(os.path.dirname(art.__file__), "lib", "libart_module_hip.so")).hip_module_chained_convs
    chained.restype = ctypes.c_long
    rng = np.random.default_rng(n)
    for k in range(5):
        x = rng.integers(0, 256, case.input.shape, dtype=np.uint8)
        inputs[case.input.name][:] = x
        before = chained()
        parade.run(inputs, outputs)
        assert chained() - before == (3 if k else 0), k
        want = casecpu.run_case(case, x)[case.output.name].reshape(n, -1)
        assert np.array_equal(outputs[case.output.name], want), k
