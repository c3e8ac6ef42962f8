"""The native half of the torch binding on plan-only contexts: no GPU needed."""
import importlib.machinery
import os
import subprocess
import sys

import pytest
import torch

from oxydllm_amd import _lib, build, ops
from tests.helpers import fake

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
K, N, G = 256, 512, 128


def packed(dt=_lib.F16):
    return fake((K, N // 8), _lib.I32), fake((K // G, N // 8), _lib.I32), fake((K // G, N), dt)


def packed_layer(ctx):
    return ops.PackedQuantLinear(4, ops.PACK_OUT, *packed(), None, torch.float16, ctx=ctx)


@pytest.fixture
def plan():
    return ops.Context(plan_only=True)


def test_module_is_tagged_and_reported_when_missing(monkeypatch, tmp_path):
    """Another interpreter does not load it, and a tree with the library alone builds it."""
    assert build.TORCH_LIB.endswith(importlib.machinery.EXTENSION_SUFFIXES[0])
    assert sys.implementation.cache_tag in build.TORCH_LIB  # cpython-310
    assert build.missing() == []
    monkeypatch.setattr(build, "TORCH_LIB", str(tmp_path / "not_there.so"))
    assert build.missing() == [str(tmp_path / "not_there.so")]


def test_plan_only_use_without_a_gpu_torch(tmp_path):
    """The module built for a torch without ROCm links nothing of it, and plan-only contexts work; a call that needs a
    stream says why it cannot have one."""
    out = str(tmp_path / os.path.basename(build.TORCH_LIB))
    build.build_torch_binding(out, gpu=False, opt="-O0")
    needed = subprocess.run(["readelf", "-d", out], capture_output=True, text=True, check=True).stdout
    assert "hip" not in needed, needed
    code = f"""
import importlib.util, sys
import torch
sys.path.insert(0, {ROOT!r})
spec = importlib.util.spec_from_file_location("oxydllm_amd._oxq_torch", {out!r})
module = importlib.util.module_from_spec(spec)
spec.loader.exec_module(module)
sys.modules["oxydllm_amd._oxq_torch"] = module
from oxydllm_amd import _lib, ops
assert ops._native is module
from tests.helpers import fake
plan = ops.Context(plan_only=True)
layer = ops.PackedQuantLinear(4, ops.PACK_OUT, fake(({K}, {N // 8}), _lib.I32), fake(({K // G}, {N // 8}), _lib.I32),
                              fake(({K // G}, {N}), _lib.F16), None, torch.float16, ctx=plan)
layer.forward(fake((3, {K}), _lib.F16), out=fake((3, {N}), _lib.F16))
assert plan.last_plan()["kernel"].startswith("pk4_"), plan.last_plan()
try:
    module.current_device()
except RuntimeError as e:
    assert "no GPU support" in str(e)
else:
    raise AssertionError("current_device() without a GPU torch")
print("ok")
"""
    res = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True)
    assert res.returncode == 0 and res.stdout.strip() == "ok", res.stderr[-2000:]


def test_descriptors_in_place_of_tensors(plan):
    out = fake((3, N), _lib.F16)
    before = sys.getrefcount(out)
    layer = packed_layer(plan)
    for _ in range(4):
        assert layer.forward(fake((3, K), _lib.F16), out=out) is out
    assert sys.getrefcount(out) == before
    native = ops._native
    assert native.w4a16_matmul(plan.native, fake((2, K), _lib.F16), out := fake((2, N), _lib.F16), N, *packed()) is out
    assert plan.last_plan()["launches"] >= 1
    with pytest.raises(TypeError, match="expected a tensor"):  # nothing to take an output's type and device from
        layer.forward(fake((3, K), _lib.F16))


def test_wrong_arguments(plan):
    layer, x, out = packed_layer(plan), fake((3, K), _lib.F16), fake((3, N), _lib.F16)
    for bad in ("x", 3, [1.0], object()):
        with pytest.raises(TypeError, match="expected a tensor"):
            layer.forward(bad, out=out)
        with pytest.raises(TypeError, match="expected a tensor"):
            layer.forward(x, out=bad)
    with pytest.raises(ops.OxqError) as e:
        layer.forward(torch.zeros((3, K), dtype=torch.float64), out=out)
    assert e.value.status == -2 and "unsupported torch dtype" in e.value.message
    for shape in ((), (1,) * 5):
        with pytest.raises(ops.OxqError) as e:
            layer.forward(torch.zeros(shape, dtype=torch.float16), out=out)
        assert e.value.status == -3 and f"rank {len(shape)} out of [1, 4]" in e.value.message
    with pytest.raises(ops.OxqError) as e:  # the library's own checks and message
        layer.forward(fake((3, K + 8), _lib.F16), out=out)
    assert e.value.status == -3 and "in_features" in e.value.message
    with pytest.raises(ops.OxqError) as e:  # host tensors, with an output the binding makes
        layer.forward(torch.zeros((3, K), dtype=torch.float16))
    assert e.value.status == -7
    with pytest.raises(TypeError):
        layer._forward(x)
    with pytest.raises(TypeError):
        layer._forward(x, out=out)  # positional only
    with pytest.raises(TypeError):
        layer._forward(x, out, None)
    with pytest.raises(TypeError, match="expected a native handle"):
        ops._native.w4a16_matmul(plan, x, out, N, *packed())
    with pytest.raises(TypeError, match="expected 7 arguments"):
        ops._native.w4a16_matmul(plan.native, x, out)
    with pytest.raises(TypeError, match="not callable"):
        plan.native(x, out)
    with pytest.raises(OverflowError):
        ops._native.w4a16_matmul(plan.native, x, out, 1 << 80, *packed())
    with pytest.raises(TypeError):
        ops.moe_route(fake((3, 8), _lib.F32), 2, ctx=plan)  # the outputs need the tensor's shape and device


def test_closed_handles(plan):
    x, out = fake((2, K), _lib.F16), fake((2, N), _lib.F16)
    ops._native.w4a16_matmul(plan.native, x, out, N, *packed())
    plan.close()
    plan.close()
    with pytest.raises(ops.OxqError) as e:
        ops._native.w4a16_matmul(plan.native, x, out, N, *packed())
    assert e.value.status == -1
    ctx = ops.Context(plan_only=True)
    experts = ops.Mxfp4Experts(fake((4 * 64 * 64 // 2,), _lib.U8), fake((4 * 64 * 64 // 32,), _lib.U8), None, 4, 64, 64, ctx=ctx)
    experts.close()
    with pytest.raises(ops.OxqError) as e:
        experts.matmul(fake((2, 64), _lib.BF16), fake((5,), _lib.I32), None, out=fake((2, 64), _lib.BF16))
    assert e.value.status == -1
