"""Q2_K and Q3_K layers that hold two copies: how many bytes of second ones a ctx's layers may hold (on a plan-only ctx; on a GPU, what
a layer without one computes)."""
import ctypes as C
import shutil
import subprocess
import sys

import numpy as np
import pytest

from oxydllm_amd import _lib, ops, synth
from tests.helpers import fake

N, K = 4096, 4096
MB = {synth.GGUF_Q2_K: 5.25, synth.GGUF_Q3_K: 7.125}  # of the matrix-core copy


class Layer:
    def __init__(self, ctx, fmt, dt=_lib.BF16, n=N, at=0):
        self.lib, self.ctx, self.dt, self.n, self.at, self.h = _lib.load(), ctx, dt, n, at, C.c_void_p()
        elems, size = synth.GGUF_BLOCK_LAYOUT[fmt]
        rc = self.lib.oxq_qlinear_new(ctx.handle, fmt, C.byref(self.tensor((n * (K // elems) * size,), _lib.U8)), K, n, None, dt, C.byref(self.h))
        assert rc == 0, self.lib.oxq_last_error().decode()

    def tensor(self, shape, dt):
        t = fake(shape, dt)
        t.data = self.at
        return t

    def kernel(self, m):
        assert self.lib.oxq_qlinear_forward(self.h, None, C.byref(self.tensor((m, K), self.dt)), C.byref(self.tensor((m, self.n), self.dt))) == 0
        return self.ctx.last_plan()["kernel"]

    def both(self):
        return "_mfma_" in self.kernel(4)

    def free(self):
        self.lib.oxq_qlinear_free(self.h)


@pytest.mark.parametrize("fmt", list(MB))
@pytest.mark.parametrize("dt", [_lib.BF16, _lib.F32])
def test_second_copies_are_bounded_and_given_back(fmt, dt):
    ctx = ops.Context(plan_only=True)
    ctx.set_tuning("OXQ_GGUF_BOTH_MB", int(2 * MB[fmt] + 1))
    a, b, c = (Layer(ctx, fmt, dt) for _ in range(3))
    assert [x.both() for x in (a, b, c)] == [True, True, False]
    # the layer without one: every row count on the kernels of the rotated copy and of the file layout
    assert "_res_gemv_" in c.kernel(1) and "_res_gemv_" in c.kernel(4)
    if dt == _lib.BF16:
        assert "_mul_mm_" in c.kernel(200) and "_gemm_" in a.kernel(200)
    a.free()
    d = Layer(ctx, fmt, dt)
    assert d.both()
    ctx.set_tuning("OXQ_GGUF_BOTH_MB", 0)
    e = Layer(ctx, fmt, dt)
    assert not e.both() and d.both()
    for x in (b, c, d, e):
        x.free()


def test_other_formats_and_small_layers_do_not_count():
    ctx = ops.Context(plan_only=True)
    ctx.set_tuning("OXQ_GGUF_BOTH_MB", 6)
    others = [Layer(ctx, synth.GGUF_Q4_K, _lib.F32), Layer(ctx, synth.GGUF_Q4_K), Layer(ctx, synth.GGUF_Q2_K, n=240)]
    assert "_mfma_f32" in others[0].kernel(4) and "_mfma_bf16" in others[1].kernel(4) and not others[2].both()
    q = Layer(ctx, synth.GGUF_Q2_K)
    assert q.both()
    for x in others + [q]:
        x.free()


def test_the_default_is_a_32nd_of_the_device_and_layers_outlive_their_ctx():
    ctx = ops.Context(plan_only=True)
    layers, n = [], 28672 * 4
    while not layers or layers[-1].both():
        layers.append(Layer(ctx, synth.GGUF_Q2_K, n=n))
        assert len(layers) < 200
    held = (len(layers) - 1) * n * (K // 256) * 84
    assert held <= (288 << 30) // 32 < held + n * (K // 256) * 84
    ctx.close()
    for x in layers:
        x.free()


# The calls of the HIP runtime that building and calling a layer makes, on a device that is not there: allocations above `most` bytes
# fail, launches do nothing.
NO_DEVICE = r"""
#include <cstddef>
#include <cstdlib>
extern "C" {
size_t most = ~(size_t)0;
int failed = 0;
int hipGetDeviceCount(int *n) { return *n = 1, 0; }
int hipGetDevice(int *d) { return *d = 0, 0; }
int hipSetDevice(int) { return 0; }
int hipDeviceGetAttribute(int *v, int, int) { return *v = 256, 0; }
int hipDeviceTotalMem(size_t *b, int) { return *b = (size_t)288 << 30, 0; }
int hipMalloc(void **p, size_t b) { return b > most ? (++failed, 2) : (*p = malloc(b), 0); }
int hipFree(void *p) { return free(p), 0; }
int hipMemset(void *, int, size_t) { return 0; }
int hipDeviceSynchronize() { return 0; }
int hipStreamSynchronize(void *) { return 0; }
int hipGetSymbolAddress(void **p, const void *) { static char array[256]; return *p = array, 0; }
int hipFuncSetAttribute(const void *, int, int) { return 0; }
int hipLaunchKernel(const void *, ...) { return 0; }
int hipGetLastError() { return 0; }
}
"""


def out_of_memory(rt, fmt, dt):
    """Run by a process of its own (below), where the symbols of NO_DEVICE (rt) stand before the runtime's."""
    most, failed = C.c_size_t.in_dll(rt, "most"), C.c_int.in_dll(rt, "failed")
    ctx = ops.Context(device=0)
    ctx.set_tuning("OXQ_GGUF_BOTH_MB", int(MB[fmt] + 1))  # room for one
    most.value = int(MB[fmt] * 1.5) << 20
    a = Layer(ctx, fmt, dt, at=4096)
    assert failed.value == 1 and "_res_gemv_" in a.kernel(4), (failed.value, a.kernel(4))
    most.value = ~0 & (2**64 - 1)
    b = Layer(ctx, fmt, dt, at=4096)
    c = Layer(ctx, fmt, dt, at=4096)
    assert failed.value == 1 and b.both() and not c.both()
    for x in (a, b, c):
        x.free()
    print("given back")


@pytest.mark.parametrize("fmt", list(MB))
@pytest.mark.parametrize("dt", [_lib.BF16, _lib.F32])
def test_a_second_copy_that_cannot_be_allocated_is_left_out_and_not_counted(fmt, dt, tmp_path):
    if not shutil.which("g++"):
        pytest.skip("no g++")
    lib = tmp_path / "no_device.so"
    subprocess.run(["g++", "-shared", "-fPIC", "-x", "c++", "-", "-o", str(lib)], input=NO_DEVICE, text=True, check=True)
    code = (f"import ctypes as C; rt = C.CDLL({str(lib)!r}, mode=C.RTLD_GLOBAL)\n"  # before torch, which brings the runtime
            f"from tests.test_gguf_second_copies import out_of_memory as t; t(rt, {fmt}, {dt})")
    run = subprocess.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=300)
    assert run.returncode == 0 and "given back" in run.stdout, run.stdout + run.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("fmt", list(MB))
def test_layers_without_a_second_copy_compute_what_they_did_without_any(fmt):
    import torch
    from tests.helpers import bits_of, to_dev, tune
    n, k = 1040, 1024
    wd = to_dev(synth.gguf_weight(fmt, n, k, seed=fmt))
    for dt in (torch.bfloat16, torch.float32):
        tune("OXQ_GGUF_BOTH_MB", 0)
        bounded = ops.QLinear(fmt, wd, k, n, None, dt)
        tune("OXQ_GGUF_BOTH_MB", None)
        both = ops.QLinear(fmt, wd, k, n, None, dt)
        tune("OXQ_GGUF_MFMA", 0)
        one = ops.QLinear(fmt, wd, k, n, None, dt)
        tune("OXQ_GGUF_MFMA", None)
        x = torch.randn((40, k), generator=torch.Generator().manual_seed(1)).to(dt).cuda()
        for m in (1, 3, 8, 40):
            print(f"[case] second copy {fmt} {dt} m={m}", flush=True)
            y = bounded.forward(x[:m])
            assert "_gemm_" not in ops.default_context().last_plan()["kernel"] and "_mfma_" not in ops.default_context().last_plan()["kernel"]
            assert np.array_equal(bits_of(y), bits_of(one.forward(x[:m])))
        both.forward(x[:4])
        assert "_mfma_" in ops.default_context().last_plan()["kernel"]
