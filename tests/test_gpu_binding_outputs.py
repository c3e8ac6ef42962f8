"""Outputs that the native binding makes are what torch.empty makes: dispatch modes and torch function modes see the
allocation, and it is filled under deterministic algorithms."""
import numpy as np
import pytest
import torch
from torch.overrides import TorchFunctionMode
from torch.utils._python_dispatch import TorchDispatchMode

from oxydllm_amd import ops, synth
from tests.helpers import to_dev

pytestmark = pytest.mark.gpu


class Seen(TorchDispatchMode):
    def __init__(self):
        super().__init__()
        self.shapes = []

    def __torch_dispatch__(self, func, types, args=(), kwargs=None):
        out = func(*args, **(kwargs or {}))
        if "empty" in func.name():
            self.shapes.append(tuple(out.shape))
        return out


class SeenCalls(TorchFunctionMode):
    def __init__(self):
        super().__init__()
        self.calls = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        if func in (torch.empty, torch.empty_like):
            self.calls.append(func)
        return func(*args, **(kwargs or {}))


def packed(K, N):
    qw, qz, sc = synth.awq_checkpoint(K, N, 128, 4, seed=1)
    return to_dev(qw), to_dev(qz), to_dev(sc, torch.float16)


@pytest.mark.parametrize("mode", [Seen, SeenCalls])
def test_modes_see_the_outputs(mode):
    args = packed(256, 512)
    layer = ops.PackedQuantLinear(4, ops.PACK_OUT, *args, None, torch.float16)
    gu = ops.PackedQuantLinear(4, ops.PACK_OUT, *packed(256, 1024), None, torch.float16, gate_up_act=ops.ACT_GATED_SILU)
    down = ops.PackedQuantLinear(4, ops.PACK_OUT, *packed(512, 256), None, torch.float16)
    ffn = ops.FeedForward(ops.GATE_UP_FUSED, gu, None, down, 512)
    x = torch.randn((2, 3, 256), device="cuda").half()
    logits = torch.randn((3, 8), device="cuda")
    y = layer.forward(x)
    print("[case] outputs under a mode", flush=True)
    with mode() as seen:
        got = layer.forward(x)
        ops.w4a16_matmul(x[0], *args)
        ffn.forward(x)  # scratch and output
        ops.moe_route_group(logits, 2)  # six
        ops.silu_mul(y, y)
        layer.forward(x, out=y)  # none
    assert torch.equal(got, layer.forward(x))
    if mode is SeenCalls:
        assert seen.calls == [torch.empty] * 10 + [torch.empty_like]
    else:
        assert len(seen.shapes) == 11 and seen.shapes[0] == (2, 3, 512) and seen.shapes[1] == (3, 512), seen.shapes


def test_outputs_are_filled_under_deterministic_algorithms():
    """A plan-only context writes nothing: what the call returns is what was allocated."""
    plan = ops.Context(plan_only=True)
    logits = torch.randn((64, 32), device="cuda")
    keep = [torch.zeros(1 << 16, device="cuda") for _ in range(4)]
    del keep  # memory that was written is handed out again
    print("[case] deterministic fill", flush=True)
    torch.use_deterministic_algorithms(True)
    try:
        idx, vals = ops.moe_route(logits, 4, ctx=plan)
    finally:
        torch.use_deterministic_algorithms(False)
    assert bool(vals.isnan().all()) and bool((idx == np.iinfo(np.int32).max).all())
