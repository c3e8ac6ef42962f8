"""The counted waits of the kernels that load straight into LDS, checked in the compiled code.

Their barriers publish a stage of x once the loads into it are over, and each wait counts how many younger loads may still be
under way: weights, whose loads are plain ones that the compiler may move or leave out.  If one moves over a wait, the
count covers a load into LDS that has to be over, which no run need show.  Vector-memory instructions finish in order,
so the number of loads into LDS that can be under way at a barrier, over all paths, says whether that has happened."""
import os

import pytest

from oxydllm_amd import _lib
from tests import gpu_code

# Two buffers, the other one filled meanwhile: nothing under way at any barrier.  pk4_mid_kernel: four stages, of which
# the two after the published one are filled meanwhile, four loads a wave each; pk4_mid128_kernel and
# pk4_midfold_kernel: five, the published one the next but one, and the same two.
ALLOWED = {"pk4_gemm_kernel": 0, "pk4n_gemm_kernel": 0, "ggm_gemm_kernel": 0, "f8_gemm_kernel": 0, "f8_gemm128_kernel": 0,
           "mxfp4_gemm_kernel": 0, "pk4_mid_kernel": 8, "pk4_mid128_kernel": 8, "pk4_midfold_kernel": 8}


@pytest.fixture(scope="module")
def found(tmp_path_factory):
    if not os.path.exists(gpu_code.LLVM + "llvm-objdump"):
        pytest.skip("no llvm-objdump")
    out = {}
    for co in gpu_code.code_objects(_lib.LIB_PATH, tmp_path_factory.mktemp("co")):
        if any(name.encode() in co.read_bytes() for name in ALLOWED):
            out.update({n: c for n, c in gpu_code.kernels(co).items() if any(k in n for k in ALLOWED)})
    return out


def kernel_of(name):
    return next(k for k in ALLOWED if f"{k}<" in name)


def test_loads_into_lds_are_over_where_a_barrier_publishes_them(found):
    assert {kernel_of(n) for n in found} == set(ALLOWED) and len(found) >= 135
    for name, code in found.items():
        at = gpu_code.loads_under_way_at_barriers(code)
        assert len(at) >= 2 and max(at.values()) <= ALLOWED[kernel_of(name)], (name, {hex(a): n for a, n in at.items()})


def test_no_form_of_128_rows_or_unrounded_weights_between_decode_and_prefill_uses_scratch(found):
    """Their registers are full: one too many lies in scratch memory, and its reload waits for every load under way."""
    checked = {n: c for n, c in found.items() if "pk4_mid128_kernel<" in n or "pk4_midfold_kernel<" in n}
    assert len(checked) == 20
    for name, code in checked.items():
        assert not [a for a, op, *_ in code if op.startswith("scratch_")], name


def test_a_load_that_moved_over_its_wait_is_noticed(found):
    """The same code with every counted wait one higher, as if one weight load less came before it."""
    for kernel, allowed in ALLOWED.items():
        code = next(c for n, c in found.items() if f"{kernel}<" in n)

        def more(args):
            return gpu_code.re.sub(r"vmcnt\((\d+)\)", lambda m: f"vmcnt({int(m.group(1)) + 1})" if m.group(1) != "0" else m.group(0), args)
        moved = [(a, op, more(args) if op == "s_waitcnt" else args, t) for a, op, args, t in code]
        assert max(gpu_code.loads_under_way_at_barriers(moved).values()) > allowed, kernel
