"""What the kernel sources promise the compiler, checked without a GPU."""

from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "mlx-gptq-mxfp_amd", "csrc")


def _code(name: str) -> str:
    with open(os.path.join(CSRC, name)) as f:
        txt = f.read()
    return re.sub(r"/\*.*?\*/|//[^\n]*", "", txt, flags=re.S)


@pytest.mark.parametrize(
    "name", sorted(n for n in os.listdir(CSRC) if n.endswith((".hip", ".h"))))
def test_lds_is_handed_over_with_fences(name):
    """The bare barrier builtin orders no memory for the compiler, so a read of
    what another wave brought to LDS could move above it: waves hand LDS over
    through __syncthreads (lds_handover). The exception is the Hessian kernel,
    which keeps several stages of loads in flight over its barriers (a fence
    would wait for all of them) and fixes its order by sched_barrier."""
    bare = len(re.findall(r"__builtin_amdgcn_s_barrier\b", _code(name)))
    assert bare == 0 or name == "hessian.hip"


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not available")
def test_piecewise_loads_need_no_more_than_their_elements_alignment(tmp_path):
    exe = tmp_path / "check_loads"
    subprocess.run(["hipcc", "-O1", "-std=c++17", "-Xarch_host", "-fsanitize=alignment",
                    "-Xarch_host", "-fsanitize-trap=alignment", "-I", CSRC,
                    os.path.join(os.path.dirname(__file__), "native", "check_unaligned_loads.hip"),
                    "-o", str(exe)], check=True, capture_output=True)
    res = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert res.returncode == 0, res.stdout + res.stderr


def test_pointers_that_may_be_unaligned_are_read_piecewise():
    """The general deferred update takes any U and Err, the final sum of the
    relative error any partials: no 16-byte type is laid over them."""
    update = _code("gptq_affine.hip").split("lazy_update_kernel(")[1].split("__global__")[0]
    total = _code("gptq_mxfp.hip").split("rel_err_kernel(")[1].split("__global__")[0]
    assert not re.search(r"float4\*>\((Eb|Ub|Err|U)\b", update)
    assert "double2" not in total
