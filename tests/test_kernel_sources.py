"""What the kernel sources promise the compiler, checked without a GPU."""

from __future__ import annotations

import os
import re

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
