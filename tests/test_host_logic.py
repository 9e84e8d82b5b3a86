"""Host-side API behaviour that needs no GPU: argument validation raises the
reference's exception types before any device work, and the product path
refuses to compute without a HIP device (no CPU fallback)."""

from __future__ import annotations

import numpy as np
import pytest
import torch

from mlx_gptq import grid, packing


def test_mode_defaults_and_errors():
    assert grid.mode_defaults("mxfp4") == (32, 4)
    assert grid.mode_defaults("mxfp8") == (32, 8)
    assert grid.mode_defaults("affine") == (64, 4)
    with pytest.raises(ValueError):
        grid.mode_defaults("int3")
    with pytest.raises(ValueError):
        grid._mxfp_max("affine")
    assert grid._E2M1_VALUES[7] == 6.0 and grid.MX_GROUP_SIZE == 32


def test_pack_validation_precedes_device_work():
    with pytest.raises(ValueError):
        packing.pack_q(np.zeros((2, 8), dtype=np.uint8), 3)
    with pytest.raises(AssertionError):
        packing.pack_mxfp4(np.zeros(4, dtype=np.uint8))


def test_rtn_mxfp_validation():
    with pytest.raises(ValueError):
        grid.rtn_quantize_mxfp(torch.zeros(2, 48), "mxfp4")


@pytest.mark.skipif(torch.cuda.is_available(), reason="checks the no-GPU behaviour")
def test_no_cpu_fallback_without_gpu():
    with pytest.raises(RuntimeError, match="HIP devices only"):
        grid.rtn_quantize_mxfp(torch.zeros(2, 64), "mxfp4")
    with pytest.raises(RuntimeError, match="HIP devices only"):
        packing.pack_q(np.zeros((2, 8), dtype=np.uint8), 4)


def test_packed_out_validation():
    """solve_gptq's packed_out is checked for shape, dtype, layout, device and
    alignment before any launch (gptq._check_packed), for the pack widths
    pack_q accepts (packing.py:15-26)."""
    from mlx_gptq import gptq

    dev = torch.device("cpu")
    ok = torch.zeros(2, 3, 64 * 4 // 32, dtype=torch.int32)
    gptq._check_packed(ok, (2, 3, 64), 4, dev)
    gptq._check_packed(torch.zeros(2, 3, 16, dtype=torch.int32), (2, 3, 64), 8, dev)
    bad = [torch.zeros(2, 3, 9, dtype=torch.int32),            # wrong width
           torch.zeros(2, 3, 8, dtype=torch.int64),            # wrong dtype
           torch.zeros(2, 3, 16, dtype=torch.int32)[..., ::2]]  # not contiguous
    for b in bad:
        with pytest.raises(ValueError, match="packed_out"):
            gptq._check_packed(b, (2, 3, 64), 4, dev)
    with pytest.raises(ValueError, match="cannot pack"):
        gptq._check_packed(ok, (2, 3, 64), 3, dev)
    with pytest.raises(ValueError, match="packed_out"):
        gptq._check_packed(ok, (2, 3, 64), 4, torch.device("meta"))


@pytest.mark.parametrize("C,R", [(64, 64), (768, 2048), (2048, 1536), (4096, 14336), (1000, 100)])
def test_expert_bytes_of_an_affine_solve_counts_every_buffer(C, R):
    """What one expert's affine solve allocates: H, W_dq, codes, scales and
    biases, U, the factorisation's workspace and the errors of the column loop."""
    from mlx_gptq import _native as nat
    from mlx_gptq import span_solve

    err_cols = min(C, 512)
    buffers = (4 * C * C + 4 * R * C + R * C + 2 * 2 * R * (C // 64) + 4 * C * C
               + int(nat.load().mgq_hinv_full_workspace_size(1, C)) + 4 * R * err_cols)
    assert span_solve.expert_bytes(C, R, "affine") >= buffers
    assert span_solve.expert_span_size(C, R, 3.5 * buffers / (1 << 30), "affine") <= 3


@pytest.mark.parametrize("steps", [0, 1, 20, 123, 124, 127, 128])
def test_clip_steps_have_one_bound(steps):
    """choose_qparams and both solver entries take the same numbers of clip steps
    (empty calls: nothing is launched)."""
    from mlx_gptq import _native as nat

    calls = [("mgq_choose_qparams", None, 0, 64, 4, 1, 0, steps, 0.2, None, None, None, None, None),
             ("mgq_gptq_affine_block", None, None, 0, 1, 64, 0, 64, 64, 4, 1, 0, steps, 0.2, None,
              None, None, None, None),
             ("mgq_gptq_affine", None, None, 0, 1, 64, 64, 64, 4, 1, 0, steps, 0.2, None, None, None,
              None, 64, None)]
    for c in calls:
        if 1 <= steps < 128:
            nat.call(*c)
        else:
            with pytest.raises(ValueError):
                nat.call(*c)
