"""HIP affine GPTQ solver (full damped Cholesky-inverse + lazy-block column
loop with the MSE clip search) vs the reference golden vectors and the CPU
oracle.

Gates: final codes agree on >= 99.5% of
elements; proxy loss tr((W-Q) H (W-Q)^T) within 1%; W_dq is exactly the
decode q*s + b of the emitted codes and stored params. The full-matrix U is
checked against an fp64 factor of the same damped matrix (the reference's
fp32 LAPACK result is within its own rounding of that) and the reference's
escalation warnings / RuntimeError are reproduced on crafted inputs.
"""

from __future__ import annotations

import logging

import pytest
import torch

from oracle import gptq_ref, hessian_ref
from tests import golden_io

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _agree(a: torch.Tensor, b: torch.Tensor) -> float:
    return float((a.cpu() == b.cpu()).float().mean())


def _proxy(W, Wq, H):
    return gptq_ref.proxy_loss(W.cpu(), Wq.cpu(), H.cpu())


def _setup(B=2, R=32, C=128, N=512, seed=0, scale=1.0, outliers=0):
    g = torch.Generator().manual_seed(seed)
    base = torch.randn(N, C, generator=g)
    X = base + 0.5 * torch.roll(base, 1, dims=1)
    X = X * torch.exp(torch.randn(C, generator=g) * 0.5)
    if outliers:
        X[:, torch.randperm(C, generator=g)[:outliers]] *= 20.0
    W = torch.randn(B, R, C, generator=g) * scale
    H = (X.T @ X).unsqueeze(0).repeat(B, 1, 1).contiguous()
    for b in range(1, B):
        H[b] *= 1.0 + 0.5 * b
    return W, H, X


def _check_vs(W, q, s, b, W_dq, rq, rs, rb, rW, H_after, min_agree=0.995):
    from mlx_gptq import grid

    G = W.shape[-1] // s.shape[-1]
    assert _agree(q, rq) >= min_agree, _agree(q, rq)
    if s.dtype == torch.float32:
        # unrounded params carry the last-ulp differences of the error
        # recurrence (reduction order of the lazy-update GEMM) straight through
        assert torch.allclose(s.cpu(), rs, rtol=1e-4, atol=0)
        assert torch.allclose(b.cpu(), rb, rtol=1e-4, atol=1e-7)
    else:
        assert _agree(s, rs) >= 0.99 and _agree(b, rb) >= 0.99
    assert torch.equal(grid.dequantize_artifact(q, s, b, "affine", G), W_dq)
    pl, pl_ref = _proxy(W, W_dq, H_after), _proxy(W, rW, H_after)
    assert torch.all((pl - pl_ref).abs() <= 0.01 * pl_ref.abs()), (pl, pl_ref)


@pytest.mark.parametrize("name", ["affine4_g64", "affine4_g32_f32", "affine2_g32",
                                  "affine8_g128_minmax"])
def test_affine_matches_reference_golden(name):
    from mlx_gptq import gptq

    t, meta = golden_io.load()
    kw = golden_io.case_kwargs(meta["cases"][name])
    W, H = t[f"{name}.W"], t[f"{name}.H"]
    Hd = H.clone().to(DEV)
    q, s, b, W_dq, rel = gptq.solve_gptq(W.to(DEV), Hd, **kw)
    assert torch.equal(Hd.cpu(), t[f"{name}.H_after"])
    assert s.dtype == t[f"{name}.scales"].dtype and b.dtype == t[f"{name}.biases"].dtype
    _check_vs(W, q, s, b, W_dq, t[f"{name}.q"], t[f"{name}.scales"], t[f"{name}.biases"],
              t[f"{name}.W_dq"], t[f"{name}.H_after"])
    assert torch.allclose(rel.cpu(), t[f"{name}.rel"], rtol=5e-3)
    # observed: every code equal to the reference's, and every rounded
    # (bf16 / f16) scale and bias; held to that
    assert torch.equal(q.cpu(), t[f"{name}.q"])
    if s.dtype != torch.float32:
        assert torch.equal(s.cpu(), t[f"{name}.scales"]) and torch.equal(b.cpu(), t[f"{name}.biases"])


@pytest.mark.parametrize("bits,G,clip,storage,block", [
    (4, 64, "mse", torch.bfloat16, 128),
    (3, 32, "mse", torch.float16, 128),
    (4, 128, "mse", torch.bfloat16, 128),
    (8, 64, "minmax", torch.bfloat16, 128),
    (4, 64, "mse", torch.bfloat16, 100),   # bs = 64 (block trimmed to a group multiple)
    (4, 32, "mse", torch.bfloat16, 512),
])
def test_affine_matches_oracle(bits, G, clip, storage, block):
    from mlx_gptq import gptq

    W, H, _ = _setup(B=2, R=96, C=384, N=2048, seed=7, scale=0.02, outliers=4)
    H[1, 50, :] = 0.0
    H[1, :, 50] = 0.0  # a dead column in one item
    Wg, Hg = W.clone().to(DEV), H.clone().to(DEV)
    q, s, b, W_dq, rel = gptq.gptq_quantize(Wg, Hg, bits, G, clip=clip, storage_dtype=storage,
                                           block_size=block)
    assert W_dq.data_ptr() == Wg.data_ptr() and rel is None
    Wr, Hr = W.clone(), H.clone()
    rq, rs, rb, rW, _ = gptq_ref.gptq_quantize(Wr, Hr, bits, G, clip=clip, storage_dtype=storage,
                                               block_size=block)
    assert torch.equal(Hg.cpu(), Hr)
    assert int(q.max()) <= 2**bits - 1
    _check_vs(W, q, s, b, W_dq, rq, rs, rb, rW, Hr)


@pytest.mark.parametrize("case,w_mult,h_mult", [
    ("tiny_H", 1.0, 1e-20),    # U's diagonal above 2^24: no RN(1/d), every error division exact-path
    ("tiny_W", 1e-31, 1.0),    # numerators below 2^-100: the error divisions leave the fast range
    ("huge_W", 1e31, 1.0),     # numerators above 2^101
])
def test_affine_out_of_range_operands_vs_oracle(case, w_mult, h_mult):
    """The column loop divides with Markstein's correction and only records
    operands outside its exact range; a group that met any is solved again
    with the guarded division. These inputs put (almost) every group on that
    second path; the codes, params and W_dq must still be the oracle's."""
    from mlx_gptq import gptq

    W, H, _ = _setup(B=2, R=64, C=256, N=1024, seed=11, scale=0.02, outliers=2)
    W = W * w_mult
    H = H * h_mult
    Wg, Hg = W.clone().to(DEV), H.clone().to(DEV)
    q, s, b, W_dq, _ = gptq.gptq_quantize(Wg, Hg, 4, 64, storage_dtype=torch.float32)
    Wr, Hr = W.clone(), H.clone()
    rq, rs, rb, rW, _ = gptq_ref.gptq_quantize(Wr, Hr, 4, 64, storage_dtype=torch.float32)
    assert torch.isfinite(W_dq).all()
    _check_vs(W, q, s, b, W_dq, rq, rs, rb, rW, Hr)


def test_affine_nonfinite_weights_leave_other_rows_on_the_oracle():
    """NaN and inf weights: a row's errors only reach that row's later
    columns, so every other row must still match the oracle. The column loop
    sends a group whose chain met a NaN or an infinity to its exact pass, and
    the clip search's ranges must not be thrown off for the rest."""
    from mlx_gptq import grid, gptq

    W, H, _ = _setup(B=2, R=64, C=256, N=1024, seed=13, scale=0.02)
    W[0, 3, 70] = float("nan")
    W[1, 10, 5] = float("inf")
    W[1, 11, 127] = -float("inf")
    W[0, 50, 200:210] = float("nan")
    Wg, Hg = W.clone().to(DEV), H.clone().to(DEV)
    q, s, b, W_dq, _ = gptq.gptq_quantize(Wg, Hg, 4, 64, storage_dtype=torch.float32)
    Wr, Hr = W.clone(), H.clone()
    rq, rs, rb, rW, _ = gptq_ref.gptq_quantize(Wr, Hr, 4, 64, storage_dtype=torch.float32)
    good = torch.isfinite(W).all(dim=-1)  # [B, R]
    assert int((~good).sum()) == 4
    q, s, b, W_dq = q.cpu(), s.cpu(), b.cpu(), W_dq.cpu()
    assert int(q.max()) <= 15
    assert _agree(q[good], rq[good]) >= 0.995
    assert torch.allclose(s[good], rs[good], rtol=1e-4, atol=0)
    assert torch.allclose(b[good], rb[good], rtol=1e-4, atol=1e-7)
    dec = grid.dequantize_artifact(q, s, b, "affine", 64)
    assert torch.equal(dec[good], W_dq[good])
    for i in range(2):
        rows = good[i]
        pl = gptq_ref.proxy_loss(W[i, rows][None], W_dq[i, rows][None], Hr[i][None])
        pl_ref = gptq_ref.proxy_loss(W[i, rows][None], rW[i, rows][None], Hr[i][None])
        assert torch.isfinite(pl).all() and (pl - pl_ref).abs() <= 0.01 * pl_ref.abs()


def test_affine_config1_shape_vs_oracle():
    """BASELINE config 1 (single Linear 2048x2048, affine 4-bit, G=64, block
    128, MSE clip) at its real size, on 8192 lognormal tokens with 1% x20
    outlier channels."""
    from mlx_gptq import gptq

    g = torch.Generator().manual_seed(17)
    C = 2048
    X = torch.randn(8192, C, generator=g) * torch.exp(torch.randn(C, generator=g))
    X[:, torch.randperm(C, generator=g)[:20]] *= 20.0
    W = (torch.randn(1, C, C, generator=g) * 0.02).to(torch.bfloat16)
    H = (X.T @ X).unsqueeze(0).contiguous()
    q, s, b, W_dq, rel = gptq.solve_gptq(W.to(DEV), H.clone().to(DEV), 4, 64)
    rq, rs, rb, rW, rrel = gptq_ref.solve_gptq(W, H.clone(), 4, 64)
    _check_vs(W.float(), q, s, b, W_dq, rq, rs, rb, rW, H)
    assert torch.allclose(rel.cpu(), rrel, rtol=1e-2)


def test_affine_config1_chain_full_size():
    """Config 1 end to end as the bench runs it: the bf16 calibration rows in
    a capture.Stash, H from Stash.hessian (the GPU SYRK), the affine solve on
    the device; against the oracle's stash Hessian of the same rows (fp32
    addmm, capture.py:68-76) and the oracle's solve."""
    from mlx_gptq import capture, gptq, synth

    L = synth.dense_config(1, device=DEV)
    X, W = L.inputs["x"], L.mats[0].W
    C = X.shape[1]
    st = capture.Stash("x", C)
    st.add(X)
    H = st.hessian(torch.device(DEV)).unsqueeze(0)
    Xc = X.cpu()
    assert hessian_ref.rel_frobenius(H[0].cpu(), hessian_ref.hessian_fp64(Xc)) < 1e-5
    q, s, b, W_dq, rel = gptq.solve_gptq(W, H.clone(), **L.mats[0].solve)
    Hr = hessian_ref.stash_hessian([Xc], C).unsqueeze(0)
    rq, rs, rb, rW, rrel = gptq_ref.solve_gptq(W.cpu(), Hr.clone(), 4, 64)
    _check_vs(W.float().cpu(), q, s, b, W_dq, rq, rs, rb, rW, Hr)
    assert torch.allclose(rel.cpu(), rrel, rtol=1e-2)


@pytest.mark.parametrize("C", [320, 200])  # 5 diagonal 64-blocks; 3 and a ragged 8-row block
def test_prepare_hinv_full_vs_fp64(C):
    from mlx_gptq import gptq

    g = torch.Generator().manual_seed(3)
    B = 3
    A = torch.randn(B, C, 2 * C, generator=g) * torch.exp(torch.randn(B, C, 1, generator=g))
    H = A @ A.transpose(1, 2)
    U = gptq._prepare_hinv(H.to(DEV), 0.01).cpu()
    assert torch.equal(U, U.triu()) and bool((U.diagonal(dim1=-2, dim2=-1) > 0).all())
    dmean = H.diagonal(dim1=-2, dim2=-1).mean(-1).clamp(min=1e-8)
    Hd = H.clone()
    Hd.diagonal(dim1=-2, dim2=-1).add_((dmean * 0.01).unsqueeze(-1))
    U64 = torch.linalg.cholesky(torch.cholesky_inverse(torch.linalg.cholesky(Hd.double())),
                                upper=True)
    rel = (U.double() - U64).norm(dim=(1, 2)) / U64.norm(dim=(1, 2))
    assert float(rel.max()) < 1e-5, rel
    Ur = gptq_ref.prepare_hinv(H.clone(), 0.01)
    rel_ref = (Ur.double() - U64).norm(dim=(1, 2)) / U64.norm(dim=(1, 2))
    assert float(rel.max()) <= float(rel_ref.max()) + 1e-6


@pytest.mark.parametrize("B,C", [(1, 1), (2, 33), (3, 65), (2, 333), (1, 1025), (20, 640)])
def test_prepare_hinv_full_tiles(B, C):
    """Ragged and odd sizes (rows that are not 16-byte aligned in H, a last
    block of 1 to 63 columns, K ends inside a chunk) and both tile sizes (20
    items of 640 take 64 x 64 tiles at the top node, one item 32 x 32): U
    against the float64 factor of the same damped matrix, within a few fp32
    roundings (2^-24 each, the entries' own), and the same bits for an item
    whether it is factored alone or in the batch."""
    from mlx_gptq import gptq

    g = torch.Generator().manual_seed(C)
    A = torch.randn(B, C, C + 8, generator=g) * torch.exp(torch.randn(B, C, 1, generator=g))
    H = A @ A.transpose(1, 2)
    U = gptq._prepare_hinv(H.to(DEV), 0.01).cpu()
    assert torch.equal(U, U.triu())
    # the damped matrix as the solver forms it: lam and the sum rounded to fp32
    lam = H.double().diagonal(dim1=-2, dim2=-1).mean(-1).float() * torch.tensor(0.01)
    for b in {0, B - 1}:
        Hd = H[b].tril()
        Hd = (Hd + Hd.tril(-1).T).double()
        Hd.diagonal().copy_((H[b].diagonal() + lam[b]).double())
        want = torch.linalg.cholesky(torch.linalg.inv(Hd), upper=True)
        rel = float((U[b].double() - want).norm() / want.norm())
        assert rel < 4 * 2.0 ** -24, (b, rel)
        if B > 1:
            one = gptq._prepare_hinv(H[b : b + 1].to(DEV), 0.01).cpu()
            assert torch.equal(one[0], U[b])


@pytest.mark.parametrize("C", [1100, 2112])
def test_prepare_hinv_full_does_not_depend_on_the_batch(C):
    """Up to five items deal their tiles out one by one, more by contiguous
    parts: every tile is formed once either way, with the same bits."""
    from mlx_gptq import gptq

    g = torch.Generator(device=DEV).manual_seed(C)
    X = torch.randn(C + 64, C, generator=g, device=DEV)
    H = X.T @ X
    one = gptq._prepare_hinv(H[None].clone(), 0.01)
    assert torch.isfinite(one).all()
    for B in (2, 4, 5, 6, 7, 9):
        U = gptq._prepare_hinv(H[None].repeat(B, 1, 1), 0.01)
        assert torch.equal(U, one.expand(B, C, C)), B


@pytest.mark.parametrize("C", [2, 15, 16, 17, 31, 47, 48, 49, 63, 64])
def test_prepare_hinv_full_leaf_blocks(C):
    """One 64-leaf with its 16 x 16 blocks whole, cut and missing: U against the
    float64 factor within a few fp32 roundings (2^-24 each, the entries' own),
    and a negative pivot found in whichever block holds it."""
    from mlx_gptq import gptq_affine

    g = torch.Generator().manual_seed(C)
    A = torch.randn(1, C, C + 8, generator=g) * torch.exp(torch.randn(1, C, 1, generator=g))
    H = A @ A.transpose(1, 2)
    bad = sorted({0, C // 2, C - 1})
    Hs = H.repeat(1 + len(bad), 1, 1)
    for n, c in enumerate(bad):
        Hs[1 + n, c, c] = -H.diagonal(dim1=-2, dim2=-1).sum()
    U, attempts = gptq_affine.prepare_hinv_full(Hs.to(DEV), 0.01, 1)
    assert list(attempts) == [1] + [0] * len(bad)
    lam = H[0].double().diagonal().mean().float() * torch.tensor(0.01)
    Hd = H[0].tril()
    Hd = (Hd + Hd.tril(-1).T).double()
    Hd.diagonal().copy_((H[0].diagonal() + lam).double())
    want = torch.linalg.cholesky(torch.linalg.inv(Hd), upper=True)
    assert float((U[0].cpu().double() - want).norm() / want.norm()) < 4 * 2.0 ** -24


def _indefinite(B, C, neg):
    """Diagonal-dominant SPD items with item i's diagonal entry 5 set to
    neg[i]: the damped matrix needs damp >= -neg / mean(diag) to factor."""
    g = torch.Generator().manual_seed(23)
    H = torch.zeros(B, C, C)
    for i in range(B):
        A = torch.randn(C, C, generator=g) * 0.01
        H[i] = A @ A.T + torch.eye(C)
        if neg[i] is not None:
            H[i, 5, :] = 0.0
            H[i, :, 5] = 0.0
            H[i, 5, 5] = neg[i]
    return H


def test_full_escalation_warnings_match_oracle(caplog):
    from mlx_gptq import gptq

    C = 96
    H = _indefinite(3, C, [None, -0.05, -2.0])  # needs damp 0.1 and 10
    with caplog.at_level(logging.WARNING, logger="oracle.gptq_ref"):
        events = []
        Ur = gptq_ref.prepare_hinv(H.clone(), 0.01, events=events)
    ref_msgs = [r.getMessage() for r in caplog.records]
    assert len(ref_msgs) >= 2
    caplog.clear()
    with caplog.at_level(logging.WARNING, logger="mlx_gptq.gptq"):
        U = gptq._prepare_hinv(H.to(DEV), 0.01).cpu()
    assert [r.getMessage() for r in caplog.records] == ref_msgs
    rel = (U - Ur).norm() / Ur.norm()
    assert float(rel) < 1e-4

    Hf = _indefinite(4, C, [None, -1e6, -0.05, None])  # item 1 never factors
    caplog.clear()
    with caplog.at_level(logging.WARNING, logger="oracle.gptq_ref"):
        with pytest.raises(RuntimeError) as ei_ref:
            gptq_ref.prepare_hinv(Hf.clone(), 0.01)
    ref_msgs = [r.getMessage() for r in caplog.records]
    caplog.clear()
    with caplog.at_level(logging.WARNING, logger="mlx_gptq.gptq"):
        with pytest.raises(RuntimeError) as ei:
            gptq._prepare_hinv(Hf.to(DEV), 0.01)
    assert str(ei.value) == str(ei_ref.value)
    assert [r.getMessage() for r in caplog.records] == ref_msgs


def test_solve_falls_back_when_the_first_damped_pass_fails(caplog):
    """solve_gptq launches the affine column loop before it knows the first
    damped pass succeeded. When an item needs more damping, it must solve
    again on the synchronous path: the outputs are those of gptq_quantize on
    a copy of W, with the reference's warnings; an item that never factors
    raises the reference's RuntimeError."""
    from mlx_gptq import gptq

    def coupled(B, C, off):
        # SPD items with a positive diagonal (so the dead-column fix keeps
        # them) and entries (5, 6), (6, 5) set to off[i]: the 2x2 block
        # [[1, o], [o, 1]] needs a damping above o - 1 to factor
        gg = torch.Generator().manual_seed(23)
        Hc = torch.zeros(B, C, C)
        for i in range(B):
            A = torch.randn(C, C, generator=gg) * 0.01
            Hc[i] = A @ A.T + torch.eye(C)
            if off[i] is not None:
                Hc[i, 5, 6] = Hc[i, 6, 5] = off[i]
        return Hc

    C = 128
    H = coupled(3, C, [None, 1.05, 3.0])  # needs damp 0.1 and 10
    g = torch.Generator().manual_seed(31)
    W = torch.randn(3, 48, C, generator=g) * 0.02
    with caplog.at_level(logging.WARNING, logger="mlx_gptq.gptq"):
        q, s, b, W_dq, rel = gptq.solve_gptq(W.to(DEV), H.clone().to(DEV), 4, 64)
    msgs = [r.getMessage() for r in caplog.records]
    caplog.clear()
    with caplog.at_level(logging.WARNING, logger="mlx_gptq.gptq"):
        Wc = W.clone().to(DEV)
        q2, s2, b2, W2, _ = gptq.gptq_quantize(Wc, H.clone().to(DEV), 4, 64)
    assert msgs == [r.getMessage() for r in caplog.records] and len(msgs) >= 2
    assert torch.equal(q, q2) and torch.equal(s, s2) and torch.equal(b, b2)
    assert torch.equal(W_dq, W2)
    assert torch.isfinite(rel).all()

    Hf = coupled(3, C, [None, 1e6, None])  # item 1 never factors
    caplog.clear()
    with caplog.at_level(logging.WARNING, logger="oracle.gptq_ref"):
        with pytest.raises(RuntimeError) as ei_ref:
            gptq_ref.prepare_hinv(Hf.clone(), 0.01)
    ref_msgs = [r.getMessage() for r in caplog.records]
    caplog.clear()
    with caplog.at_level(logging.WARNING, logger="mlx_gptq.gptq"):
        with pytest.raises(RuntimeError) as ei:
            gptq.solve_gptq(W.to(DEV), Hf.clone().to(DEV), 4, 64)
    assert str(ei.value) == str(ei_ref.value)
    assert [r.getMessage() for r in caplog.records] == ref_msgs


def test_solve_fallback_keeps_dead_columns_zeroed(caplog):
    """A batch where one item has dead columns (diag 0 and < 0) and another
    needs damp 0.1: the speculative first pass fails, and the synchronous
    retry must still zero the dead columns of its fresh copy of W, as the
    reference's gptq_quantize does (gptq.py:216-222) before it escalates.
    Checked against the oracle's solve_gptq on the same inputs."""
    from mlx_gptq import gptq

    C, R = 128, 48
    gg = torch.Generator().manual_seed(41)
    H = torch.zeros(3, C, C)
    for i in range(3):
        A = torch.randn(C, C, generator=gg) * 0.01
        H[i] = A @ A.T + torch.eye(C)
    H[1, 5, 6] = H[1, 6, 5] = 1.05  # needs damp 0.1 to factor
    for c, v in ((17, 0.0), (90, -2.0)):  # dead columns of item 0
        H[0, c, :] = 0.0
        H[0, :, c] = 0.0
        H[0, c, c] = v
    W = torch.randn(3, R, C, generator=gg) * 0.02
    rq, rs, rb, rW, rrel = gptq_ref.solve_gptq(W.clone(), H.clone(), 4, 64)
    Hd = H.clone().to(DEV)
    with caplog.at_level(logging.WARNING, logger="mlx_gptq.gptq"):
        q, s, b, W_dq, rel = gptq.solve_gptq(W.to(DEV), Hd, 4, 64)
    assert len(caplog.records) >= 1  # the escalation did run
    # the dead columns hold w = 0 before quantization, as in the oracle
    assert _agree(q[0, :, [17, 90]], rq[0, :, [17, 90]]) >= 0.98
    assert _agree(q[0], rq[0]) >= 0.995
    H_after = H.clone()
    H_after[0, 17, 17] = H_after[0, 90, 90] = 1.0
    assert torch.equal(Hd.cpu(), H_after)  # the dead-column fix in place, once
    _check_vs(W, q, s, b, W_dq, rq, rs, rb, rW, H_after)
    assert torch.allclose(rel.cpu(), rrel, rtol=1e-3, atol=0)


def test_affine_batched_equals_per_item():
    """Reference tests/test_gptq.py:44-52 (bit-exact), affine mode."""
    from mlx_gptq import gptq

    W, H, _ = _setup(B=3, R=40, C=256)
    qb, sb, bb, wb, _ = gptq.solve_gptq(W.to(DEV), H.clone().to(DEV), 4, 64)
    for i in range(3):
        qi, si, bi, wi, _ = gptq.solve_gptq(W[i : i + 1].to(DEV), H[i : i + 1].clone().to(DEV), 4, 64)
        assert torch.equal(qb[i], qi[0]) and torch.equal(sb[i], si[0])
        assert torch.equal(bb[i], bi[0]) and torch.equal(wb[i], wi[0])


def test_affine_gptq_improves_activation_error():
    """Reference tests/test_gptq.py:19-26."""
    from mlx_gptq import grid, gptq

    W, H, X = _setup(B=1, R=64, C=256, N=2048, seed=11)
    _, _, _, W_g, _ = gptq.solve_gptq(W.to(DEV), H.to(DEV), 4, 64)
    _, _, _, W_r = grid.rtn_quantize(W.to(DEV), 4, 64)
    e_g = ((X @ (W_g.cpu() - W).transpose(1, 2)) ** 2).mean()
    e_r = ((X @ (W_r.cpu() - W).transpose(1, 2)) ** 2).mean()
    assert e_g < e_r


def test_affine_zero_hessian_finite():
    """Reference tests/test_gptq.py:55-60."""
    from mlx_gptq import gptq

    W = torch.randn(1, 8, 128)
    H = torch.zeros(1, 128, 128)
    q, s, b, W_dq, rel = gptq.solve_gptq(W.to(DEV), H.to(DEV), 4, 64)
    assert torch.isfinite(W_dq).all()
    assert torch.count_nonzero(W_dq) == 0


def test_affine_shape_errors():
    from mlx_gptq import gptq

    W = torch.zeros(1, 4, 96, device=DEV)
    H = torch.eye(96, device=DEV).unsqueeze(0)
    with pytest.raises(AssertionError):
        gptq.gptq_quantize(W, H.clone(), 4, 64)
    with pytest.raises(AssertionError):
        gptq.gptq_quantize(W, torch.eye(64, device=DEV).unsqueeze(0), 4, 32)


@pytest.mark.parametrize("dt", [torch.float32, torch.bfloat16, torch.float16, torch.float64])
def test_rel_err_kernel_matches_the_reference_formula(dt):
    """gptq_affine.rel_err (mgq_rel_err: double partial sums, fixed order)
    against gptq.py:300-302's formula evaluated in float64 on the host; an
    all-zero original takes the 1e-12 floor of the denominator; B = 3,
    ragged n."""
    from mlx_gptq import gptq_affine

    g = torch.Generator().manual_seed(31)
    W = (torch.randn(3, 37, 1001, generator=g) * 0.02).to(dt)
    W[2] = 0
    Wdq = W.float() + torch.randn(3, 37, 1001, generator=g) * 1e-3
    got = gptq_affine.rel_err(Wdq.to(DEV), W.to(DEV)).cpu()
    W64, D64 = W.double(), Wdq.double()
    want = (D64 - W64).flatten(1).norm(dim=1) / W64.flatten(1).norm(dim=1).clamp(min=1e-12)
    assert got.dtype == torch.float32
    assert torch.allclose(got.double(), want, rtol=1e-6, atol=0)
    assert want[2] > 1e10  # the floor case


@pytest.mark.parametrize("parts", [1, 65, 1025, 8192, 20011])
def test_rel_err_any_number_of_partials(parts):
    """One partial a thread, some threads without one, more than one round of
    the final sum: the fp64 ratio to an fp32 square root and division."""
    from mlx_gptq import _native as nat

    B, n = 3, 40000
    g = torch.Generator().manual_seed(parts)
    W = torch.randn(B, n, generator=g)
    Wdq = W + 0.1 * torch.randn(B, n, generator=g)
    Wd, Wqd = W.to(DEV), Wdq.to(DEV)
    part = torch.full((B, parts, 2), float("nan"), dtype=torch.float64, device=DEV)
    rel = torch.empty(B, dtype=torch.float32, device=DEV)
    nat.call("mgq_rel_err", Wqd.data_ptr(), Wd.data_ptr(), nat.dtype_code(W.dtype), B, n,
             part.data_ptr(), parts, rel.data_ptr(), nat.stream_of(DEV))
    want = (Wdq - W).double().norm(dim=1) / W.double().norm(dim=1)
    assert ((rel.cpu().double() - want).abs() <= 4 * 2.0 ** -24 * want).all()


@pytest.mark.parametrize("G", [32, 64, 128])
def test_affine_rows_do_not_depend_on_how_many_are_solved(G):
    """The column loop takes its variant (shares of the clip candidates, a
    DPP row or a quad of lanes per row, workgroup size) from the number of
    rows. A row's result depends on nothing but the row and U, so 37 rows
    repeated 1 (four shares), 28 (two), 111 (one) and 2680 times (a quad per
    row; a ragged last workgroup) give the same bits in every repetition."""
    from mlx_gptq import gptq

    W, H, _ = _setup(B=1, R=37, C=128, N=512, seed=17 + G, scale=0.02)
    W[0, 5, 3:60] = 0.0
    W[0, 6] *= 1e-34  # leaves the fast divisions' range
    want = gptq.gptq_quantize(W.to(DEV), H.clone().to(DEV), 4, G)
    for times in (28, 111, 2680):
        got = gptq.gptq_quantize(W.repeat(1, times, 1).to(DEV), H.clone().to(DEV), 4, G)
        for x, y in zip(want[:4], got[:4]):
            assert torch.equal(y.view(times, 37, -1), x.expand(times, -1, -1)), times


@pytest.mark.parametrize("G,C", [(48, 240), (20, 200), (96, 192), (16, 80), (8, 40)])
def test_affine_other_group_sizes_match_oracle(G, C):
    """Group sizes that do not fill the lanes' slots."""
    from mlx_gptq import gptq

    W, H, _ = _setup(B=2, R=45, C=C, N=1024, seed=G, scale=0.02, outliers=2)
    rW, rH = W.clone(), H.clone()
    q, s, b, W_dq, _ = gptq.gptq_quantize(W.clone().to(DEV), H.clone().to(DEV), 4, G)
    rq, rs, rb, rW, _ = gptq_ref.gptq_quantize(rW, rH, 4, G)
    _check_vs(W, q, s, b, W_dq, rq, rs, rb, rW, rH)


@pytest.mark.parametrize("B,R,C,block,G", [
    (2, 70, 1216, 128, 64),   # two spans of four blocks and a ragged third
    (1, 200, 640, 256, 64),   # spans of two blocks
    (1, 45, 360, 120, 24),    # a last chunk of 24 k per block
    (3, 33, 1000, 40, 8),     # spans of twelve short blocks
    (1, 65, 660, 66, 66),     # n not a multiple of 8: a launch per block
])
def test_affine_deferred_updates_equal_one_update_per_block(B, R, C, block, G):
    """mgq_gptq_affine updates the columns past a span of blocks once for all
    of them; the bits are those of mgq_gptq_affine_block block by block, for
    every number of blocks that Err has room for."""
    from mlx_gptq import _native as nat

    g = torch.Generator().manual_seed(C)
    W0 = torch.randn(B, R, C, generator=g) * 0.02
    U = (torch.randn(B, C, C, generator=g).triu(1) * 0.05
         + torch.diag_embed(torch.rand(B, C, generator=g) + 0.5)).to(DEV)
    stream = nat.stream_of(torch.device(DEV))

    def buffers(err_cols):
        return (W0.to(DEV), torch.zeros(B, R, C, dtype=torch.uint8, device=DEV),
                torch.zeros(B, R, C // G, device=DEV), torch.zeros(B, R, C // G, device=DEV),
                torch.zeros(B, R, err_cols, device=DEV))

    ref = buffers(block)
    W, q, s, b, err = ref
    for i1 in range(0, C, block):
        n = min(block, C - i1)
        nat.call("mgq_gptq_affine_block", W.data_ptr(), U.data_ptr(), B, R, C, i1, n, G, 4, 1, 0,
                 20, 0.2, q.data_ptr(), s.data_ptr(), b.data_ptr(), err.data_ptr(), stream)
    for err_cols in (block, 2 * block + 4, max(block, 512 // block * block)):
        got = buffers(err_cols)
        W, q, s, b, err = got
        nat.call("mgq_gptq_affine", W.data_ptr(), U.data_ptr(), B, R, C, block, G, 4, 1, 0, 20, 0.2,
                 q.data_ptr(), s.data_ptr(), b.data_ptr(), err.data_ptr(), err_cols, stream)
        for x, y in zip(ref[:4], got[:4]):
            assert torch.equal(x, y), err_cols
    with pytest.raises(RuntimeError):
        nat.call("mgq_gptq_affine", W.data_ptr(), U.data_ptr(), B, R, C, block, G, 4, 1, 0, 20, 0.2,
                 q.data_ptr(), s.data_ptr(), b.data_ptr(), err.data_ptr(), block - 1, stream)


def test_affine_block_unaligned_factor_gives_the_same_bits():
    """U off its 16-byte alignment takes 4-byte loads instead of 16-byte ones."""
    from mlx_gptq import _native as nat

    g = torch.Generator().manual_seed(3)
    R, C = 21, 256
    W0 = torch.randn(1, R, C, generator=g) * 0.02
    U0 = torch.randn(C, C, generator=g).triu(1) * 0.05 + torch.diag(torch.rand(C, generator=g) + 0.5)
    out = []
    for shift in (0, 1):
        flat = torch.zeros(C * C + shift, device=DEV)
        flat[shift:] = U0.flatten().to(DEV)
        W, U = W0.to(DEV), flat[shift:]
        q = torch.zeros(1, R, C, dtype=torch.uint8, device=DEV)
        s, b = torch.zeros(2, 1, R, C // 64, device=DEV)
        err = torch.zeros(1, R, 128, device=DEV)
        nat.call("mgq_gptq_affine_block", W.data_ptr(), U.data_ptr(), 1, R, C, 0, 128, 64, 4, 1, 0,
                 20, 0.2, q.data_ptr(), s.data_ptr(), b.data_ptr(), err.data_ptr(),
                 nat.stream_of(torch.device(DEV)))
        out.append((W, q, s, b, err))
    for x, y in zip(*out):
        assert torch.equal(x, y)


@pytest.mark.parametrize("u_shift,err_shift", [(1, 0), (0, 1), (3, 2)])
def test_affine_loop_takes_u_and_err_at_any_address(u_shift, err_shift):
    """U and Err moved off their 16-byte alignment, together and alone: the
    general deferred update instead of the piecewise one, a launch per block
    instead of one per span, the same bits."""
    from mlx_gptq import _native as nat

    g = torch.Generator().manual_seed(5)
    R, C, G, cols = 70, 640, 64, 512
    W0 = torch.randn(1, R, C, generator=g) * 0.02
    U0 = torch.randn(C, C, generator=g).triu(1) * 0.05 + torch.diag(torch.rand(C, generator=g) + 0.5)
    out = []
    for us, es in ((0, 0), (u_shift, err_shift)):
        u = torch.zeros(C * C + us, device=DEV)
        u[us:] = U0.flatten().to(DEV)
        err = torch.zeros(R * cols + es, device=DEV)
        W = W0.to(DEV)
        q = torch.zeros(1, R, C, dtype=torch.uint8, device=DEV)
        s, b = torch.zeros(2, 1, R, C // G, device=DEV)
        nat.call("mgq_gptq_affine", W.data_ptr(), u[us:].data_ptr(), 1, R, C, 128, G, 4, 1, 0, 20,
                 0.2, q.data_ptr(), s.data_ptr(), b.data_ptr(), err[es:].data_ptr(), cols,
                 nat.stream_of(torch.device(DEV)))
        out.append((W, q, s, b))
    for x, y in zip(*out):
        assert torch.equal(x, y)


def test_rel_err_partials_at_any_double():
    """The partials' buffer is aligned to one double only."""
    from mlx_gptq import _native as nat

    B, n, parts = 2, 5000, 37
    g = torch.Generator().manual_seed(2)
    W = torch.randn(B, n, generator=g).to(DEV)
    Wdq = W + 0.1 * torch.randn(B, n, generator=g).to(DEV)
    part = torch.zeros(2 * B * parts + 1, dtype=torch.float64, device=DEV)
    rel = torch.empty(2, B, dtype=torch.float32, device=DEV)
    for o in (0, 1):
        nat.call("mgq_rel_err", Wdq.data_ptr(), W.data_ptr(), nat.dtype_code(W.dtype), B, n,
                 part[o:].data_ptr(), parts, rel[o].data_ptr(), nat.stream_of(DEV))
    assert torch.equal(rel[0], rel[1])


@pytest.mark.parametrize("G,C,block", [(4, 136, 128), (7, 140, 128), (24, 264, 128), (40, 240, 128),
                                       (48, 528, 256), (62, 186, 128), (77, 231, 128), (112, 224, 128)])
@pytest.mark.parametrize("clip", ["mse", "minmax"])
def test_affine_other_group_sizes_few_rows_and_many(G, C, block, clip):
    """Few rows take a wave each, many 16 lanes each; a row's result is the same
    bits either way: blocks whose part of U is in LDS and larger ones, odd row
    lengths, one and two columns a lane, rows that leave the fast divisions' range."""
    from mlx_gptq import gptq

    W, H, _ = _setup(B=1, R=37, C=C, N=2 * C + 64, seed=G, scale=0.02)
    W[0, 5, 3:60] = 0.0
    W[0, 6] *= 1e-34
    W[0, 7, 2] = float("inf")
    want = gptq.gptq_quantize(W.to(DEV), H.clone().to(DEV), 4, G, clip=clip, block_size=block)
    times = 120 if G >= 8 and block <= 128 else 240
    got = gptq.gptq_quantize(W.repeat(1, times, 1).to(DEV), H.clone().to(DEV), 4, G, clip=clip,
                             block_size=block)
    for x, y in zip(want[:4], got[:4]):
        x = x.expand(times, -1, -1)
        y = y.view(x.shape)
        assert torch.equal(x.isnan(), y.isnan())
        assert torch.equal(x.nan_to_num(7.0), y.nan_to_num(7.0))


@pytest.mark.parametrize("B,R,C", [(1, 1, 1), (1, 37, 300), (1, 2049, 64), (3, 1100, 520),
                                   (40, 65, 700), (65537, 1, 2)])
def test_dead_fix_any_split_of_the_rows(B, R, C):
    """Columns with a diagonal <= 0 (-0 and negative too) are zeroed in every
    row, however the rows are split; a NaN diagonal is not dead."""
    from mlx_gptq import _native as nat

    g = torch.Generator().manual_seed(R)
    d = torch.tensor([1.0, 0.0, -0.0, -2.0, float("nan"), 3.0])[
        torch.randint(0, 6, (B, C), generator=g)].to(DEV)
    W = torch.randn(B, R, C, generator=g).to(DEV)
    H = torch.full((B, C, C), 0.5, device=DEV)
    H.diagonal(dim1=-2, dim2=-1).copy_(d)
    dead = d <= 0
    want = W.masked_fill(dead.unsqueeze(1), 0.0)
    nat.call("mgq_dead_fix", W.data_ptr(), B, R, C, H.data_ptr(), nat.stream_of(torch.device(DEV)))
    assert torch.equal(W, want)
    after = H.diagonal(dim1=-2, dim2=-1)
    assert torch.equal(after.nan_to_num(7.0), torch.where(dead, 1.0, d).nan_to_num(7.0))


@pytest.mark.parametrize("G", [48, 64])
@pytest.mark.parametrize("steps", [1, 63, 64, 127])
def test_clip_search_of_the_loop_takes_as_many_steps_as_choose_qparams(G, steps):
    """The first group's scales and biases are choose_qparams' of the weights as
    they are: one batch of 64 candidates, a second one, the largest number."""
    from mlx_gptq import _native as nat
    from mlx_gptq import grid

    g = torch.Generator().manual_seed(steps)
    R = 300
    W = (torch.randn(1, R, G, generator=g) * 0.02).to(DEV)
    _, _, rs, rb = grid.choose_qparams(W, 4, "mse", torch.float32, steps, 0.5)
    U = torch.eye(G, device=DEV)
    q = torch.zeros(1, R, G, dtype=torch.uint8, device=DEV)
    s, b = torch.zeros(2, 1, R, 1, device=DEV)
    err = torch.zeros(1, R, G, device=DEV)
    nat.call("mgq_gptq_affine_block", W.data_ptr(), U.data_ptr(), 1, R, G, 0, G, G, 4, 1, 0, steps, 0.5,
             q.data_ptr(), s.data_ptr(), b.data_ptr(), err.data_ptr(),
             nat.stream_of(torch.device(DEV)))
    # the error sums add in another order: a tie may go the other way
    assert int(((s[..., 0] != rs) | (b[..., 0] != rb)).sum()) <= R // 100


@pytest.mark.parametrize("parts", [255, 256, 257])
def test_rel_err_both_workgroup_sizes(parts):
    """256 threads up to 256 partials, 1024 above, many items: the fp64 ratio to
    an fp32 square root and division."""
    from mlx_gptq import _native as nat

    B, n = 300, 3000
    g = torch.Generator().manual_seed(parts)
    W = torch.randn(B, n, generator=g)
    Wdq = W + 0.1 * torch.randn(B, n, generator=g)
    part = torch.full((B, parts, 2), float("nan"), dtype=torch.float64, device=DEV)
    rel = torch.empty(B, dtype=torch.float32, device=DEV)
    Wd, Wqd = W.to(DEV), Wdq.to(DEV)
    nat.call("mgq_rel_err", Wqd.data_ptr(), Wd.data_ptr(), nat.dtype_code(W.dtype), B, n,
             part.data_ptr(), parts, rel.data_ptr(), nat.stream_of(DEV))
    want = (Wdq - W).double().norm(dim=1) / W.double().norm(dim=1)
    assert ((rel.cpu().double() - want).abs() <= 4 * 2.0 ** -24 * want).all()
