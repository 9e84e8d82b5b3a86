"""The Stage-A drop-in on the GPU:

* ``CaptureManager`` on a toy decoder layer (two ``nn.Linear`` sharing one
  input, and a transformers ``Qwen3MoeSparseMoeBlock``): every stash's
  ``hessian(device)`` -- the linears' and every expert's ``stashes[key]``
  view -- is within 1e-5 relative Frobenius of fp64 X^T X of the rows that
  module or expert slice actually received (recorded the way the reference
  records them, capture.py:160-207), with the same-input dedup of
  capture.py:167-178;
* ``solve_gptq`` / ``gptq_quantize`` on host tensors equal the on-device
  call bit for bit, with the in-place W and H (dead-column) updates landing
  in the caller's host tensors;
* ``span_solve.solve_fused_task`` over several spans agrees with the oracle
  (the reference algorithm restated on the CPU) expert by expert.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch
import torch.nn.functional as F
from torch.overrides import TorchFunctionMode

from mlx_gptq import capture, gptq, span_solve
from oracle import gptq_ref, hessian_ref

transformers = pytest.importorskip("transformers")
from transformers import Qwen3MoeConfig  # noqa: E402
from transformers.models.qwen3_moe.modeling_qwen3_moe import Qwen3MoeSparseMoeBlock  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda", 0)


class _Layer(torch.nn.Module):
    def __init__(self, hidden=256, inter=128, E=8, k=2):
        super().__init__()
        cfg = Qwen3MoeConfig(hidden_size=hidden, moe_intermediate_size=inter, num_experts=E,
                             num_experts_per_tok=k, norm_topk_prob=True)
        self.q_proj = torch.nn.Linear(hidden, hidden, bias=False)
        self.k_proj = torch.nn.Linear(hidden, hidden, bias=False)
        self.o_proj = torch.nn.Linear(hidden, hidden, bias=False)
        self.mlp = Qwen3MoeSparseMoeBlock(cfg)

    def forward(self, x):
        h = self.o_proj(self.q_proj(x) * torch.sigmoid(self.k_proj(x)))
        return x + self.mlp(h)


class _Recorder(TorchFunctionMode):
    """Inputs of every F.linear on an expert slice, keyed (param, expert)."""

    def __init__(self, experts):
        super().__init__()
        self.ptr = {}
        for pname, p in experts.named_parameters(recurse=False):
            for e in range(p.shape[0]):
                self.ptr[p.data_ptr() + e * p.stride(0) * p.element_size()] = (pname, e)
        self.rows = {}

    def __torch_function__(self, func, types, args=(), kwargs=None):
        kwargs = kwargs or {}
        if func is F.linear and len(args) >= 2 and isinstance(args[1], torch.Tensor):
            hit = self.ptr.get(args[1].data_ptr())
            if hit is not None:
                self.rows.setdefault(hit, []).append(args[0].detach().to(torch.bfloat16).cpu())
        return func(*args, **kwargs)


def _rel(a, ref) -> float:
    return hessian_ref.rel_frobenius(a.cpu(), ref)


def _capture(layer, batches, hidden):
    mgr = capture.CaptureManager(layer, r"o_proj", 32)
    rec = _Recorder(layer.mlp.experts)
    lin_rows = []
    hook = layer.q_proj.register_forward_pre_hook(
        lambda m, a: lin_rows.append(a[0].detach().reshape(-1, hidden).to(torch.bfloat16).cpu()))
    g = torch.Generator().manual_seed(11)
    with torch.no_grad(), mgr, rec:
        for shape in batches:
            mgr.begin_batch()
            layer(torch.randn(*shape, hidden, generator=g).to(DEV, torch.bfloat16))
    hook.remove()
    return mgr, rec, torch.cat(lin_rows)


def test_capture_manager_hessians_match_received_rows():
    hidden, inter, E = 256, 128, 8
    torch.manual_seed(0)
    layer = _Layer(hidden, inter, E).to(DEV, torch.bfloat16)
    for p in layer.mlp.parameters():
        torch.nn.init.normal_(p, std=0.1)
    mgr, rec, lin_rows = _capture(layer, [(2, 64), (1, 150), (3, 40)], hidden)
    # o_proj is excluded; q_proj and k_proj take one tensor: k_proj shares q_proj's stash
    assert [t.name for t in mgr.linear_tasks] == ["q_proj", "k_proj"]
    assert [t.stash_key for t in mgr.linear_tasks] == ["q_proj", "q_proj"]
    assert mgr.stashes["k_proj"].tokens == 0
    st = mgr.stashes["q_proj"]
    assert st.tokens == lin_rows.shape[0] == 2 * 64 + 150 + 3 * 40
    assert _rel(st.hessian(DEV), hessian_ref.hessian_fp64(lin_rows)) < 1e-5
    mgr.check_capture_happened()
    stats = mgr.expert_token_stats()
    for task in mgr.fused_tasks:
        C = task.param.shape[-1]
        counts = []
        for e, key in enumerate(task.stash_keys):
            parts = rec.rows.get((task.param_name, e), [])
            rows = torch.cat(parts) if parts else torch.zeros(0, C, dtype=torch.bfloat16)
            view = mgr.stashes[key]
            assert view.tokens == rows.shape[0], (key, view.tokens, rows.shape[0])
            counts.append(view.tokens)
            H = view.hessian(DEV)
            assert H.shape == (C, C) and H.device == DEV
            if rows.shape[0] == 0:
                assert bool((H == 0).all())
            else:
                assert _rel(H, hessian_ref.hessian_fp64(rows)) < 1e-5, key
        c = sorted(counts)
        assert stats[f"{task.module_name}.{task.param_name}"] == (c[0], c[len(c) // 2], c[-1],
                                                                   c.count(0))
        # the batched fast path equals the per-expert views
        Hs = mgr.expert_hessians(task, DEV, range(2, 6))
        for i, e in enumerate(range(2, 6)):
            assert torch.equal(Hs[i], mgr.stashes[task.stash_keys[e]].hessian(DEV))
    assert mgr.total_stash_bytes() > 0
    mgr.drop_all()
    assert mgr.total_stash_bytes() == 0


@pytest.mark.parametrize("mode,bits,G", [("mxfp4", 4, 32), ("mxfp8", 8, 32), ("affine", 4, 64)])
def test_host_tensors_solve_bit_exactly_like_device_tensors(mode, bits, G):
    g = torch.Generator().manual_seed(21)
    B, R, C = 2, 48, 256
    W = torch.randn(B, R, C, generator=g) * 0.02
    X = torch.randn(B, 600, C, generator=g) * torch.exp(torch.randn(C, generator=g))
    H = (X.transpose(1, 2) @ X).contiguous()
    H[:, 7, :] = 0.0
    H[:, :, 7] = 0.0  # a dead column: zeroed in W_dq, diagonal set to 1 in place
    out_d = gptq.solve_gptq(W.to(DEV), H.clone().to(DEV), bits, G, mode=mode)
    H_host = H.clone()
    out_h = gptq.solve_gptq(W, H_host, bits, G, mode=mode)
    for a, b in zip(out_h, out_d):
        if a is None:
            assert b is None
            continue
        assert a.device.type == "cpu"
        assert torch.equal(a, b.cpu())
    assert float(H_host[0, 7, 7]) == 1.0 and float(H_host[1, 7, 7]) == 1.0
    if mode != "affine":  # an affine zero dequantizes to q*s + b, not 0
        assert bool((out_h[3][:, :, 7] == 0).all())
    # gptq_quantize: W (host, fp32) becomes W_dq in place
    W_in = W.clone()
    q, s, b, W_dq, _ = gptq.gptq_quantize(W_in, H.clone(), bits, G, mode=mode)
    assert W_dq is W_in and torch.equal(W_in, out_d[3].cpu()) and torch.equal(q, out_d[0].cpu())


def _oracle_expert(W_e, rows, bits, mode):
    C = W_e.shape[-1]
    H = hessian_ref.stash_hessian([rows], C).unsqueeze(0)
    return gptq_ref.solve_gptq(W_e.unsqueeze(0).float(), H, bits, 32, mode=mode)


def test_span_solver_matches_the_oracle_per_expert():
    hidden, inter, E = 256, 128, 8
    torch.manual_seed(1)
    layer = _Layer(hidden, inter, E, k=2).to(DEV, torch.bfloat16)
    for p in layer.mlp.parameters():
        torch.nn.init.normal_(p, std=0.05)
    mgr, rec, _ = _capture(layer, [(2, 128), (1, 256)], hidden)
    ref_w = {t.param_name: t.param.detach().clone() for t in mgr.fused_tasks}
    for task in mgr.fused_tasks:
        E_, R, C = task.param.shape
        per = span_solve.expert_bytes(C, R, "mxfp4")
        budget = 3.5 * per / (1 << 30)  # three experts per span: spans 0-2, 3-5, 6-7
        assert span_solve.expert_span_size(C, R, budget, "mxfp4") == 3
        res = span_solve.solve_fused_task(mgr, task, 4, 32, DEV, vram_gb=budget, mode="mxfp4")
        assert [r.expert for r in res] == list(range(E))
        for r in res:
            parts = rec.rows.get((task.param_name, r.expert), [])
            rows = torch.cat(parts) if parts else torch.zeros(0, C, dtype=torch.bfloat16)
            assert r.tokens == rows.shape[0] and r.fallback is None
            W_e = ref_w[task.param_name][r.expert].cpu()
            rq, rs, _, rW, rrel = _oracle_expert(W_e, rows, 4, "mxfp4")
            agree = float((r.q == rq[0]).float().mean())
            assert agree >= 0.995, (task.param_name, r.expert, agree)
            assert abs(r.rel_err - float(rrel[0])) <= 0.01 * float(rrel[0]) + 1e-7
            # write-back: the parameter now holds the dequantized expert
            dq = task.param.detach()[r.expert].float().cpu()
            assert torch.equal(dq, rW[0].to(torch.bfloat16).float()) or agree < 1.0


@pytest.mark.parametrize("B,R,C", [(4, 256, 1024), (3, 4096, 512), (5, 640, 640)])
def test_affine_span_stays_within_the_bytes_counted_for_it(B, R, C):
    """The peak of a span's solve (Hessians included, its source weights not),
    the retry after a failed factorisation too."""
    g = torch.Generator(device=DEV).manual_seed(C)
    W = torch.randn(B, R, C, generator=g, device=DEV)
    x = torch.randn(C // 2, C, generator=g, device=DEV)
    singular = x.T @ x - 0.02 * torch.eye(C, device=DEV) * C
    for H in ((x.T @ x + torch.eye(C, device=DEV) * C), singular):
        H = H[None].repeat(B, 1, 1)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        out = gptq.solve_gptq(W, H, 4, 64)
        torch.cuda.synchronize()
        used = torch.cuda.max_memory_allocated() - before + H.numel() * 4
        assert used <= B * span_solve.expert_bytes(C, R, "affine") + (1 << 20)
        del out, H
