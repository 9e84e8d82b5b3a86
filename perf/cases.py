"""Performance cases of the calibration solver.

Each case is one call (or short sequence of calls) that a calibration or
packing program makes through the public ``mlx_gptq`` API: routed capture and
Hessians, dense Hessians, the GPTQ solves in the MXFP and affine modes, the
round-to-nearest fallback, the range audit, the read side of stored
artifacts, and one whole step on a small matrix. Sizes are the ones of the
benchmark layers (``bench.py``) or generic.

``listed()`` are the fixed cases, ``draw()`` gives others over the same
ranges, ``prepare()`` builds what the program holds before the call,
``run()`` is one pass, ``exact()`` the same result in float64 from plain
torch.
"""

from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

# the package lives in a directory whose name is no Python identifier
sys.path.insert(0, os.path.join(os.getcwd(), "mlx-gptq-mxfp_amd"))

from mlx_gptq import artifacts, capture, gptq, grid, packing, validate_artifacts  # noqa: E402

DEV = "cuda"
_DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
_OFFSETS = {"mxfp4": (0, -1, -2, -3, -4, 1, 2), "mxfp8": (0, -1, 1)}


# --------------------------------------------------------------------------
# the cases
# --------------------------------------------------------------------------


def _solve(mode, experts, rows, cols, **kw):
    """A solve_gptq case with the API's usual arguments filled in."""
    c = {"kind": "solve", "mode": mode, "experts": experts, "rows": rows, "cols": cols, "bits": 4,
         "group": 32, "algorithm": "auto", "clip": "mse", "storage": "bf16", "wdtype": "bf16",
         "packed": True}
    if mode == "affine":
        c["group"] = 64
    if mode == "mxfp8":
        c["bits"] = 8
    c.update(kw)
    return c


def listed():
    return [
        # routed capture of an MoE layer's gate/up inputs: 64 batches stashed
        # with their top-8 expert ids, then every expert's Hessian
        {"name": "moe_capture", "kind": "capture", "experts": 128, "channels": 2048,
         "tokens": 131072, "top_k": 8, "batch": 2048},
        # Hessian of a dense MLP input from its stash
        {"name": "hessian_mlp", "kind": "hessian", "tokens": 65536, "channels": 4096},
        # every routed expert of an MoE layer in one MXFP4 safe-scale solve
        {"name": "moe_mxfp4", **_solve("mxfp4", 124, 1536, 2048)},
        # a dense MLP matrix, MXFP8 groupwise
        {"name": "mlp_mxfp8", **_solve("mxfp8", 1, 14336, 4096)},
        # a single linear layer on the affine grid, the API's default mode
        {"name": "linear_affine", **_solve("affine", 1, 2048, 2048)},
        # a span of experts on the affine grid
        {"name": "moe_affine", **_solve("affine", 32, 1536, 2048)},
        # a dense MLP matrix at 8 bits, groups of 128
        {"name": "mlp_affine8", **_solve("affine", 1, 14336, 4096, bits=8, group=128)},
        # one whole step on a small ragged matrix: stash, Hessian, solve, pack
        {"name": "small_step", "kind": "step", "mode": "mxfp4", "rows": 257, "cols": 736,
         "tokens": 301, "wdtype": "bf16"},
        # affine round-to-nearest of the experts that saw no token, packed
        {"name": "rtn_affine", "kind": "rtn", "mode": "affine", "experts": 4, "rows": 1536,
         "cols": 2048, "bits": 4, "group": 64, "clip": "mse", "storage": "bf16", "wdtype": "bf16"},
        # MXFP4 round-to-nearest of a large matrix without calibration, packed
        {"name": "rtn_mxfp4", "kind": "rtn", "mode": "mxfp4", "experts": 1, "rows": 25600,
         "cols": 5120, "bits": 4, "group": 32, "clip": "mse", "storage": "bf16", "wdtype": "bf16"},
        # range audit of an MXFP8 artifact against its source
        {"name": "audit_mxfp8", "kind": "audit", "mode": "mxfp8", "rows": 14336, "cols": 4096,
         "bits": 8, "group": 32, "wdtype": "bf16"},
        # read side of a stored 4-bit affine artifact: unpack, dequantize
        {"name": "read_affine", "kind": "read", "mode": "affine", "rows": 14336, "cols": 4096,
         "bits": 4, "group": 64, "storage": "bf16"},
    ]


def _log_int(rng, lo, hi, multiple=1):
    """An integer in [lo, hi], even over the logarithm, a multiple of `multiple`."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return max(multiple, min(hi // multiple, max(1, round(v / multiple))) * multiple)


def draw(rng):
    kind = rng.choice(("capture", "hessian", "mxfp", "mxfp", "affine", "affine", "affine", "step",
                       "rtn", "rtn", "audit", "read"))
    wdtype = rng.choice(("bf16", "bf16", "bf16", "f16", "f32"))
    storage = rng.choice(("bf16", "bf16", "f16"))
    if kind == "capture":
        return {"kind": "capture", "experts": rng.choice((8, 32, 64, 128)),
                "channels": _log_int(rng, 256, 2048, 8), "tokens": _log_int(rng, 512, 131072),
                "top_k": rng.choice((1, 2, 4, 8)), "batch": rng.choice((512, 2048, 4096))}
    if kind == "hessian":
        return {"kind": "hessian", "tokens": _log_int(rng, 256, 65536),
                "channels": _log_int(rng, 128, 4096, rng.choice((1, 8, 64)))}
    if kind == "mxfp":
        mode = rng.choice(("mxfp4", "mxfp4", "mxfp8"))
        cols = _log_int(rng, 128, 4096, 32)
        experts = rng.choice((1, 1, 4, 32, 124))
        rows = _log_int(rng, 64, max(64, min(14336, 390_000_000 // (experts * cols))))
        return _solve(mode, experts, rows, cols, wdtype=wdtype, packed=rng.random() < 0.75,
                      algorithm=rng.choice(("auto", "auto", "groupwise", "safe-scale-search")))
    if kind == "affine":
        group = rng.choice((32, 64, 64, 128))
        cols = _log_int(rng, 256, 4096, group)
        experts = rng.choice((1, 1, 4, 16, 32))
        experts = max(1, min(experts, 140_000_000 // (cols * cols)))
        rows = _log_int(rng, 64, max(64, min(14336, 100_000_000 // (experts * cols))))
        return _solve("affine", experts, rows, cols, bits=rng.choice((4, 4, 4, 8)), group=group,
                      clip=rng.choice(("mse", "mse", "minmax")), storage=storage, wdtype=wdtype,
                      packed=rng.random() < 0.5)
    if kind == "step":
        return {"kind": "step", "mode": rng.choice(("mxfp4", "mxfp8", "affine")),
                "rows": _log_int(rng, 16, 2048), "cols": _log_int(rng, 64, 1024, 64),
                "tokens": _log_int(rng, 16, 2048), "wdtype": wdtype}
    mode = rng.choice(("affine", "mxfp4", "mxfp8"))
    group = rng.choice((32, 64, 64, 128)) if mode == "affine" else 32
    bits = rng.choice((2, 4, 4, 8)) if mode == "affine" else {"mxfp4": 4, "mxfp8": 8}[mode]
    cols = _log_int(rng, 128, 5120, max(group, 32))
    rows = _log_int(rng, 64, 25600)
    if kind == "rtn":
        return {"kind": "rtn", "mode": mode, "experts": 1, "rows": rows, "cols": cols, "bits": bits,
                "group": group, "clip": rng.choice(("mse", "mse", "minmax")), "storage": storage,
                "wdtype": wdtype}
    if kind == "audit":
        return {"kind": "audit", "mode": mode, "rows": rows, "cols": cols, "bits": bits,
                "group": group, "wdtype": wdtype}
    return {"kind": "read", "mode": mode, "rows": rows, "cols": cols, "bits": bits, "group": group,
            "storage": storage}


# --------------------------------------------------------------------------
# inputs
# --------------------------------------------------------------------------


def _gen(seed, salt):
    return torch.Generator(device=DEV).manual_seed(seed * 1009 + salt)


def _rows(n, channels, seed, salt):
    """Calibration rows: N(0, 1) times a lognormal scale per channel, one
    channel in a hundred an outlier."""
    g = _gen(seed, salt)
    scale = torch.exp(torch.randn(channels, generator=g, device=DEV))
    scale[torch.randperm(channels, generator=g, device=DEV)[: channels // 100]] *= 20.0
    out = torch.empty(n, channels, dtype=torch.bfloat16, device=DEV)
    for a in range(0, n, 32768):
        b = min(n, a + 32768)
        out[a:b] = torch.randn(b - a, channels, generator=g, device=DEV) * scale
    return out


def _weights(shape, dtype, seed, salt):
    w = torch.randn(shape, generator=_gen(seed, salt), device=DEV).mul_(0.02)
    return w.to(_DTYPES[dtype])


def _hessians(experts, cols, seed):
    """One Hessian per expert, each from its own number of rows."""
    H = torch.empty(experts, cols, cols, device=DEV)
    counts = np.random.RandomState(seed % 2**31).randint(cols, 2 * cols + 1, experts)
    for e in range(experts):
        x = _rows(int(counts[e]), cols, seed, 100 + e).float()
        torch.mm(x.t(), x, out=H[e])
    return H


def _artifact(case, seed):
    """Source weights and the codes, scales and biases stored for them."""
    src = _weights((case["rows"], case["cols"]), case.get("wdtype", "bf16"), seed, 3)
    store = _DTYPES[case.get("storage", "bf16")]
    w = src.double().reshape(case["rows"], -1, case["group"])
    if case["mode"] == "affine":
        lo, hi = w.amin(-1), w.amax(-1)
        s = ((hi - lo) / (2 ** case["bits"] - 1)).to(store)
        b = lo.to(store)
        q = ((w - b.double().unsqueeze(-1)) / s.double().clamp(min=1e-12).unsqueeze(-1)).round_()
        q = q.clamp_(0, 2 ** case["bits"] - 1).to(torch.uint8).reshape(src.shape)
        return src, q, s, b
    e = _e8m0(w.abs().amax(-1), case["mode"])
    q = _mx_code(w / torch.exp2(e).unsqueeze(-1), case["mode"]).reshape(src.shape)
    return src, q, (e + 127).to(torch.uint8), None


def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind == "capture":
        X = _rows(case["tokens"], case["channels"], seed, 1)
        E, k = case["experts"], case["top_k"]
        g = _gen(seed, 2)
        # a skewed router: a Zipf-like bias over a random order of the experts
        bias = -1.1 * torch.log(torch.randperm(E, generator=g, device=DEV) + 1.0)
        logits = torch.randn(case["tokens"], E, generator=g, device=DEV) * 2.0 + bias
        s["top_k"] = logits.topk(k, dim=1).indices
        s["X"] = X
    elif kind == "hessian":
        s["stash"] = capture.Stash("x", case["channels"])
        s["stash"].add(_rows(case["tokens"], case["channels"], seed, 1))
    elif kind == "solve":
        s["W"] = _weights((case["experts"], case["rows"], case["cols"]), case["wdtype"], seed, 2)
        s["H"] = _hessians(case["experts"], case["cols"], seed)
    elif kind == "step":
        s["W"] = _weights((1, case["rows"], case["cols"]), case["wdtype"], seed, 2)
        s["X"] = _rows(case["tokens"], case["cols"], seed, 1)
    elif kind == "rtn":
        s["W"] = _weights((case["experts"], case["rows"], case["cols"]), case["wdtype"], seed, 2)
    elif kind == "audit":
        s["source"], s["q"], s["scales"], s["biases"] = _artifact(case, seed)
    else:
        _, q, s["scales"], s["biases"] = _artifact(case, seed)
        if case["bits"] == 4:
            c = q.reshape(case["rows"], -1, 2)
            q = c[..., 0] | (c[..., 1] << 4)
        s["stored"] = q.contiguous()
    return s


# --------------------------------------------------------------------------
# one pass
# --------------------------------------------------------------------------


def _call_solve(case, W, H):
    B, R, C = W.shape
    packed = None
    if case["packed"]:
        packed = torch.empty(B, R, C * case["bits"] // 32, dtype=torch.int32, device=W.device)
    q, s, b, w_dq, rel = gptq.solve_gptq(
        W, H, case["bits"], case["group"], clip=case["clip"],
        storage_dtype=_DTYPES[case["storage"]], mode=case["mode"],
        mxfp_algorithm=case["algorithm"], packed_out=packed)
    return {"q": q, "scales": s, "biases": b, "w_dq": w_dq, "rel_err": rel, "packed": packed}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "capture":
        stash = capture.RoutedStash("gate_up", case["channels"], case["experts"])
        for a in range(0, case["tokens"], case["batch"]):
            stash.add_routed(state["X"][a:a + case["batch"]], state["top_k"][a:a + case["batch"]])
        return {"H": stash.hessians(DEV)}
    if kind == "hessian":
        return {"H": state["stash"].hessian(DEV)}
    if kind == "solve":
        return _call_solve(case, state["W"], state["H"])
    if kind == "step":
        st = capture.Stash("x", case["cols"])
        st.add(state["X"])
        H = st.hessian(DEV).unsqueeze(0)
        out = _call_solve(_step_solve(case), state["W"], H)
        return {"H": H, **out}
    if kind == "rtn":
        W, bits = state["W"], case["bits"]
        if case["mode"] == "affine":
            q, s, b, dq = grid.rtn_quantize(W, bits, case["group"], case["clip"],
                                            _DTYPES[case["storage"]])
        else:
            q, s, b, dq = grid.rtn_quantize_mxfp(W, case["mode"])
        return {"q": q, "scales": s, "biases": b, "w_dq": dq,
                "packed": packing.pack_q(q, bits).view(torch.int32)}
    if kind == "audit":
        return validate_artifacts.range_audit(state["source"], state["q"], state["scales"],
                                              state["biases"], case["mode"], case["group"])
    q = state["stored"]
    if case["bits"] == 4:
        q = artifacts.unpack_nibbles(q)
    return {"q": q, "w_dq": grid.dequantize_artifact(q, state["scales"], state["biases"],
                                                     case["mode"], case["group"])}


def _step_solve(case):
    return _solve(case["mode"], 1, case["rows"], case["cols"], wdtype=case["wdtype"])


# --------------------------------------------------------------------------
# what a pass cannot do without
# --------------------------------------------------------------------------


def _solve_work(c):
    n = c["experts"] * c["rows"] * c["cols"]
    size = _DTYPES[c["wdtype"]].itemsize
    out = n * (4 + 1) + (n * c["bits"] / 8 if c["packed"] else 0)  # W_dq, codes, packed codes
    C, G = c["cols"], c["group"]
    if c["mode"] == "affine":
        # H and the scales and biases; factor and inverse, the column updates,
        # the clip candidates
        cand = 21 if c["clip"] == "mse" else 1
        return {"bytes": n * size + out + 4 * c["experts"] * C * C
                + 2 * n / G * _DTYPES[c["storage"]].itemsize,
                "flops": c["experts"] * 2 / 3 * C ** 3 + n * C + n * cand * 8}
    safe = c["algorithm"] == "safe-scale-search" or (c["algorithm"] == "auto" and c["mode"] == "mxfp4")
    cand = len(_OFFSETS[c["mode"]]) + 1 if safe else 0
    # the 32 x 32 diagonal blocks of H and one scale byte per group; the
    # column updates and the quadratic forms of the candidates
    return {"bytes": n * size + out + 4 * c["experts"] * C * 32 + n / 32,
            "flops": n * 31 + n * cand * 2 * 32}


def work(case):
    kind = case["kind"]
    if kind == "capture":
        C, T, E = case["channels"], case["tokens"], case["experts"]
        return {"bytes": 2 * T * C + 8 * T * case["top_k"] + 4 * E * C * C,
                "flops": T * case["top_k"] * C * (C + 1)}
    if kind == "hessian":
        C, T = case["channels"], case["tokens"]
        return {"bytes": 2 * T * C + 4 * C * C, "flops": T * C * (C + 1)}
    if kind == "solve":
        return _solve_work(case)
    if kind == "step":
        C, T = case["cols"], case["tokens"]
        w = _solve_work(_step_solve(case))
        return {"bytes": w["bytes"] + 2 * T * C, "flops": w["flops"] + T * C * (C + 1)}
    n = case.get("experts", 1) * case["rows"] * case["cols"]
    params = n / 32 if case["mode"] != "affine" else (
        2 * n / case["group"] * _DTYPES[case.get("storage", "bf16")].itemsize)
    if kind == "rtn":
        cand = 21 if case["mode"] == "affine" and case["clip"] == "mse" else 1
        return {"bytes": n * (_DTYPES[case["wdtype"]].itemsize + 5 + case["bits"] / 8) + params,
                "flops": n * cand * 8}
    if kind == "audit":
        return {"bytes": n * (_DTYPES[case["wdtype"]].itemsize + 1) + params, "flops": 4 * n}
    stored = n / 2 if case["bits"] == 4 else n
    return {"bytes": stored + (n if case["bits"] == 4 else 0) + 4 * n + params, "flops": 2 * n}


def tolerance(case):
    kind = case["kind"]
    if kind in ("capture", "hessian"):
        # fp32 sums: up to 4.4e-7 from float64 over these sizes
        return {"rel": 2e-6, "max": 2e-4}
    if kind in ("audit", "read"):
        return "exact"
    if kind == "rtn":
        # a clip candidate whose error ties another's to the last bits
        return "exact" if case["mode"] != "affine" else {"rel": 2e-3, "max": 0.99, "differ": 1e-3}
    if case["mode"] == "affine":
        # a code that flips at a rounding boundary moves the rest of its row:
        # up to 0.012 from float64 at 2048 columns and 4 bits
        return {"rel": 0.03, "max": 0.99, "differ": 0.01}
    # the same inside one group of 32: up to 4.1e-4 from float64 on the listed
    # matrices; one flipped code is 5e-3 of the smallest drawn one (8192
    # values, 1024 packed words)
    return {"rel": 0.01, "max": 0.99, "differ": 2e-3}


# --------------------------------------------------------------------------
# the same in float64
# --------------------------------------------------------------------------


def _e8m0(amax, mode):
    """Exponent of the shared scale: log2(amax / largest value), half to even."""
    e = torch.log2(amax / {"mxfp4": 6.0, "mxfp8": 448.0}[mode]).round()
    return torch.where(amax == 0, torch.zeros_like(e), e.clamp(-127, 127))


def _mx_value(x, mode):
    """x (float64, in units of the scale) on the E2M1 or E4M3 grid, half to even."""
    top, low, mant = (6.0, 0, 1) if mode == "mxfp4" else (448.0, -6, 3)
    a = x.abs().clamp(max=top)
    e = torch.floor(torch.log2(a.clamp(min=2.0 ** low))).clamp(min=low)
    step = torch.exp2(e - mant)
    return torch.copysign((a / step).round() * step, x)


def _mx_code(x, mode):
    """Code of each grid value (sign, exponent and mantissa bits)."""
    v = _mx_value(x, mode)
    a = v.abs()
    low, mant, top = (0, 1, 8) if mode == "mxfp4" else (-6, 3, 128)
    e = torch.floor(torch.log2(a.clamp(min=2.0 ** low))).clamp(min=low)
    mag = torch.where(a < 2.0 ** low, a * 2.0 ** (mant - low),
                      (e - low + 1) * 2 ** mant + (a / torch.exp2(e) - 1) * 2 ** mant)
    return (mag + torch.where(v < 0, float(top), 0.0)).to(torch.uint8)


def _hinv(H, damp=0.01):
    """Upper U with U^T U = (H + damp * mean(diag) I)^-1, per item, in float64."""
    n = H.shape[-1]
    lam = damp * H.diagonal(dim1=-2, dim2=-1).mean(-1).clamp(min=1e-8)
    Hd = H + lam[:, None, None] * torch.eye(n, dtype=H.dtype, device=H.device)
    V = torch.linalg.cholesky(Hd.flip(-1, -2)).flip(-1, -2)  # Hd = V V^T, V upper
    eye = torch.eye(n, dtype=H.dtype, device=H.device).expand_as(V)
    return torch.linalg.solve_triangular(V, eye, upper=True)


def _clip_search(w, case):
    """(scales, biases) of [..., group] values, rounded to the storage type."""
    store = _DTYPES[case["storage"]]
    maxq = 2 ** case["bits"] - 1
    lo, hi = w.amin(-1), w.amax(-1)
    steps = 20 if case["clip"] == "mse" else 0
    best = s = b = None
    for i in range(steps + 1):
        p = 1.0 - 0.2 * i / max(steps, 1)
        cs = ((hi - lo) * (p / maxq)).to(store).double()
        cb = (lo * p).to(store).double()
        _, dq = _affine(w, cs.unsqueeze(-1), cb.unsqueeze(-1), maxq)
        err = (dq - w).square_().sum(-1)
        if best is None:
            best, s, b = err, cs, cb
        else:
            t = err < best
            best, s, b = torch.where(t, err, best), torch.where(t, cs, s), torch.where(t, cb, b)
    return s, b


def _affine(w, s, b, maxq):
    q = ((w - b) / torch.where(s.abs() < 1e-12, 1.0, s)).round_().clamp_(0, maxq)
    return q, q * s + b


def _exact_affine(case, W, H):
    B, R, C = W.shape
    G = case["group"]
    maxq = 2 ** case["bits"] - 1
    bs = max(128, G) // G * G
    out, scales, biases = torch.empty_like(W), [], []
    U = torch.empty_like(H)
    for e in range(B):
        U[e] = _hinv(H[e:e + 1])[0]
    for i1 in range(0, C, bs):
        i2 = min(i1 + bs, C)
        w = W[:, :, i1:i2].clone()
        err = torch.empty_like(w)
        for j in range(i2 - i1):
            if j % G == 0:
                s, b = _clip_search(w[:, :, j:j + G], case)
                scales.append(s)
                biases.append(b)
            _, dq = _affine(w[:, :, j], s, b, maxq)
            err[:, :, j] = (w[:, :, j] - dq) / U[:, i1 + j, i1 + j].unsqueeze(-1)
            w[:, :, j + 1:] -= err[:, :, j:j + 1] * U[:, i1 + j:i1 + j + 1, i1 + j + 1:i2]
            out[:, :, i1 + j] = dq
        for e in range(B):
            W[e, :, i2:] -= err[e] @ U[e, i1:i2, i2:]
    return out, torch.stack(scales, -1), torch.stack(biases, -1)


def _exact_mxfp(case, W, H):
    mode = case["mode"]
    algorithm = case["algorithm"]
    if algorithm == "auto":
        algorithm = "safe-scale-search" if mode == "mxfp4" else "groupwise"
    out = torch.empty(W.shape, dtype=torch.float64, device=W.device)
    for g in range(0, W.shape[2], 32):
        w0 = W[:, :, g:g + 32].double()
        Hg = H[:, g:g + 32, g:g + 32].double()
        U = _hinv(Hg)
        e0 = _e8m0(w0.abs().amax(-1), mode)

        def quad(d):
            return (torch.matmul(d, Hg) * d).sum(-1)

        e_sel, best = e0, None
        if algorithm == "safe-scale-search":
            for off in _OFFSETS[mode]:
                e = (e0 + off).clamp(-127, 127)
                sc = torch.exp2(e).unsqueeze(-1)
                obj = quad(_mx_value(w0 / sc, mode) * sc - w0)
                if best is None:
                    best, e_sel = obj, e
                else:
                    t = obj < best
                    best, e_sel = torch.where(t, obj, best), torch.where(t, e, e_sel)
        sc = torch.exp2(e_sel).unsqueeze(-1)
        rtn = _mx_value(w0 / sc, mode) * sc
        w, dq = w0.clone(), torch.empty_like(w0)
        for c in range(32):
            dq[:, :, c] = _mx_value(w[:, :, c] / sc[:, :, 0], mode) * sc[:, :, 0]
            err = (w[:, :, c] - dq[:, :, c]) / U[:, c, c].unsqueeze(-1)
            w[:, :, c + 1:] -= err.unsqueeze(-1) * U[:, c:c + 1, c + 1:]
        keep = (dq.abs() <= (w0.abs().amax(-1, keepdim=True) * 32.0).clamp(min=2.0 ** -126)).all(-1)
        if best is not None:
            keep &= quad(dq - w0) <= best
        out[:, :, g:g + 32] = torch.where(keep.unsqueeze(-1), dq, rtn)
    return out


def _exact_solve(case, W, H):
    s = b = None
    if case["mode"] == "affine":
        w_dq, s, b = _exact_affine(case, W.double(), H.double())
    else:
        w_dq = _exact_mxfp(case, W, H)
    num = torch.stack([(w_dq[e] - W[e].double()).norm() for e in range(W.shape[0])])
    den = torch.stack([W[e].double().norm() for e in range(W.shape[0])])
    return {"q": None, "scales": s, "biases": b, "w_dq": w_dq, "rel_err": num / den, "packed": None}


@torch.no_grad()
def exact(case, seed):
    kind = case["kind"]
    st = prepare(case, seed)
    if kind == "capture":
        C, E = case["channels"], case["experts"]
        H = torch.zeros(E, C, C, dtype=torch.float64, device=DEV)
        for e in range(E):
            rows = (st["top_k"] == e).any(1).nonzero().flatten()
            for a in range(0, rows.numel(), 32768):
                x = st["X"].index_select(0, rows[a:a + 32768]).double()
                H[e] += x.t() @ x
        return {"H": H}
    if kind == "hessian":
        X = st["stash"].rows_on(DEV)
        H = torch.zeros(case["channels"], case["channels"], dtype=torch.float64, device=DEV)
        for a in range(0, X.shape[0], 32768):
            x = X[a:a + 32768].double()
            H += x.t() @ x
        return {"H": H}
    if kind == "solve":
        return _exact_solve(case, st["W"], st["H"])
    if kind == "step":
        x = st["X"].double()
        H = (x.t() @ x).unsqueeze(0)
        return {"H": H, **_exact_solve(_step_solve(case), st["W"], H)}
    if kind == "rtn":
        W = st["W"].double()
        w = W.reshape(*W.shape[:-1], -1, case["group"])
        if case["mode"] == "affine":
            s, b = _clip_search(w, case)
            _, dq = _affine(w, s.unsqueeze(-1), b.unsqueeze(-1), 2 ** case["bits"] - 1)
        else:
            s = b = None
            sc = torch.exp2(_e8m0(w.abs().amax(-1, keepdim=True), case["mode"]))
            dq = _mx_value(w / sc, case["mode"]) * sc
        return {"q": None, "scales": s, "biases": b, "w_dq": dq.reshape(W.shape), "packed": None}
    if kind == "audit":
        src = st["source"].double().reshape(case["rows"], -1, 32)
        dq = _dequantized(case, st["q"], st["scales"], st["biases"]).reshape(src.shape)
        smax, amax = src.abs().amax(-1), dq.abs().amax(-1)
        ratio = amax / (smax * 32.0).clamp(min=2.0 ** -126)
        return {"nonfinite": None, "exceed": None, "ratio": float(ratio.max()),
                "source_max": float(smax.max()), "artifact_max": float(amax.max())}
    q = st["stored"]
    if case["bits"] == 4:
        q = torch.stack((q & 15, q >> 4), -1).reshape(case["rows"], -1)
    return {"q": None, "w_dq": _dequantized(case, q, st["scales"], st["biases"])}


def _dequantized(case, q, scales, biases):
    v = q.double().reshape(case["rows"], -1, case["group"])
    if case["mode"] == "affine":
        return (v * scales.double().unsqueeze(-1) + biases.double().unsqueeze(-1)).reshape(q.shape)
    low, mant, top = (0, 1, 8) if case["mode"] == "mxfp4" else (-6, 3, 128)
    neg = v >= top
    mag = torch.where(neg, v - top, v)
    e = torch.floor(mag / 2 ** mant)
    m = mag - e * 2 ** mant
    a = torch.where(e == 0, m * 2.0 ** (low - mant),
                    torch.exp2(e - 1 + low) * (1 + m / 2 ** mant))
    sc = torch.exp2(scales.double().reshape(case["rows"], -1, 1) - 127)
    return (torch.where(neg, -a, a) * sc).reshape(q.shape)
