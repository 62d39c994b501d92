"""Performance cases: the work a training or evaluation program has this framework do.

``listed()`` names the fixed cases, ``draw(rng)`` makes further ones over the same
ranges; ``prepare`` / ``run`` execute one through the public entry points,
``work`` gives the bytes and flops it cannot do without, ``exact`` the result in
64 bits from plain torch, ``tolerance`` how far a correct result may be from it.

Every kind is a piece of the decoder's step (forward and backward) or a whole
call. The single layers go through the C entry points of include/nlearn_hip.h
on buffers the caller keeps, as an XLA FFI handler or a C program calls them:
``linear`` a projection, ``ffn`` the feed-forward block, ``attention`` the core
between QKV and output projection, ``norm`` the residual add with its
LayerNorm. The others go through the Python functions: ``lm_head`` the logits
with their loss as training runs them, ``fused_ce`` the same without keeping
the logits, ``forward`` the logits of a prompt (evaluation, no gradients),
``step`` one training step in its HIP graph.
"""
from __future__ import annotations

import dataclasses
import math

import torch
import torch.nn.functional as F

from nlearn_amd import _lib
from nlearn_amd.kernels.cross_entropy import linear_cross_entropy, lm_head_cross_entropy
from nlearn_amd.model import (BASELINE, count_params_cfg, device_param, flops_per_step, init_model, model_forward,
                              tree_leaves)
from nlearn_amd.train import AdamW, make_train_step

_BF16 = torch.bfloat16
_DEV = "cuda"
_D_HEAD = 64


# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------


def listed() -> list:
    return [
        # one short sequence through the QKV projection: latency and launches
        {"name": "linear_short", "kind": "linear", "tokens": 96, "d": 512, "n": 1536, "grad": True},
        # 8 sequences of 512 through the attention output projection
        {"name": "linear_bs8", "kind": "linear", "tokens": 4096, "d": 512, "n": 512, "grad": True},
        # the feed-forward block of a small batch (4 x 512)
        {"name": "ffn_bs4", "kind": "ffn", "tokens": 2048, "d": 512, "f": 2048},
        # ... and of the default batch (32 x 512)
        {"name": "ffn_bs32", "kind": "ffn", "tokens": 16384, "d": 512, "f": 2048},
        # attention of the default batch
        {"name": "attention_bs32", "kind": "attention", "batch": 32, "seq": 512, "heads": 8, "causal": True},
        # the long-sequence training shape
        {"name": "attention_long", "kind": "attention", "batch": 4, "seq": 4096, "heads": 8, "causal": True},
        # two sequences of an odd length (a last, short batch)
        {"name": "attention_ragged", "kind": "attention", "batch": 2, "seq": 777, "heads": 8, "causal": True},
        # residual add + LayerNorm of the default batch
        {"name": "norm_bs32", "kind": "norm", "rows": 16384, "d": 512},
        # logits and loss of the default batch, in the two chunks training uses
        {"name": "lm_head_bs32", "kind": "lm_head", "tokens": 16384, "d": 512, "vocab": 50257, "chunks": 2},
        # logits-free loss of four sequences of 511
        {"name": "fused_ce_ragged", "kind": "fused_ce", "tokens": 2044, "d": 512, "vocab": 50257},
        # logits of one prompt
        {"name": "forward_prompt", "kind": "forward", "batch": 1, "seq": 200},
        # a training step of 8 sequences of 512
        {"name": "step_bs8", "kind": "step", "batch": 8, "seq": 512},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    kind = rng.choice(["linear", "linear", "ffn", "ffn", "attention", "attention", "norm", "lm_head", "fused_ce",
                       "forward", "step"])
    d = rng.choice([256, 512, 512, 768, 1024])
    if kind == "linear":
        return {"kind": kind, "tokens": _log_int(rng, 64, 16384), "d": d, "n": d * rng.choice([1, 3]),
                "grad": rng.random() < 0.75}
    if kind == "ffn":
        return {"kind": kind, "tokens": _log_int(rng, 64, 16384), "d": d, "f": 4 * d}
    if kind == "attention":
        seq = _log_int(rng, 16, 4096)
        return {"kind": kind, "batch": _log_int(rng, 1, min(64, max(1, 16384 // seq))), "seq": seq,
                "heads": rng.choice([4, 8, 8, 12, 16]), "causal": rng.random() < 0.8}
    if kind == "norm":
        return {"kind": kind, "rows": _log_int(rng, 64, 32768), "d": d}
    if kind == "lm_head":
        return {"kind": kind, "tokens": _log_int(rng, 128, 16384), "d": 512,
                "vocab": rng.choice([50257, _log_int(rng, 4096, 50257)]), "chunks": rng.choice([1, 2])}
    if kind == "fused_ce":
        return {"kind": kind, "tokens": _log_int(rng, 128, 4096), "d": 512,
                "vocab": rng.choice([50257, _log_int(rng, 4096, 50257)])}
    if kind == "forward":
        return {"kind": kind, "batch": rng.randint(1, 8), "seq": _log_int(rng, 16, 512)}
    seq = _log_int(rng, 64, 512)
    return {"kind": kind, "batch": _log_int(rng, 1, 4096 // seq), "seq": seq}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _randn(gen, shape, std: float = 1.0, dtype=_BF16) -> torch.Tensor:
    return (torch.randn(shape, generator=gen, device=_DEV, dtype=torch.float32) * std).to(dtype)


def _tokens(gen, shape, vocab: int) -> torch.Tensor:
    """Token ids with the 1/rank frequencies of text."""
    u = torch.rand(shape, generator=gen, device=_DEV, dtype=torch.float64)
    return (torch.exp(u * math.log(vocab + 1.0)) - 1.0).to(torch.int32).clamp_(0, vocab - 1)


def _inputs(case: dict, seed: int) -> dict:
    """The case's tensors, from the seed alone: bf16 activations of unit scale
    (they leave a LayerNorm), fp32 weights N(0, 0.02), cotangents of the size a
    mean loss gives them."""
    g = torch.Generator(device=_DEV).manual_seed(seed)
    k = case["kind"]
    if k == "linear":
        M, d, n = case["tokens"], case["d"], case["n"]
        return {"x": _randn(g, (M, d)), "W": _randn(g, (d, n), 0.02, torch.float32), "dy": _randn(g, (M, n), 1e-3)}
    if k == "ffn":
        M, d, f = case["tokens"], case["d"], case["f"]
        return {"x": _randn(g, (M, d)), "W1": _randn(g, (d, f), 0.02, torch.float32),
                "b1": _randn(g, (f,), 0.02, torch.float32), "W2": _randn(g, (f, d), 0.02, torch.float32),
                "b2": _randn(g, (d,), 0.02, torch.float32), "dy": _randn(g, (M, d), 1e-3)}
    if k == "attention":
        B, S, H = case["batch"], case["seq"], case["heads"]
        return {"qkv": _randn(g, (B, S, 3, H, _D_HEAD)), "dy": _randn(g, (B, S, H * _D_HEAD), 1e-3)}
    if k == "norm":
        M, d = case["rows"], case["d"]
        return {"x": _randn(g, (M, d)), "r": _randn(g, (M, d), 0.5),
                "gamma": 1.0 + _randn(g, (d,), 0.05, torch.float32), "beta": _randn(g, (d,), 0.05, torch.float32),
                "dy": _randn(g, (M, d), 1e-3), "ds": _randn(g, (M, d), 1e-3)}
    if k in ("lm_head", "fused_ce"):
        M, d, V = case["tokens"], case["d"], case["vocab"]
        return {"x": _randn(g, (M, d)), "W": _randn(g, (d, V), 0.02, torch.float32), "t": _tokens(g, (M,), V)}
    cfg = _config(case)
    seq = case["seq"] + (1 if k == "step" else 0)
    return {"ids": _tokens(g, (case["batch"], seq), cfg.vocab_size)}


def _config(case: dict):
    return dataclasses.replace(BASELINE, max_seq_len=max(BASELINE.max_seq_len, case["seq"]))


def _empty(shape, dtype=_BF16) -> torch.Tensor:
    return torch.empty(shape, dtype=dtype, device=_DEV)


def _bytes(n: int) -> torch.Tensor:
    return _empty((max(int(n), 16),), torch.uint8)


def _ptr(t):
    return None if t is None else t.data_ptr()


_OP = {"N": _lib.NL_OP_N, "T": _lib.NL_OP_T}
_EPI_NONE, _EPI_BIAS, _EPI_BIAS_GELU, _EPI_DGELU = 0, 1, 2, 3


def _gemm(keep, A, B, ops: str, C, epi: int = _EPI_NONE, bias=None, aux=None):
    """nl_gemm_fused over dense operands: (name, arguments after the stream)."""
    M, N = C.shape
    K = A.shape[1] if ops[0] == "N" else A.shape[0]
    ws = _bytes(_lib.load().nl_gemm_ws_bytes(_OP[ops[0]], _OP[ops[1]], M, N, K))
    keep.append(ws)
    return ("nl_gemm_fused", (_OP[ops[0]], _OP[ops[1]], M, N, K, 1.0, _ptr(A), A.shape[1], _ptr(B), B.shape[1], 0.0,
                              _ptr(C), _lib.NL_DTYPE_F32 if C.dtype == torch.float32 else _lib.NL_DTYPE_BF16, N, None,
                              epi, _ptr(bias), _ptr(aux), N if aux is not None else 0, _ptr(ws), ws.numel()))


def _colsum(keep, x, out):
    rows, cols = x.shape
    ws = _bytes(_lib.load().nl_colsum_ws_bytes(rows, cols))
    keep.append(ws)
    return ("nl_colsum_bf16", (rows, cols, _ptr(x), cols, _ptr(out), 0, _ptr(ws), ws.numel()))


def _calls(case: dict, st: dict):
    """The C calls of one pass over st's buffers, and the tensors they leave."""
    k, keep = case["kind"], st["keep"]
    if k == "linear":
        x, W, dy = st["x"], st["W"].to(_BF16), st["dy"]
        keep.append(W)
        y = _empty(dy.shape)
        calls, outs = [_gemm(keep, x, W, "NN", y)], [y]
        if case["grad"]:
            dx, dW = _empty(x.shape), _empty(W.shape, torch.float32)
            calls += [_gemm(keep, dy, W, "NT", dx), _gemm(keep, x, dy, "TN", dW)]
            outs += [dx, dW]
        return calls, outs
    if k == "ffn":
        x, W1, W2, b1, b2, dy = st["x"], st["W1"].to(_BF16), st["W2"].to(_BF16), st["b1"], st["b2"], st["dy"]
        M, f = x.shape[0], W1.shape[1]
        u, h, du = _empty((M, f)), _empty((M, f)), _empty((M, f))
        y, dx = _empty(x.shape), _empty(x.shape)
        dW1, dW2 = _empty(W1.shape, torch.float32), _empty(W2.shape, torch.float32)
        db1, db2 = _empty(b1.shape, torch.float32), _empty(b2.shape, torch.float32)
        keep += [W1, W2, u, h, du]
        return [_gemm(keep, x, W1, "NN", h, _EPI_BIAS_GELU, b1, u), _gemm(keep, h, W2, "NN", y, _EPI_BIAS, b2),
                _colsum(keep, dy, db2), _gemm(keep, h, dy, "TN", dW2), _gemm(keep, dy, W2, "NT", du, _EPI_DGELU, None, u),
                _colsum(keep, du, db1), _gemm(keep, x, du, "TN", dW1), _gemm(keep, du, W1, "NT", dx)], \
            [y, dx, dW1, db1, dW2, db2]
    if k == "attention":
        B, S, H = case["batch"], case["seq"], case["heads"]
        qkv, dO = st["qkv"], st["dy"]
        o, dqkv, L = _empty(dO.shape), _empty(qkv.shape), _empty((B, H, S), torch.float32)
        ws = _bytes(_lib.load().nl_flash_attention_bwd_ws_bytes(B, H, S))
        keep += [L, ws]
        s3 = _lib.AttnStride(3 * S * H * _D_HEAD, _D_HEAD, 3 * H * _D_HEAD)
        s1 = _lib.AttnStride(S * H * _D_HEAD, _D_HEAD, H * _D_HEAD)
        dims = (B, H, S, _D_HEAD, 1.0 / math.sqrt(_D_HEAD), int(case["causal"]))
        ins = [a for i in range(3) for a in (_ptr(qkv[:, :, i]), s3)]
        grads = [a for i in range(3) for a in (_ptr(dqkv[:, :, i]), s3)]
        return [("nl_flash_attention_fwd", (*dims, *ins, _ptr(o), s1, _ptr(L))),
                ("nl_flash_attention_bwd", (*dims, *ins, _ptr(o), s1, _ptr(dO), s1, _ptr(L), *grads, _ptr(ws)))], \
            [o, dqkv]
    rows, d = st["x"].shape
    y, s, dx = _empty((rows, d)), _empty((rows, d)), _empty((rows, d))
    mean, rstd = _empty((rows,), torch.float32), _empty((rows,), torch.float32)
    dg, db = _empty((d,), torch.float32), _empty((d,), torch.float32)
    ws = _bytes(_lib.load().nl_layernorm_bwd_ws_bytes(rows, d))
    keep += [mean, rstd, ws]
    return [("nl_layernorm_fwd", (rows, d, _ptr(st["x"]), _ptr(st["r"]), _ptr(s), _ptr(st["gamma"]), _ptr(st["beta"]),
                                  1e-5, _ptr(y), _ptr(mean), _ptr(rstd))),
            ("nl_layernorm_bwd", (rows, d, _ptr(st["dy"]), _ptr(s), _ptr(mean), _ptr(rstd), _ptr(st["gamma"]),
                                  _ptr(st["ds"]), _ptr(dx), _ptr(dg), _ptr(db), 0, _ptr(ws), ws.numel()))], \
        [y, s, dx, dg, db]


_C_KINDS = ("linear", "ffn", "attention", "norm")


def prepare(case: dict, seed: int) -> dict:
    st = _inputs(case, seed)
    k = case["kind"]
    if k in _C_KINDS:
        st["keep"] = []
        st["calls"], st["outs"] = _calls(case, st)
    elif k in ("lm_head", "fused_ce"):
        st["W"] = device_param(st["W"].cpu().numpy(), _DEV)  # the row layout the model gives its head
        st["x"].requires_grad_(True)
        st["W"].requires_grad_(True)
    else:
        st["cfg"] = _config(case)
        st["params"] = init_model(seed, st["cfg"], _DEV)
    if k == "step":
        # a fine-tuning rate: the weights hardly move from pass to pass
        opt = AdamW(lambda _count: 1e-6)
        st["opt_state"] = opt.init(st["params"])
        st["step"] = make_train_step(opt, st["cfg"], graph=True, warmup=1)
        for _ in range(2):  # the eager warm-up step, then capture and first replay
            st["step"](st["params"], st["opt_state"], st["ids"])
        torch.cuda.synchronize()
    st["kind"], st["case"] = k, case
    return st


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------


def run(st: dict):
    k = st["kind"]
    if k in _C_KINDS:
        stream = torch.cuda.current_stream().cuda_stream
        for name, args in st["calls"]:
            _lib.call(name, stream, *args)
        return st["outs"]
    if k == "lm_head":
        loss = lm_head_cross_entropy(st["x"], st["W"], st["t"], st["case"]["chunks"])
        return [loss.detach(), *torch.autograd.grad(loss, (st["x"], st["W"]))]
    if k == "fused_ce":
        loss = linear_cross_entropy(st["x"], st["W"], st["t"])
        return [loss.detach(), *torch.autograd.grad(loss, (st["x"], st["W"]))]
    if k == "forward":
        with torch.no_grad():
            return [model_forward(st["params"], st["ids"], st["cfg"])]
    _, _, loss = st["step"](st["params"], st["opt_state"], st["ids"])
    return [loss, *(p.main_grad for p in tree_leaves(st["params"]))]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------


def work(case: dict) -> dict:
    """Inputs read once, outputs written once (bf16 activations and weight
    copies, fp32 weight gradients), and the matrix products' flops."""
    k = case["kind"]
    if k == "linear":
        M, K, N = case["tokens"], case["d"], case["n"]
        if not case["grad"]:
            return {"bytes": 2 * (M * K + K * N + M * N), "flops": 2 * M * N * K}
        return {"bytes": 2 * (2 * M * K + K * N + 2 * M * N) + 4 * K * N, "flops": 6 * M * N * K}
    if k == "ffn":
        M, d, f = case["tokens"], case["d"], case["f"]
        return {"bytes": 2 * (4 * M * d + 2 * d * f) + 4 * (2 * d * f + 2 * (d + f)), "flops": 12 * M * d * f}
    if k == "attention":
        B, S, H = case["batch"], case["seq"], case["heads"]
        pairs = B * H * S * S // (2 if case["causal"] else 1)
        return {"bytes": 2 * B * S * H * _D_HEAD * 8, "flops": 14 * pairs * _D_HEAD}
    if k == "norm":
        return {"bytes": 2 * 7 * case["rows"] * case["d"] + 16 * case["d"], "flops": 20 * case["rows"] * case["d"]}
    if k in ("lm_head", "fused_ce"):
        M, d, V = case["tokens"], case["d"], case["vocab"]
        return {"bytes": 2 * (2 * M * d + d * V) + 4 * (d * V + M), "flops": 6 * M * d * V}
    cfg = _config(case)
    B, S, n = case["batch"], case["seq"], count_params_cfg(cfg)
    fl = flops_per_step(cfg, B, S)
    if k == "forward":
        layers = n - cfg.vocab_size * cfg.d_model
        return {"bytes": 2 * layers + 4 * B * S + 2 * B * S * cfg.vocab_size,
                "flops": fl["gemm"] / 3 + fl["attention"] / 3.5}
    # the weights, gradients and moments an update reads and writes, and the bf16 weight copies
    return {"bytes": n * (4 + 3 * 8 + 2 * 2) + 4 * B * (S + 1), "flops": fl["total"]}


def tolerance(case: dict) -> dict:
    return _TOLERANCE[case["kind"]]


# bf16 results (and bf16 intermediates inside the pass) against 64 bits: about
# four times the largest error measured over the listed sizes and drawn ones
# (linear 1.7e-3, ffn 3.2e-3, attention 2.4e-3, norm 2.4e-3, lm_head 1.7e-3,
# fused_ce 3.6e-3, forward 7.7e-3, step 3.7e-2: gradients through four layers)
_TOLERANCE = {
    "linear": {"rel": 7e-3},
    "ffn": {"rel": 1.3e-2},
    "attention": {"rel": 1e-2},
    "norm": {"rel": 1e-2},
    "lm_head": {"rel": 7e-3},
    "fused_ce": {"rel": 1.4e-2},
    "forward": {"rel": 3e-2},
    "step": {"rel": 0.15},
}


# ---------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------


def _leaf64(t: torch.Tensor) -> torch.Tensor:
    return t.detach().double().requires_grad_(True)


def _weight64(t: torch.Tensor) -> torch.Tensor:
    """A GEMM weight: the products read its bf16 copy."""
    return _leaf64(t.detach().to(_BF16))


def _attention64(q, k, v, causal: bool) -> torch.Tensor:
    """(n, S, D) attention."""
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) / math.sqrt(q.shape[-1])
    if causal:
        S = q.shape[1]
        s = s.masked_fill(torch.ones(S, S, dtype=torch.bool, device=q.device).triu(1), -math.inf)
    return torch.matmul(torch.softmax(s, -1), v)


def _model64(p, ids, cfg) -> torch.Tensor:
    """Logits of the decoder with 64-bit parameters ``p``."""
    B, S = ids.shape
    d, H = cfg.d_model, cfg.n_heads
    ln = lambda q, x: F.layer_norm(x, (d,), q["gamma"], q["beta"], cfg.ln_eps)  # noqa: E731
    x = p["embeddings"]["token_embed"][ids.long()] + p["embeddings"]["pos_embed"][:S]
    for b in p["blocks"]:
        qkv = (ln(b["ln1"], x) @ b["attn"]["W_qkv"]).view(B, S, 3, H, d // H).permute(2, 0, 3, 1, 4)
        q, k, v = (t.reshape(B * H, S, d // H) for t in qkv)
        o = _attention64(q, k, v, True).view(B, H, S, d // H).permute(0, 2, 1, 3).reshape(B, S, d)
        x = x + o @ b["attn"]["W_o"]
        m = b["ffn"]
        x = x + F.gelu(ln(b["ln2"], x) @ m["W1"] + m["b1"], approximate="tanh") @ m["W2"] + m["b2"]
    return ln(p["ln_final"], x) @ p["lm_head"]


def exact(case: dict, seed: int):
    st = _inputs(case, seed)
    k = case["kind"]
    if k == "linear":
        x, W = _leaf64(st["x"]), _weight64(st["W"])
        y = x @ W
        if not case["grad"]:
            return [y.detach()]
        return [y.detach(), *torch.autograd.grad(y, (x, W), st["dy"].double())]
    if k == "ffn":
        ins = (_leaf64(st["x"]), _weight64(st["W1"]), _leaf64(st["b1"]), _weight64(st["W2"]), _leaf64(st["b2"]))
        y = F.gelu(ins[0] @ ins[1] + ins[2], approximate="tanh") @ ins[3] + ins[4]
        return [y.detach(), *torch.autograd.grad(y, ins, st["dy"].double())]
    if k == "attention":
        B, S, H = case["batch"], case["seq"], case["heads"]
        o = torch.empty((B, S, H * _D_HEAD), dtype=torch.float64, device=_DEV)
        dqkv = torch.empty((B, S, 3, H, _D_HEAD), dtype=torch.float64, device=_DEV)
        for b in range(B):  # one sequence at a time bounds the score matrices
            qkv = _leaf64(st["qkv"][b])
            q, kk, v = (qkv[:, i].transpose(0, 1).contiguous() for i in range(3))
            ob = _attention64(q, kk, v, case["causal"]).transpose(0, 1).reshape(S, H * _D_HEAD)
            o[b] = ob.detach()
            dqkv[b] = torch.autograd.grad(ob, qkv, st["dy"][b].double())[0]
        return [o, dqkv]
    if k == "norm":
        ins = tuple(_leaf64(st[n]) for n in ("x", "r", "gamma", "beta"))
        s = ins[0] + ins[1]
        y = F.layer_norm(s, (case["d"],), ins[2], ins[3], 1e-5)
        dx, _, dg, db = torch.autograd.grad((y, s), ins, (st["dy"].double(), st["ds"].double()))
        return [y.detach(), s.detach(), dx, dg, db]
    if k in ("lm_head", "fused_ce"):
        M = case["tokens"]
        x, W = st["x"].double(), st["W"].to(_BF16).double()
        loss = torch.zeros((), dtype=torch.float64, device=_DEV)
        dx, dW = torch.empty_like(x), torch.zeros_like(W)
        for r in range(0, M, 2048):  # a panel of rows at a time bounds the logits
            xr, tr = x[r:r + 2048], st["t"][r:r + 2048].long()
            lg = xr @ W
            lse = torch.logsumexp(lg, 1, keepdim=True)
            loss += (lse[:, 0] - lg.gather(1, tr[:, None])[:, 0]).sum() / M
            dl = torch.exp(lg - lse)
            dl.scatter_add_(1, tr[:, None], torch.full_like(lse, -1.0))
            dl /= M
            dx[r:r + 2048] = dl @ W.t()
            dW += xr.t() @ dl
        return [loss, dx, dW]
    cfg = _config(case)
    names = ("W_qkv", "W_o", "W1", "W2", "lm_head")
    params = init_model(seed, cfg, _DEV)

    def to64(t, key=None):
        if isinstance(t, dict):
            return {n: to64(v, n) for n, v in t.items()}
        if isinstance(t, list):
            return [to64(v) for v in t]
        return _weight64(t) if key in names else _leaf64(t)

    p64 = to64(params)
    if k == "forward":
        with torch.no_grad():
            return [_model64(p64, st["ids"], cfg)]
    logits = _model64(p64, st["ids"][:, :-1], cfg)
    loss = F.cross_entropy(logits.reshape(-1, cfg.vocab_size), st["ids"][:, 1:].reshape(-1).long())
    return [loss.detach(), *torch.autograd.grad(loss, tree_leaves(p64))]
