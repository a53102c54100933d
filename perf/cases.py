"""Performance cases of the token-mixer library: what a user's program has it
do, through the public front end (q35mix.Context), at the mixer shapes of the
4B-class configuration (qwen35_config: 16 k / 32 v DeltaNet heads of 128, 16 q
heads on 4 kv heads of 256, hidden 2560) and, in drawn cases, other head counts
the tests hold.

Kinds of case:
  dn_decode     one token of one DeltaNet layer for n sequences
  dn_prefill    T tokens of one DeltaNet layer, from a zero or a running state
  attn_decode   one token of one attention layer for n sequences over their caches
  attn_prefill  T tokens of one attention layer behind `start` cached rows
  linear        a quantized projection of `tokens` rows (GGUF weight types)
  linear_f32    an F32 projection (the beta / alpha projections)
  boundary      residual add + RMSNorm + Q8_K blocks of `tokens` rows
  layer_decode  one whole DeltaNet layer of one decode step: boundary, the
                four input projections, the mixer, the output projection

Activations are torch tensors; the library takes device pointers.  Its states
and caches are filled and returned through torch views of its own buffers.
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "qwen3.5sharp_amd"))
import q35mix  # noqa: E402

EPS = 1e-6
HD, DK, HIDDEN = 256, 128, 2560
ROPE_HALF, ROPE_BASE = 32, 1e7
STQ1_0, Q2_0C, Q4_K, Q5_K, Q6_K, IQ4_XS = 1, 2, 4, 5, 6, 14
BLOCK_BYTES = {STQ1_0: 42, Q2_0C: 130, Q4_K: 144, Q5_K: 176, Q6_K: 210, IQ4_XS: 136}
BLOCK_VALUES = {STQ1_0: 256, Q2_0C: 512, Q4_K: 256, Q5_K: 256, Q6_K: 256, IQ4_XS: 256}


def listed():
    return [
        # Decode of one sequence: the mixer of each of the stack's DeltaNet layers, once per token.
        {"name": "dn_decode_1", "kind": "dn_decode", "n": 1, "nk": 16, "nv": 32},
        # A 2048-token prompt, first chunk of a conversation.
        {"name": "dn_prefill_2048", "kind": "dn_prefill", "T": 2048, "running": False, "nk": 16, "nv": 32},
        # A short user turn behind a conversation: an odd token count, a running state.
        {"name": "dn_prefill_77", "kind": "dn_prefill", "T": 77, "running": True, "nk": 16, "nv": 32},
        # Decode of one sequence in a conversation of 8K tokens.
        {"name": "attn_decode_8k", "kind": "attn_decode", "n": 1, "rows": 8192, "ragged": False, "nh": 16, "nkv": 4},
        # Batched decode of 8 long conversations of unequal lengths.
        {"name": "attn_decode_8x32k", "kind": "attn_decode", "n": 8, "rows": 32640, "ragged": True, "nh": 16, "nkv": 4},
        # The 2048-token prompt's attention layers.
        {"name": "attn_prefill_2048", "kind": "attn_prefill", "start": 0, "T": 2048, "nh": 16, "nkv": 4},
        # The next user turn of a conversation: few tokens over a long cache.
        {"name": "attn_prefill_turn", "kind": "attn_prefill", "start": 8000, "T": 133, "nh": 16, "nkv": 4},
        # The qkv projection of one decoded token (Q4_K_M files).
        {"name": "linear_q4k_1", "kind": "linear", "qtype": Q4_K, "n_in": 2560, "n_out": 8192, "tokens": 1, "order": 0},
        # The output projection of a batch of 8 decoded tokens (Q6_K in Q4_K_M files).
        {"name": "linear_q6k_8", "kind": "linear", "qtype": Q6_K, "n_in": 4096, "n_out": 2560, "tokens": 8, "order": 0},
        # The qkv projection of the 2048-token prompt.
        {"name": "linear_q4k_2048", "kind": "linear", "qtype": Q4_K, "n_in": 2560, "n_out": 8192, "tokens": 2048,
         "order": 0},
        # The qkv projection of a medium prompt with Q5_K weights (Q5_K_M files).
        {"name": "linear_q5k_500", "kind": "linear", "qtype": Q5_K, "n_in": 2560, "n_out": 8192, "tokens": 500,
         "order": 0},
        # One whole DeltaNet layer of a decode step, F32 beta / alpha projections among it.
        {"name": "layer_decode_1", "kind": "layer_decode", "n": 1, "nk": 16, "nv": 32},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    """One more case: sizes spread over their logarithm, no dearer than the largest listed one."""
    kind = rng.choice(["dn_decode", "dn_prefill", "attn_decode", "attn_prefill", "attn_prefill", "linear", "linear",
                       "linear", "linear", "linear_f32", "boundary", "layer_decode"])
    nk, nv = rng.choice([(16, 32), (16, 32), (16, 32), (16, 16), (8, 32)])
    nh, nkv = rng.choice([(16, 4), (16, 4), (16, 4), (8, 4), (16, 2)])
    if kind == "dn_decode":
        return {"kind": kind, "n": _log_int(rng, 1, 64), "nk": nk, "nv": nv}
    if kind == "layer_decode":
        return {"kind": kind, "n": _log_int(rng, 1, 32), "nk": 16, "nv": 32}
    if kind == "dn_prefill":
        return {"kind": kind, "T": _log_int(rng, 3, 4096), "running": rng.random() < 0.5, "nk": nk, "nv": nv}
    if kind == "attn_decode":
        n = _log_int(rng, 1, 24)
        return {"kind": kind, "n": n, "rows": _log_int(rng, 16, min(32640, 200000 // n)), "ragged": rng.random() < 0.5,
                "nh": nh, "nkv": nkv}
    if kind == "attn_prefill":
        start = 0 if rng.random() < 0.4 else _log_int(rng, 16, 16000)
        top = 2048        # T (start + T / 2) within that of 2048 tokens from an empty cache
        while top * (start + top / 2) > 2048 * 1024:
            top -= 1
        return {"kind": kind, "start": start, "T": _log_int(rng, 2, top), "nh": nh, "nkv": nkv}
    if kind == "boundary":
        return {"kind": kind, "dim": rng.choice([2560, 2560, 4096, 1024]), "tokens": _log_int(rng, 1, 2048)}
    if kind == "linear_f32":
        return {"kind": kind, "n_in": rng.choice([2560, 2560, 4096, 1000]), "n_out": rng.choice([32, 32, 16, 250]),
                "tokens": _log_int(rng, 1, 2048)}
    qtype = rng.choice([Q4_K, Q4_K, Q6_K, Q6_K, Q5_K, IQ4_XS, Q2_0C, STQ1_0])
    n_in, n_out = rng.choice([(2560, 8192), (2560, 4096), (2560, 1024), (4096, 2560), (2560, 32),
                              (512 * rng.randint(1, 12), rng.randint(40, 5000))])
    return {"kind": kind, "qtype": qtype, "n_in": n_in, "n_out": n_out,
            "tokens": _log_int(rng, 1, 2048) if rng.random() < 0.75 else 1,
            "order": 1 if qtype == Q6_K and rng.random() < 0.25 else 0}


# ------------------------------------------------------------------ inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(0x51355000 + seed)
    return g


def _normal(g, *shape, mean=0.0, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * std + mean


def _uniform(g, n, lo, hi):
    return torch.rand(n, generator=g, device="cuda", dtype=torch.float32) * (hi - lo) + lo


def _dn_weights(g, nk, nv):
    conv_dim = (2 * nk + nv) * DK
    return {"conv_w": _normal(g, 4, conv_dim, std=0.5), "ssm_a": -torch.exp(_uniform(g, nv, 0.0, 2.3)),
            "dt_bias": _normal(g, nv, std=0.1), "ssm_norm": _normal(g, DK, mean=1.0, std=0.02)}


def _dn_inputs(g, rows, nk, nv):
    return {"qkv": _normal(g, rows, (2 * nk + nv) * DK), "z": _normal(g, rows, nv * DK),
            "b": _normal(g, rows, nv), "a": _normal(g, rows, nv)}


def _dn_states(g, n, nk, nv):
    return {"state": _normal(g, n, nv, DK, DK, std=0.1), "win": _normal(g, n, (2 * nk + nv) * DK, 3)}


def _attn_inputs(g, rows, nh, nkv):
    return {"q_gate": _normal(g, rows, 2 * nh * HD), "k": _normal(g, rows, nkv * HD), "v": _normal(g, rows, nkv * HD)}


def _attn_weights(g):
    return {"q_norm": _normal(g, HD, mean=1.0, std=0.02), "k_norm": _normal(g, HD, mean=1.0, std=0.02)}


def _quant_rows(g, qtype, n_out, n_in):
    """Well-formed weight blocks: uniform quants, fp16 scales of trained weights' size."""
    nblk = n_out * (n_in // BLOCK_VALUES[qtype])
    b = torch.randint(0, 256, (nblk, BLOCK_BYTES[qtype]), generator=g, device="cuda", dtype=torch.uint8)
    d = _uniform(g, nblk, 0.004, 0.02)
    half = (d * 0.05 if qtype == IQ4_XS else d).half().view(torch.uint8).view(nblk, 2)
    at = {STQ1_0: 40, Q6_K: 208}.get(qtype, 0)
    b[:, at:at + 2] = half
    if qtype in (Q4_K, Q5_K):
        b[:, 2:4] = _uniform(g, nblk, 0.004, 0.02).half().view(torch.uint8).view(nblk, 2)
    return b


def _lens(case):
    n, rows = case["n"], case["rows"]
    return [max(1, rows - (i * rows) // (3 * n)) if case["ragged"] else rows for i in range(n)]


def _cache_rows(seed, seq, which, nkv, rows):
    """K or V rows of one sequence, [kv_heads][rows][256]."""
    return _normal(_gen(seed * 131 + 17 * seq + which + 1), nkv, rows, HD)


def _inputs(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    if kind in ("dn_decode", "dn_prefill"):
        n = case.get("n", 1)
        rows = case["T"] if kind == "dn_prefill" else n
        x = _dn_inputs(g, rows, case["nk"], case["nv"])
        x.update(_dn_weights(g, case["nk"], case["nv"]))
        x.update(_dn_states(g, n, case["nk"], case["nv"]))
        if kind == "dn_prefill" and not case["running"]:
            x["state"].zero_()
            x["win"].zero_()
        return x
    if kind in ("attn_decode", "attn_prefill"):
        x = _attn_inputs(g, case["T"] if kind == "attn_prefill" else case["n"], case["nh"], case["nkv"])
        x.update(_attn_weights(g))
        return x
    if kind == "linear":
        return {"w": _quant_rows(g, case["qtype"], case["n_out"], case["n_in"]),
                "x": _normal(g, case["tokens"], case["n_in"])}
    if kind == "linear_f32":
        return {"w": _normal(g, case["n_out"], case["n_in"], std=0.02), "x": _normal(g, case["tokens"], case["n_in"])}
    if kind == "boundary":
        return {"hidden": _normal(g, case["tokens"], case["dim"]),
                "delta": _normal(g, case["tokens"], case["dim"], std=0.1), "w": _normal(g, case["dim"], std=0.02)}
    assert kind == "layer_decode", kind
    n, nk, nv = case["n"], case["nk"], case["nv"]
    x = {"hidden": _normal(g, n, HIDDEN), "delta": _normal(g, n, HIDDEN, std=0.1), "w": _normal(g, HIDDEN, std=0.02),
         "w_qkv": _quant_rows(g, Q4_K, (2 * nk + nv) * DK, HIDDEN), "w_gate": _quant_rows(g, Q4_K, nv * DK, HIDDEN),
         "w_beta": _normal(g, nv, HIDDEN, std=0.02), "w_alpha": _normal(g, nv, HIDDEN, std=0.02),
         "w_out": _quant_rows(g, Q6_K, HIDDEN, nv * DK)}
    x.update(_dn_weights(g, nk, nv))
    x.update(_dn_states(g, n, nk, nv))
    return x


# ------------------------------------------------------------------ the library's buffers

class _Owner:
    """A context that closes once neither the state nor a view of its buffers is left."""

    def __init__(self, *a, **k):
        self.ctx = q35mix.Context(*a, **k)

    def __del__(self):
        self.ctx.close()


class _Foreign:
    def __init__(self, owner, ptr, shape, strides):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "strides": strides, "typestr": "<f4",
                                         "data": (ptr, False), "version": 2}


def _view(owner, n, kind, shape):
    """Layer 0's buffers of sequences 0 .. n - 1, which lie at one distance, as one tensor [n][shape]."""
    ptrs = [owner.ctx.state_device_ptr(0, i, kind)[0] for i in range(n)]
    inner = [4 * math.prod(shape[k + 1:]) for k in range(len(shape))]
    step = ptrs[1] - ptrs[0] if n > 1 else 4 * math.prod(shape)
    assert all(p == ptrs[0] + i * step for i, p in enumerate(ptrs))
    return torch.as_tensor(_Foreign(owner, ptrs[0], (n, *shape), (step, *inner)), device="cuda")


class _Buf:
    """A torch tensor as the front end takes device buffers (.ptr)."""

    def __init__(self, t):
        assert t.is_contiguous()
        self.t, self.ptr, self.nbytes = t, t.data_ptr(), t.numel() * t.element_size()


def _bufs(x, *names):
    return [_Buf(x[k]) for k in names]


def _host(x, *names):
    return {k: x[k].cpu().numpy() for k in names}


def _dn_context(x, n, nk, nv):
    o = _Owner(q35mix.qwen35_config(num_layers=1, n_k_heads=nk, n_v_heads=nv, is_recurrent=[1]), n_seqs=n, kv_capacity=16)
    o.ctx.set_deltanet_weights(0, _host(x, "conv_w", "ssm_a", "dt_bias", "ssm_norm"))
    states = _view(o, n, q35mix.STATE_RECURRENT, (nv, DK, DK))
    wins = _view(o, n, q35mix.STATE_CONV, ((2 * nk + nv) * DK, 3))
    states.copy_(x["state"])
    host = x["win"].cpu().numpy()
    for i in range(n):
        o.ctx.state_write(0, i, q35mix.STATE_CONV, host[i])
    return o, states, wins


def _attn_context(case, x, seed, lens, room):
    o = _Owner(q35mix.qwen35_config(num_layers=1, num_heads=case["nh"], num_kv_heads=case["nkv"], is_recurrent=[0]),
               n_seqs=len(lens), kv_capacity=max(lens) + room)
    o.ctx.set_attn_weights(0, _host(x, "q_norm", "k_norm"))
    caches = [_view(o, len(lens), kind, (case["nkv"], max(lens) + room, HD))
              for kind in (q35mix.STATE_KEYS, q35mix.STATE_VALUES)]
    for i, rows in enumerate(lens):
        if rows:
            for which, c in enumerate(caches):
                c[i, :, :rows].copy_(_cache_rows(seed, i, which, case["nkv"], rows))
            o.ctx.advance(i, rows)
    return o, caches


def prepare(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    s = {"kind": kind, "case": case}
    empty = lambda *shape: torch.zeros(*shape, device="cuda", dtype=torch.float32)  # noqa: E731
    if kind in ("dn_decode", "dn_prefill"):
        n = case.get("n", 1)
        s["owner"], s["states"], s["wins"] = _dn_context(x, n, case["nk"], case["nv"])
        s["out"] = empty(x["z"].shape)
        s["args"] = _bufs(x, "qkv", "z", "b", "a") + [_Buf(s["out"])]
        s["seqs"] = list(range(n))
    elif kind == "attn_decode":
        lens = _lens(case)
        s["owner"], caches = _attn_context(case, x, seed, lens, 1)
        s["rows"] = [c[i, :, r] for i, r in enumerate(lens) for c in caches]       # the rows a pass writes
        s["out"] = empty(case["n"], case["nh"] * HD)
        s["args"] = _bufs(x, "q_gate", "k", "v") + [_Buf(s["out"])]
        s["seqs"] = list(range(case["n"]))
    elif kind == "attn_prefill":
        s["owner"], caches = _attn_context(case, x, seed, [case["start"]], case["T"])
        s["rows"] = [c[0, :, case["start"]:] for c in caches]
        s["out"] = empty(case["T"], case["nh"] * HD)
        s["args"] = _bufs(x, "q_gate", "k", "v") + [_Buf(s["out"])]
    else:
        n = case["n"] if kind == "layer_decode" else 1
        if kind == "layer_decode":
            s["owner"], s["states"], s["wins"] = _dn_context(x, n, case["nk"], case["nv"])
        else:
            s["owner"] = _Owner(q35mix.qwen35_config(num_layers=1, is_recurrent=[1]), n_seqs=1, kv_capacity=16)
        if case.get("order"):
            s["owner"].ctx.set_projection_order(q35mix.PROJ_BLOCK)
        if kind in ("linear", "linear_f32"):
            s["out"] = empty(case["tokens"], case["n_out"])
            s["args"] = _bufs(x, "w", "x") + [_Buf(s["out"])]
        else:
            rows, dim = (case["tokens"], case["dim"]) if kind == "boundary" else (n, HIDDEN)
            s["hidden"], s["y"] = x["hidden"], empty(rows, dim)
            q8 = torch.zeros(q35mix.lib().q35m_q8k_bytes(dim, rows), device="cuda", dtype=torch.uint8)
            s["q8"] = q8
            s["args"] = _bufs(x, "hidden", "delta", "w") + [_Buf(s["y"]), _Buf(q8)]
        if kind == "layer_decode":
            s["weights"] = _bufs(x, "w_qkv", "w_gate", "w_beta", "w_alpha", "w_out")
            nv = case["nv"]
            s["mid"] = [_Buf(empty(n, c)) for c in ((2 * case["nk"] + nv) * DK, nv * DK, nv, nv, nv * DK)]
            s["out"] = empty(n, HIDDEN)
            s["final"] = _Buf(s["out"])
            s["seqs"] = list(range(n))
    s["ctx"] = s["owner"].ctx
    return s


def run(s):
    ctx, case, a = s["ctx"], s["case"], s["args"]
    kind = s["kind"]
    if kind == "dn_decode":
        ctx.deltanet_decode(0, s["seqs"], *a)
        return {"out": s["out"], "states": s["states"], "windows": s["wins"]}
    if kind == "dn_prefill":
        ctx.deltanet_prefill(0, 0, case["T"], *a)
        return {"out": s["out"], "states": s["states"], "windows": s["wins"]}
    if kind == "attn_decode":
        ctx.attn_decode(0, s["seqs"], *a)
        return {"out": s["out"], "rows": s["rows"]}
    if kind == "attn_prefill":
        ctx.attn_prefill(0, 0, case["T"], *a)
        return {"out": s["out"], "rows": s["rows"]}
    if kind == "linear":
        ctx.linear_q(case["qtype"], *a, case["n_in"], case["n_out"], case["tokens"])
        return s["out"]
    if kind == "linear_f32":
        ctx.linear_f32(*a, case["n_in"], case["n_out"], case["tokens"])
        return s["out"]
    if kind == "boundary":
        ctx.add_rmsnorm(*a, case["dim"], case["tokens"], EPS)
        return {"hidden": s["hidden"], "y": s["y"], "q8": s["q8"]}
    # One DeltaNet layer of a decode step, as the reference chains it: the
    # residual add and norm (with the projections' Q8_K), qkv, gate, beta and
    # alpha, the mixer, the output projection.
    n, nk, nv = case["n"], case["nk"], case["nv"]
    w_qkv, w_gate, w_beta, w_alpha, w_out = s["weights"]
    qkv, z, b, al, mixed = s["mid"]
    y, q8 = a[3], a[4]
    ctx.add_rmsnorm(*a, HIDDEN, n, EPS)
    ctx.linear_q_prequant(Q4_K, w_qkv, q8, qkv, HIDDEN, (2 * nk + nv) * DK, n)
    ctx.linear_q_prequant(Q4_K, w_gate, q8, z, HIDDEN, nv * DK, n)
    ctx.linear_f32(w_beta, y, b, HIDDEN, nv, n)
    ctx.linear_f32(w_alpha, y, al, HIDDEN, nv, n)
    ctx.deltanet_decode(0, s["seqs"], qkv, z, b, al, mixed)
    ctx.linear_q(Q6_K, w_out, mixed, s["final"], nv * DK, HIDDEN, n)
    return {"out": s["out"], "hidden": s["hidden"], "states": s["states"]}


# ------------------------------------------------------------------ work and tolerance

def work(case):
    """Bytes: inputs, weights and states read once, outputs and states written once.  Flops: the delta rule's three
    128 x 128 products a head and token, the causal Q K^T and P V, the projections' products."""
    kind = case["kind"]
    if kind in ("dn_decode", "dn_prefill", "layer_decode"):
        nk, nv = case["nk"], case["nv"]
        n = case.get("n", 1)
        rows = case.get("T", n)
        conv = (2 * nk + nv) * DK
        b = 4 * (n * (2 * nv * DK * DK + 6 * conv) + 4 * conv + rows * (conv + 2 * nv * DK + 2 * nv))
        f = rows * nv * 6 * DK * DK
        if kind == "layer_decode":
            w = (conv + nv * DK) * HIDDEN // 256 * 144 + nv * DK * HIDDEN // 256 * 210 + 8 * nv * HIDDEN
            b += w + 4 * n * HIDDEN * 5
            f += 2 * n * HIDDEN * (conv + 2 * nv * DK + 2 * nv)
        return {"bytes": b, "flops": f}
    if kind in ("attn_decode", "attn_prefill"):
        nh, nkv = case["nh"], case["nkv"]
        if kind == "attn_decode":
            lens, rows = _lens(case), case["n"]
            pairs = sum(lens) + rows
        else:
            lens, rows = [case["start"]], case["T"]
            pairs = rows * case["start"] + rows * (rows + 1) // 2
        return {"bytes": 4 * HD * (2 * nkv * (sum(lens) + 2 * rows) + 3 * nh * rows), "flops": 4 * HD * nh * pairs}
    if kind == "linear":
        n = case["n_in"] * case["n_out"]
        return {"bytes": n // BLOCK_VALUES[case["qtype"]] * BLOCK_BYTES[case["qtype"]]
                + 4 * case["tokens"] * (case["n_in"] + case["n_out"]), "flops": 2 * n * case["tokens"]}
    if kind == "linear_f32":
        n = case["n_in"] * case["n_out"]
        return {"bytes": 4 * (n + case["tokens"] * (case["n_in"] + case["n_out"])), "flops": 2 * n * case["tokens"]}
    n = case["tokens"] * case["dim"]
    return {"bytes": 16 * n + 4 * case["dim"] + n // 256 * 304, "flops": 6 * n}


def tolerance(case):
    """The projections and the boundary keep the reference's arithmetic bit for bit (their contract), except Q6_K in
    the opt-in block order; the mixers are fp32 with free summation orders."""
    kind = case["kind"]
    if kind in ("linear_f32", "boundary"):
        return "exact"
    if kind == "linear":
        return {"rel": 2e-6, "max": 2e-5} if case["order"] else "exact"
    if kind == "layer_decode":
        # the mixer's output is rounded to 8 bits for the last projection: a value at a rounding edge moves a step
        return {"rel": 2e-3, "max": 2e-2}
    if kind in ("dn_decode", "dn_prefill"):
        return {"rel": 1e-6, "max": 4e-5}
    return {"rel": 8e-6, "max": 1e-4}


# ------------------------------------------------------------------ 64-bit results

def _softplus64(x):
    ex = torch.exp(x)
    series = ex - ex ** 2 / 2 + ex ** 3 / 3 - ex ** 4 / 4
    return torch.where(x > 20, x, torch.where(x < -10, ex, torch.where(ex < 0.5, series, torch.log1p(ex))))


def _silu64(x):
    return x / (1 + torch.exp(-x))


def _delta64(conv, z, b, a, x, S, nk, nv):
    """Sequential delta rule over rows of [T][batch]...; S [batch][nv][dk][dv] is updated in place."""
    T, batch = conv.shape[0], conv.shape[1]
    R = nv // nk
    q = conv[..., :nk * DK].reshape(T, batch, nk, DK).repeat_interleave(R, 2)
    k = conv[..., nk * DK:2 * nk * DK].reshape(T, batch, nk, DK).repeat_interleave(R, 2)
    v = conv[..., 2 * nk * DK:].reshape(T, batch, nv, DK)
    q = q / torch.sqrt((q ** 2).sum(-1, keepdim=True) + EPS) / math.sqrt(DK)
    k = k / torch.sqrt((k ** 2).sum(-1, keepdim=True) + EPS)
    beta = 1 / (1 + torch.exp(-b))
    decay = torch.exp(x["ssm_a"].double() * _softplus64(a + x["dt_bias"].double()))
    o = torch.empty_like(v)
    for t in range(T):
        S.mul_(decay[t][..., None, None])
        d = beta[t][..., None] * (v[t] - (S * k[t][..., None]).sum(-2))
        S.addcmul_(k[t][..., None], d[..., None, :])
        o[t] = (S * q[t][..., None]).sum(-2)
    r = 1 / torch.sqrt((o ** 2).mean(-1, keepdim=True) + EPS)
    return (o * r * x["ssm_norm"].double() * _silu64(z.reshape(T, batch, nv, DK))).reshape(T, batch, nv * DK)


def _dn_decode64(x, qkv, z, b, a, nk, nv):
    S, win = x["state"].double(), x["win"].double()
    full = torch.cat([win, qkv.double()[..., None]], -1)                    # [n][conv][4], oldest first
    conv = _silu64((full * x["conv_w"].double().t()).sum(-1))
    out = _delta64(conv[None], z.double()[None], b.double()[None], a.double()[None], x, S, nk, nv)[0]
    return out, S, full[..., 1:]


def _rope_norm64(r, w, pos):
    """r [rows][heads][256] at positions pos [rows]: rotation of dims (d, d + 32), then the (1 + w) norm."""
    m = ctypes.CDLL("libm.so.6")
    m.powf.restype, m.powf.argtypes = ctypes.c_float, [ctypes.c_float, ctypes.c_float]
    fr = np.array([np.float32(1) / np.float32(m.powf(ROPE_BASE, np.float32(i) / np.float32(ROPE_HALF)))
                   for i in range(ROPE_HALF)], np.float32)
    ang = torch.from_numpy((pos.cpu().numpy().astype(np.float32)[:, None] * fr).astype(np.float64)).cuda()[:, None]
    c, s = torch.cos(ang), torch.sin(ang)
    y = r.double().clone()
    a, b = y[..., :ROPE_HALF].clone(), y[..., ROPE_HALF:2 * ROPE_HALF].clone()
    y[..., :ROPE_HALF], y[..., ROPE_HALF:2 * ROPE_HALF] = a * c - b * s, a * s + b * c
    return y / torch.sqrt((y ** 2).mean(-1, keepdim=True) + EPS) * (1 + w.double())


def _attend64(q, gate, K, V, visible):
    """q, gate [rows][heads of one kv head][256], K and V [len][256]; row i sees visible[i] cache rows."""
    mask = torch.arange(K.shape[0], device="cuda")[None] < visible[:, None]
    out = torch.empty_like(q)
    for h in range(q.shape[1]):
        s = (q[:, h] @ K.t()) / math.sqrt(HD)
        out[:, h] = torch.softmax(s.masked_fill(~mask, -math.inf), -1) @ V
    return out / (1 + torch.exp(-gate))


def _attn64(case, seed, x):
    nh, nkv = case["nh"], case["nkv"]
    G = nh // nkv
    lens = _lens(case) if case["kind"] == "attn_decode" else [case["start"]]
    T = case.get("T", 1)
    outs, rows = [], []
    for i, start in enumerate(lens):
        pick = slice(i, i + 1) if case["kind"] == "attn_decode" else slice(0, T)
        pos = start + torch.arange(T, device="cuda")
        qg = x["q_gate"][pick].double().reshape(T, nh, 2, HD)
        q = _rope_norm64(qg[:, :, 0], x["q_norm"], pos)
        kn = _rope_norm64(x["k"][pick].reshape(T, nkv, HD), x["k_norm"], pos).transpose(0, 1)
        vn = x["v"][pick].double().reshape(T, nkv, HD).transpose(0, 1)
        K0, V0 = (_cache_rows(seed, i, w, nkv, start) if start else None for w in (0, 1))
        out = torch.empty(T, nh, HD, device="cuda", dtype=torch.float64)
        for h in range(nkv):
            K = torch.cat([K0[h].double(), kn[h]]) if start else kn[h]
            V = torch.cat([V0[h].double(), vn[h]]) if start else vn[h]
            out[:, G * h:G * h + G] = _attend64(q[:, G * h:G * h + G], qg[:, G * h:G * h + G, 1], K, V, pos + 1)
        outs.append(out.reshape(T, nh * HD))
        rows += [kn[:, 0], vn[:, 0]] if case["kind"] == "attn_decode" else [kn, vn]
    return {"out": torch.cat(outs), "rows": rows}


def _q8k64(x):
    """Q8_K of rows x (fp32): the scale from the first value of largest magnitude, ties to even."""
    v = x.float().reshape(x.shape[0], -1, 256)
    first = v.gather(-1, v.abs().argmax(-1, keepdim=True))
    isc = torch.where(first == 0, torch.zeros_like(first), -127.0 / first)
    q = torch.clamp(torch.round(v * isc), -127, 127).double()
    d = torch.where(first == 0, torch.zeros_like(first), 1.0 / isc).double()
    return (q * d).reshape(x.shape)


def _k_scales(sc):
    """Q4_K / Q5_K 6-bit scales and mins of the 12 packed bytes: two [blocks][8]."""
    lo, mid, hi = sc[:, 0:4], sc[:, 4:8], sc[:, 8:12]
    return (torch.cat([lo & 63, (hi & 15) | ((lo >> 6) << 4)], 1), torch.cat([mid & 63, (hi >> 4) | ((mid >> 6) << 4)], 1))


def _dequant64(qtype, b, n_out, n_in):
    b = b.to(torch.int64)
    f16 = lambda at: b[:, at:at + 2].to(torch.uint8).contiguous().view(torch.float16).double()  # noqa: E731
    nblk = b.shape[0]
    if qtype in (Q4_K, Q5_K):
        sc, mn = _k_scales(b[:, 4:16])
        qs = b[:, -128:].reshape(nblk, 4, 1, 32)
        v = torch.cat([qs & 15, qs >> 4], 2).reshape(nblk, 8, 32)
        if qtype == Q5_K:
            bit = torch.arange(8, device=b.device).reshape(1, 8, 1)
            v = v + 16 * ((b[:, 16:48].reshape(nblk, 1, 32) >> bit) & 1)
        w = (f16(0) * sc)[..., None] * v - (f16(2) * mn)[..., None]
    elif qtype == Q6_K:
        ql, qh = b[:, :128].reshape(nblk, 2, 2, 32), b[:, 128:192].reshape(nblk, 2, 1, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)                                          # [blk][half][part][32]
        shift = torch.tensor([0, 2, 4, 6], device=b.device).reshape(1, 1, 4, 1)
        v = (lo | (((qh >> shift) & 3) << 4)) - 32
        sc = b[:, 192:208].to(torch.uint8).view(torch.int8).double().reshape(nblk, 2, 4, 2, 1)
        w = (f16(208).reshape(-1, 1, 1, 1, 1) * sc) * v.reshape(nblk, 2, 4, 2, 16)
    elif qtype == IQ4_XS:
        grid = torch.tensor([-127, -104, -83, -65, -49, -35, -22, -10, 1, 13, 25, 38, 53, 69, 89, 113], device=b.device)
        ib = torch.arange(8, device=b.device)
        ls = ((b[:, 4 + ib // 2] >> (4 * (ib % 2))) & 15) | ((((b[:, 2:3] + 256 * b[:, 3:4]) >> (2 * ib)) & 3) << 4)
        qs = b[:, 8:].reshape(nblk, 8, 16)
        w = (f16(0) * (ls - 32))[..., None] * grid[torch.cat([qs & 15, qs >> 4], 2)]
    elif qtype == Q2_0C:
        codes = torch.stack([(b[:, 2:] >> (2 * k)) & 3 for k in range(4)], 2)
        w = f16(0)[..., None] * (2 * codes - 3)
    else:
        book = torch.tensor([0xA9, 0x89, 0x29, 0x09, 0xA6, 0x86, 0x26, 0x06, 0x9A, 0x92, 0x1A, 0x12, 0x6A, 0x62, 0x4A,
                             0x42, 0x01, 0x21, 0x81, 0xA1, 0x04, 0x24, 0x84, 0xA4, 0x10, 0x18, 0x90, 0x98, 0x40, 0x48,
                             0x60, 0x68], device=b.device)
        slot = torch.stack([b[:, :32] & 15, b[:, :32] >> 4], 2).reshape(nblk, 64)
        sign = torch.stack([(b[:, 32:40] >> k) & 1 for k in range(8)], 2).reshape(nblk, 64)
        pat = book[16 * sign + slot]
        lanes = torch.stack([((pat >> (2 * k)) & 3) - 1 for k in range(4)], 2).reshape(nblk, 4, 16, 4)
        w = f16(40).reshape(-1, 1, 1, 1) * lanes.transpose(2, 3)
    return w.reshape(n_out, n_in)


def exact(case, seed):
    x = _inputs(case, seed)
    kind = case["kind"]
    if kind == "dn_decode":
        out, S, win = _dn_decode64(x, x["qkv"], x["z"], x["b"], x["a"], case["nk"], case["nv"])
        return {"out": out, "states": S, "windows": win}
    if kind == "dn_prefill":
        T, w, v = case["T"], x["conv_w"].double(), x["qkv"].double()
        acc = torch.zeros_like(v)
        for j in range(min(4, T)):                   # tap j meets the input j tokens back, zeros before the first
            acc[j:] += w[j] * v[:T - j]
        S = x["state"].double()
        out = _delta64(_silu64(acc)[:, None], x["z"].double()[:, None], x["b"].double()[:, None],
                       x["a"].double()[:, None], x, S, case["nk"], case["nv"])[:, 0]
        return {"out": out, "states": S, "windows": v[None, T - 3:].transpose(1, 2)}
    if kind in ("attn_decode", "attn_prefill"):
        return _attn64(case, seed, x)
    if kind == "linear":
        return _q8k64(x["x"]) @ _dequant64(case["qtype"], x["w"], case["n_out"], case["n_in"]).t()
    if kind == "linear_f32":
        return x["x"].double() @ x["w"].double().t()
    h = (x["hidden"] + x["delta"]).double()
    y = h / torch.sqrt((h ** 2).mean(-1, keepdim=True) + EPS) * (1 + x["w"].double())
    if kind == "boundary":
        return {"hidden": h, "y": y, "q8": None}
    n, nk, nv = case["n"], case["nk"], case["nv"]
    xq = _q8k64(y)
    qkv = xq @ _dequant64(Q4_K, x["w_qkv"], (2 * nk + nv) * DK, HIDDEN).t()
    z = xq @ _dequant64(Q4_K, x["w_gate"], nv * DK, HIDDEN).t()
    b, a = y @ x["w_beta"].double().t(), y @ x["w_alpha"].double().t()
    mixed, S, _ = _dn_decode64(x, qkv, z, b, a, nk, nv)
    out = _q8k64(mixed) @ _dequant64(Q6_K, x["w_out"], HIDDEN, nv * DK).t()
    return {"out": out, "hidden": h, "states": S}
