"""The work whose speed counts: attention calls as programs make them.

Every case is one call of a public entry point, ``forward_flash2`` (fp16,
head_dim 64, contiguous) or ``forward_flash2_ex`` (fp16 or bf16, head_dim 64
or 128, strided views, N_q != N_k, log-sum-exp, decode with a workspace).

A case is a dict:
  api     "flash2" or "ex"
  dtype   "f16" or "bf16"
  dim     head_dim, 64 or 128
  b, h    batch and heads
  nq, nk  query rows and keys
  causal  bottom-right aligned mask
  layout  "bhnd" (contiguous) or "bnhd" (tensors stored [B, N, H, D], passed
          as transposed views, the layout of projection outputs)
  out     whether the caller keeps an output buffer
  lse     whether the log-sum-exp is returned too
  ws      whether the caller keeps a split-KV workspace (decode loops do)
  scale   standard deviation of the inputs
"""

from __future__ import annotations

import math

import torch

import flashlite_amd as fl

_SM_SCALE = {64: 0.125, 128: 0.08838834764831845}


def _case(name, api, dtype, dim, b, h, nq, nk, causal, layout="bhnd", out=False, lse=False,
          ws=False, scale=1.0):
    c = dict(api=api, dtype=dtype, dim=dim, b=b, h=h, nq=nq, nk=nk, causal=causal, layout=layout,
             out=out, lse=lse, ws=ws, scale=scale)
    if name is not None:
        c["name"] = name
    return c


def listed():
    return [
        # The smallest call: one head, 128 rows; launch and host latency.
        _case("tiny-f16", "flash2", "f16", 64, 1, 1, 128, 128, False),
        # The benchmark's shortest sequence, into the caller's buffer.
        _case("short-f16", "flash2", "f16", 64, 2, 8, 512, 512, False, out=True),
        # An encoder batch of a head_dim-128 bf16 model, ragged length.
        _case("short-bf16-d128", "ex", "bf16", 128, 2, 8, 333, 333, False),
        # A training-style forward over projection outputs: ragged, causal,
        # log-sum-exp kept for a backward pass.
        _case("mid-bf16-causal-bnhd", "ex", "bf16", 64, 2, 8, 1999, 1999, True, layout="bnhd",
              lse=True),
        # The benchmark's headline size, both masks.
        _case("headline-f16", "flash2", "f16", 64, 2, 8, 4096, 4096, False, out=True),
        _case("headline-f16-causal", "flash2", "f16", 64, 2, 8, 4096, 4096, True, out=True),
        # A very long causal sequence.
        _case("long-f16-causal", "flash2", "f16", 64, 1, 16, 16384, 16384, True, scale=0.5),
        # Many small heads through a reused output buffer.
        _case("many-f16-causal", "flash2", "f16", 64, 32, 32, 256, 256, True, out=True),
        # Prefill of a prompt by a head_dim-128 bf16 model, projection layout.
        _case("prefill-bf16-d128", "ex", "bf16", 128, 1, 16, 3000, 3000, True, layout="bnhd",
              out=True),
        # One chunk of a chunked prefill: 512 new rows over a longer cache.
        _case("chunk-f16-d128", "ex", "f16", 128, 1, 16, 512, 4608, True, out=True),
        # Decode steps: one query row over the cache, buffers kept by the loop.
        _case("decode-f16", "ex", "f16", 64, 2, 8, 1, 4096, False, out=True, ws=True),
        _case("decode-bf16-d128", "ex", "bf16", 128, 4, 16, 1, 5000, False, out=True, ws=True),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


# A drawn case stays below the largest listed one (about 5.5e11 operations).
_MOST_FLOPS = 2.0e11
_MOST_BYTES = 3.0e8


def draw(rng):
    while True:
        kind = rng.choice(["self", "self", "self", "chunk", "decode", "decode"])
        dim = rng.choice([64, 64, 128])
        dtype = rng.choice(["f16", "bf16"])
        b = rng.choice([1, 1, 2, 2, 3, 4, 8, 32])
        h = rng.choice([1, 2, 4, 6, 8, 12, 16, 32])
        if kind == "self":
            nq = nk = _log_int(rng, 64, 16384)
            causal = rng.random() < 0.6
        elif kind == "chunk":
            nq = _log_int(rng, 33, 1024)
            nk = nq + _log_int(rng, 64, 8192)
            causal = True
        else:
            nq = rng.choice([1, 1, 1, 2, 5, 16])
            nk = _log_int(rng, 256, 16384)
            causal = nq > 1
        plain = kind == "self" and dtype == "f16" and dim == 64 and rng.random() < 0.6
        c = _case(None, "flash2" if plain else "ex", dtype, dim, b, h, nq, nk, causal,
                  layout="bhnd" if plain or rng.random() < 0.6 else "bnhd",
                  out=kind == "decode" or rng.random() < 0.5,
                  lse=not plain and rng.random() < 0.25, ws=kind == "decode",
                  scale=rng.choice([1.0, 1.0, 0.5]))
        w = work(c)
        if w["flops"] <= _MOST_FLOPS and w["bytes"] <= _MOST_BYTES:
            return c


def _dtype(case):
    return torch.float16 if case["dtype"] == "f16" else torch.bfloat16


def _inputs(case, seed):
    """q, k, v as [B, H, N, D] (views of [B, N, H, D] storage for "bnhd"):
    normal values, the usual projection of layer-normalised activations."""
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * int(seed) + 17)
    b, h, d = case["b"], case["h"], case["dim"]
    out = []
    for n in (case["nq"], case["nk"], case["nk"]):
        shape = (b, n, h, d) if case["layout"] == "bnhd" else (b, h, n, d)
        x = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
        x = (x * case["scale"]).to(_dtype(case))
        out.append(x.transpose(1, 2) if case["layout"] == "bnhd" else x)
    return out


def prepare(case, seed):
    q, k, v = _inputs(case, seed)
    state = {"q": q, "k": k, "v": v, "case": case, "sm": _SM_SCALE[case["dim"]], "out": None,
             "ws": None}
    if case["out"]:
        state["out"] = torch.empty_like(q)
    if case["ws"]:
        need = fl.splitkv_workspace_bytes(q, k, case["causal"])
        state["ws"] = torch.empty(need // 4 + 1, dtype=torch.float32, device=q.device)
    return state


def run(state):
    c = state["case"]
    if c["api"] == "flash2":
        return fl.forward_flash2(state["q"], state["k"], state["v"], state["sm"], c["causal"],
                                 state["out"])
    return fl.forward_flash2_ex(state["q"], state["k"], state["v"], state["sm"], c["causal"],
                                out=state["out"], return_lse=c["lse"], workspace=state["ws"])


def _pairs(case):
    """Visible (query, key) pairs of one head."""
    nq, nk = case["nq"], case["nk"]
    if not case["causal"]:
        return nq * nk
    first = max(0, nk - nq + 1)  # keys visible to row 0, one more per row
    return nq * first + nq * (nq - 1) // 2


def work(case):
    heads, d = case["b"] * case["h"], case["dim"]
    flops = 4 * heads * _pairs(case) * d
    elems = 2 * case["nq"] * d + 2 * case["nk"] * d  # q, o and k, v
    bytes_ = heads * (2 * elems + (4 * case["nq"] if case["lse"] else 0))
    return {"bytes": bytes_, "flops": flops}


def tolerance(case):
    # The output's rounding and that of the probabilities before the product
    # with V, each a unit in the last place or less of 11 (fp16) or 8 (bf16)
    # bits: against 64 bits the outputs are 2.4e-4 to 3.0e-4 (fp16) and
    # 2.1e-3 to 2.4e-3 (bf16) off in the norm, and at most 7.5e-3 and 3.2e-2
    # at one value (long causal sequences, whose root mean square is small
    # beside the first rows' values).  Four times that.
    if case["dtype"] == "f16":
        return {"rel": 1.2e-3, "max": 3e-2}
    return {"rel": 9e-3, "max": 1.2e-1}


def exact(case, seed):
    """Attention in 64 bits, a block of query rows of one head at a time."""
    q, k, v = _inputs(case, seed)
    b, h, nq, nk, d = case["b"], case["h"], case["nq"], case["nk"], case["dim"]
    sm = _SM_SCALE[d]
    out = torch.empty((b, h, nq, d), dtype=torch.float64, device=q.device)
    lse = torch.empty((b, h, nq), dtype=torch.float64, device=q.device)
    keys = torch.arange(nk, device=q.device)
    # heads of one batch entry go together while their scores fit 2^26 values
    step = max(1, min(h, (1 << 26) // max(1, nq * nk)))
    rows = max(1, min(nq, (1 << 26) // (step * nk)))
    for i in range(b):
        for h0 in range(0, h, step):
            hs = slice(h0, min(h, h0 + step))
            kk = k[i, hs].double().transpose(1, 2).contiguous()
            vv = v[i, hs].double().contiguous()
            for r0 in range(0, nq, rows):
                rs = slice(r0, min(nq, r0 + rows))
                s = torch.matmul(q[i, hs, rs].double().contiguous(), kk) * sm
                if case["causal"]:
                    last = torch.arange(rs.start, rs.stop, device=q.device) + (nk - nq)
                    s = s.masked_fill(keys[None, None, :] > last[None, :, None], -math.inf)
                lse[i, hs, rs] = torch.logsumexp(s, dim=-1)
                out[i, hs, rs] = torch.matmul(torch.softmax(s, dim=-1), vv)
    return (out, lse) if case["lse"] else out
