"""NaN and infinite inputs reach the rows they concern, and no other, on every
path: one pass, key-range merges inside a work-group, and key chunks with the
combine kernel.  Against softmax(Q K^T sm_scale) V in float64, whose NaN
pattern the outputs must have; the rest within gpu_util's bounds.
"""

import numpy as np
import pytest

from flashlite_amd import capi
from gpu_util import (QUARTER_CFG, SLOT_W4_CFG, STREAM_CFG, config_fits, wide_inputs, wide_tol)

pytestmark = pytest.mark.gpu

HEADS = 4  # one plant each; a case's further heads are clean


def reference(q, k, v, sm, causal):
    nq, nk = q.shape[2], k.shape[2]
    with np.errstate(invalid="ignore"):
        s = np.matmul(q.astype(np.float64), np.swapaxes(k, 2, 3).astype(np.float64)) * sm
        if causal:
            s = np.where(np.arange(nk) <= np.arange(nq)[:, None] + (nk - nq), s, -np.inf)
        p = np.exp(s - s.max(axis=-1, keepdims=True))
        p /= p.sum(axis=-1, keepdims=True)
        # (a key that is masked out weighs nothing, whatever its V holds)
        out = np.matmul(p, np.nan_to_num(v.astype(np.float64)))
        for b, h, j, c in np.argwhere(np.isnan(v)):
            seen = ~np.isneginf(s[b, h, :, j])
            out[b, h, seen, c] = np.nan
    return out


def plant(q, k, v):
    """Head 0: a NaN query row.  1: a NaN key.  2: an infinite key (a score of
    +inf makes the row NaN, one of -inf drops the key).  3: a NaN in V under
    keys whose weight underflows to 0 (0 times NaN is NaN)."""
    nq, nk = q.shape[2], k.shape[2]
    q[0, 0, nq // 2, 3] = np.nan
    k[0, 1, nk // 3, 5] = np.nan
    k[0, 2, 2 * nk // 3, 5] = np.inf
    q[0, 3] = np.abs(q[0, 3]) + 0.5
    k[0, 3, nk // 2:] = -20.0
    v[0, 3, 7 * nk // 8, 7] = np.nan


def run(kind, d, h, nq, nk, causal, dev, launch):
    import torch

    q, k, v = wide_inputs(kind, 1, HEADS, nq, nk, d, seed=nq + nk + d)
    plant(q, k, v)
    dt = torch.bfloat16 if kind == "bf16" else torch.float16
    ts = []
    for x in (q, k, v):
        t = torch.zeros((1, h) + x.shape[2:], dtype=dt, device=dev)
        t[:, :HEADS] = torch.from_numpy(x).to(dev).to(dt)
        ts.append(t)
    o = torch.full_like(ts[0], 7.0)
    p = capi.tensor_params_ex(*ts, o, 0.125, causal)
    launch(p, capi.DTYPE_BF16 if kind == "bf16" else capi.DTYPE_F16,
           torch.cuda.current_stream(dev).cuda_stream)
    torch.cuda.synchronize(dev)
    out = o[:, :HEADS].float().cpu().numpy()
    ref = reference(q, k, v, 0.125, causal)
    for head in range(HEADS):
        # A masked key's V still meets p = 0 in the tile that holds the
        # diagonal (head 3, causal): those rows are not compared.
        rows = np.arange(nq) if head != 3 else np.flatnonzero(
            np.arange(nq) + (nk - nq if causal else nk) >= 7 * nk // 8)
        got, want = out[0, head, rows], ref[0, head, rows]
        assert np.array_equal(np.isnan(got), np.isnan(want)), f"NaN pattern of head {head}"
        fin = ~np.isnan(want)
        assert np.isfinite(got[fin]).all()
        if fin.any():
            mx, mean = wide_tol(kind)
            err = np.abs(got[fin] - want[fin])
            assert err.max() <= mx + np.abs(want[fin]).max() * 2.0 ** (-8 if kind == "bf16" else -11)
            assert err.mean() <= mean + np.abs(want[fin]).mean() * 2.0 ** (-8 if kind == "bf16" else -11)


def chunked(splits):
    """Key chunks: `splits` of them, or the library's plan (0)."""
    import torch

    def go(p, dtype, stream):
        if splits:
            need = capi.splitkv_workspace_bytes(p, splits)
        else:
            need = capi.workspace_bytes(p, dtype)
        assert need > 0
        ws = torch.full((need // 4,), float("nan"), dtype=torch.float32, device="cuda:0")
        if splits:
            capi.check(capi.fwd_splitkv(p, ws.data_ptr(), need, stream, splits))
        else:
            capi.check(capi.fwd_ws(p, dtype, ws.data_ptr(), need, stream))
        torch.cuda.synchronize()

    return go


def one_pass(config):
    def go(p, dtype, stream):
        fn = capi.fwd_bf16_ex if dtype == capi.DTYPE_BF16 else capi.fwd_ex
        capi.check(fn(p, stream, config))

    return go


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("nq,nk", [(1, 3000), (5, 4096), (32, 2100)])
@pytest.mark.parametrize("kind,d", [("fp16", 64), ("fp16", 128), ("bf16", 64), ("bf16", 128)])
def test_chunks(cuda, kind, d, nq, nk, causal):
    run(kind, d, HEADS, nq, nk, causal, cuda, chunked(0))


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("splits", [2, 8, 30, 64])
def test_requested_chunks(cuda, splits, causal):
    """Pipelined and key-quarter chunks, and the combine's loop over more
    chunks than it loads up front."""
    run("fp16", 64, HEADS, 9, 4096, causal, cuda, chunked(splits))


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("kind,config", [("fp16", c) for c in range(-1, 10)] +
                         [("bf16", c) for c in range(-1, 10) if c not in (0, 1)])
def test_one_pass(cuda, kind, config, causal):
    nk = 250 if config == STREAM_CFG else 500 if config == QUARTER_CFG else 900
    assert config < 0 or config_fits(config, nk)
    run(kind, 64, HEADS, nk, nk, causal, cuda, one_pass(config))


# The dispatcher's head-dim-128 kernels by shape (256 CUs): 32-row groups,
# 64-row split, 64-row pairs, 128-row split; and the 128-row groups by id.
@pytest.mark.parametrize("h,nq,nk,causal,config", [
    (HEADS, 100, 700, True, -1), (40, 300, 301, True, -1), (40, 300, 301, False, -1),
    (24, 1025, 1025, True, -1), (100, 250, 1600, True, -1), (HEADS, 300, 301, True, SLOT_W4_CFG)])
def test_head_dim_128(cuda, h, nq, nk, causal, config):
    run("bf16", 128, h, nq, nk, causal, cuda, one_pass(config))
