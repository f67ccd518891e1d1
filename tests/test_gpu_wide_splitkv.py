"""Split-KV decode for bf16 and head_dim 128 (fl_attn_fwd_ws and
forward_flash2_ex): chunk counts from 4 to 16, ragged last chunks, several
query rows, both masks, the log-sum-exp, graph replays.  The workspace is
exactly as large as the library asks for and starts as NaN.  Tolerances:
gpu_util (against the fp32 oracle).
"""

import numpy as np
import pytest

import flashlite_amd as fl
from flashlite_amd import capi
from gpu_util import (LSE_MAX_ABS, LSE_MEAN_ABS, assert_close_oracle, wide_inputs, wide_tol)
from oracle import attention_fp32, attention_lse, error_stats

pytestmark = pytest.mark.gpu

WIDE = [("fp16", 128), ("bf16", 64), ("bf16", 128)]
SHAPES = [(2, 1, 1537), (3, 32, 1600), (5, 17, 2047), (2, 1, 8191), (40, 1, 3001), (16, 4, 4096)]


def tensors(kind, xs, dev):
    import torch

    dt = torch.bfloat16 if kind == "bf16" else torch.float16
    return [torch.from_numpy(x).to(dev).to(dt) for x in xs]


@pytest.mark.parametrize("kind,d", WIDE)
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("h,nq,nk", SHAPES)
@pytest.mark.parametrize("sm,scale", [(0.125, 1.0), (1.0, 1.5)])
def test_decode(cuda, kind, d, causal, h, nq, nk, sm, scale):
    import torch

    xs = wide_inputs(kind, 1, h, nq, nk, d, seed=h + nq + nk, qk_scale=scale)
    q, k, v = tensors(kind, xs, cuda)
    o = torch.full_like(q, float("nan"))
    lse = torch.full((1, h, nq), float("nan"), dtype=torch.float32, device=cuda)
    p = capi.tensor_params_ex(q, k, v, o, sm, causal, lse=lse)
    dt = capi.DTYPE_BF16 if kind == "bf16" else capi.DTYPE_F16
    need = capi.workspace_bytes(p, dt)
    assert need > 0
    ws = torch.full((need // 4,), float("nan"), dtype=torch.float32, device=cuda)
    stream = torch.cuda.current_stream(cuda).cuda_stream
    capi.check(capi.fwd_ws(p, dt, ws.data_ptr(), need, stream))
    torch.cuda.synchronize(cuda)
    mx, mean = wide_tol(kind)
    assert_close_oracle(o.float().cpu().numpy(), None, None, None, sm, causal, max_abs=mx,
                        mean_abs=mean, ref=attention_fp32(*xs, sm, causal),
                        peaked=sm * scale >= 0.9, mant_bits=7 if kind == "bf16" else 10)
    lmx, lmean = error_stats(lse.cpu().numpy(), attention_lse(xs[0], xs[1], sm, causal))
    assert lmx <= LSE_MAX_ABS[kind] and lmean <= LSE_MEAN_ABS[kind]
    # too small a workspace, or none: one pass
    o2 = torch.full_like(q, float("nan"))
    p2 = capi.tensor_params_ex(q, k, v, o2, sm, causal)
    capi.check(capi.fwd_ws(p2, dt, ws.data_ptr(), need - 4, stream))
    o3 = torch.full_like(q, float("nan"))
    capi.check(capi.fwd_ws(capi.tensor_params_ex(q, k, v, o3, sm, causal), dt, 0, 0, stream))
    torch.cuda.synchronize(cuda)
    assert torch.equal(o2, o3)
    assert_close_oracle(o2.float().cpu().numpy(), None, None, None, sm, causal, max_abs=mx,
                        mean_abs=mean, ref=attention_fp32(*xs, sm, causal),
                        peaked=sm * scale >= 0.9, mant_bits=7 if kind == "bf16" else 10)


@pytest.mark.parametrize("kind,d", WIDE)
def test_binding_and_graph(cuda, kind, d):
    """A decode loop's buffers: eager with and without a workspace, strided
    [B, N, H, D] caches, replays of a graph with and without a workspace."""
    import torch

    q, k, v = tensors(kind, wide_inputs(kind, 2, 4, 1, 3000, d, seed=3), cuda)
    ref = fl.forward_flash2_ex(q, k, v, 0.125)
    need = fl.splitkv_workspace_bytes(q, k, False)
    assert need > 0 and fl.splitkv_workspace_bytes(q, k, False, 1) == 0
    ws = torch.empty(need // 4, dtype=torch.float32, device=cuda)
    out = torch.empty_like(q)
    assert torch.equal(fl.forward_flash2_ex(q, k, v, 0.125, out=out, workspace=ws), ref)
    kb, vb = (x.transpose(1, 2).contiguous().transpose(1, 2) for x in (k, v))
    assert torch.equal(fl.forward_flash2_ex(q, kb, vb, 0.125, workspace=ws), ref)
    one = fl.forward_flash2_ex(q, k, v, 0.125, num_splits=1)
    # a workspace it cannot use (host memory) is no error, as before
    host = torch.empty(need // 4, dtype=torch.float32)
    assert torch.equal(fl.forward_flash2_ex(q, k, v, 0.125, workspace=host), ref)
    for w, want in ((ws, ref), (None, one)):
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            fl.forward_flash2_ex(q, k, v, 0.125, out=out, workspace=w)
        for _ in range(3):
            out.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize(cuda)
            assert torch.equal(out, want)
            torch.empty(1 << 20, device=cuda).fill_(1.0)


@pytest.mark.parametrize("kind,d", WIDE)
def test_given_outputs_allocate_nothing(cuda, kind, d):
    """Without a workspace (or with one too small) a call that is given its
    outputs makes no allocation: one pass, the same bits as under capture."""
    import torch

    q, k, v = tensors(kind, wide_inputs(kind, 2, 4, 1, 3000, d, seed=5), cuda)
    one, one_lse = fl.forward_flash2_ex(q, k, v, 0.125, return_lse=True, num_splits=1)
    out, lse = torch.empty_like(one), torch.empty_like(one_lse)
    small = torch.empty(16, dtype=torch.float32, device=cuda)
    count = lambda: torch.cuda.memory_stats(cuda)["allocation.all.allocated"]  # noqa: E731
    for w in (None, small):
        out.fill_(float("nan"))
        torch.cuda.synchronize(cuda)
        n = count()
        fl.forward_flash2_ex(q, k, v, 0.125, out=out, workspace=w)
        fl.forward_flash2_ex(q, k, v, 0.125, out=out, return_lse=True, lse=lse, workspace=w)
        assert count() == n
        torch.cuda.synchronize(cuda)
        assert torch.equal(out, one) and torch.equal(lse, one_lse)


def test_refused_chunk_counts(cuda):
    q, k, v = tensors("bf16", wide_inputs("bf16", 1, 2, 1, 3000, 64, seed=4), cuda)
    with pytest.raises(RuntimeError, match="num_splits > 1"):
        fl.forward_flash2_ex(q, k, v, num_splits=4)
    assert fl.splitkv_workspace_bytes(q, k, False, 4) == 0
