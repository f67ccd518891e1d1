"""GPU parity of the head-dim-128 configurations at the shapes where the
library's dispatcher takes each (an MI355X seen whole, 256 CUs), with the
sizes at the edges of tiles and blocks.  K and V are one head's, expanded
over the heads with stride 0, so that problems of hundreds of heads need the
oracle on a few heads only.  Tolerances: gpu_util (against the fp32 oracle).
"""

import numpy as np
import pytest

from flashlite_amd import capi
from gpu_util import (LSE_MAX_ABS, LSE_MEAN_ABS, assert_close_oracle, sample_rows, wide_inputs,
                      wide_tol)
from oracle import attention_fp32, attention_lse, error_stats

pytestmark = pytest.mark.gpu


def run_shared_kv(kind, h, nq, nk, d, causal, dev, seed, sm=0.1, qk_scale=1.0, bnhd=False):
    """One call over `h` heads that share one head's K and V; checks a few
    heads (and, for long sequences, a sample of rows) against the oracle."""
    import torch

    dt = torch.bfloat16 if kind == "bf16" else torch.float16
    checked = sorted({0, h // 2, h - 1})
    q, k, v = wide_inputs(kind, 1, len(checked), nq, nk, d, seed, qk_scale)
    g = torch.Generator(device="cpu")
    g.manual_seed(seed)
    tq = torch.randn((1, h, nq, d), generator=g).to(dev).to(dt)
    tq[:, checked] = torch.from_numpy(q).to(dev).to(dt)
    if bnhd:
        tq = tq.transpose(1, 2).contiguous().transpose(1, 2)
    tk, tv = (torch.from_numpy(x[:, :1]).to(dev).to(dt).expand(1, h, nk, d) for x in (k, v))
    o = torch.full_like(tq, float("nan"))
    lse = torch.full((1, h, nq), float("nan"), dtype=torch.float32, device=dev)
    p = capi.tensor_params_ex(tq, tk, tv, o, sm, causal, lse=lse)
    fn = capi.fwd_bf16_ex if kind == "bf16" else capi.fwd_ex
    capi.check(fn(p, torch.cuda.current_stream(dev).cuda_stream, -1))
    torch.cuda.synchronize(dev)
    assert torch.isfinite(o.float()).all() or nq > nk, "unwritten rows"
    kk, vv = (np.repeat(x[:, :1], len(checked), axis=1) for x in (k, v))
    rows = sample_rows(nq, count=64, seed=seed) if nq > 1200 else np.arange(nq)
    out = o[:, checked].float().cpu().numpy()
    mx, mean = wide_tol(kind)
    assert_close_oracle(out, None, None, None, sm, causal, rows=rows, max_abs=mx, mean_abs=mean,
                        ref=attention_fp32(q, kk, vv, sm, causal, rows=rows),
                        peaked=abs(sm) * qk_scale >= 0.9, mant_bits=7 if kind == "bf16" else 10)
    if nq <= 1200:
        ref_lse = attention_lse(q, kk, sm, causal)
        got = lse[:, checked].cpu().numpy()
        fin = np.isfinite(ref_lse)
        assert np.array_equal(fin, np.isfinite(got)), "lse -inf pattern"
        lmx, lmean = error_stats(got[fin], ref_lse[fin])
        assert lmx <= LSE_MAX_ABS[kind] + 2.0 ** -11 * np.abs(ref_lse[fin]).max()
        assert lmean <= LSE_MEAN_ABS[kind]


# (heads, N_q, N_k, causal): the configuration the dispatcher takes.
SHAPES = {
    "64-row split": [(3, 1, 1, False), (3, 33, 31, True), (3, 65, 64, True), (4, 130, 1025, False),
                     (16, 512, 700, True), (50, 450, 450, True), (3, 100, 37, True)],
    "64-row pairs": [(28, 1025, 1025, True), (26, 1089, 1089, True)],
    "128-row split": [(70, 200, 1537, False), (100, 250, 1600, True), (70, 257, 1568, False)],
    "128-row pairs": [(12, 4097, 4097, True)],
    "256-row groups": [(100, 300, 100, False), (512, 33, 4099, True), (256, 40, 4096, False)],
    "128-row groups": [(300, 100, 97, False), (300, 130, 65, True), (200, 300, 301, True)],
}


@pytest.mark.parametrize("kind", ["fp16", "bf16"])
@pytest.mark.parametrize("h,nq,nk,causal", [s for v in SHAPES.values() for s in v])
def test_dispatched_shapes(cuda, kind, h, nq, nk, causal):
    run_shared_kv(kind, h, nq, nk, 128, causal, cuda, seed=h + 7 * nq + nk)


# Scores far above the first tile's best hand the block to the checked pass.
@pytest.mark.parametrize("kind", ["fp16", "bf16"])
@pytest.mark.parametrize("h,nq,nk,causal", [SHAPES["64-row split"][3], SHAPES["64-row pairs"][0],
                                            SHAPES["128-row split"][1],
                                            SHAPES["128-row groups"][2]])
def test_peaked(cuda, kind, h, nq, nk, causal):
    run_shared_kv(kind, h, nq, nk, 128, causal, cuda, seed=h + nq, sm=1.0, qk_scale=2.0)


def test_projection_layout_and_negative_scale(cuda):
    run_shared_kv("bf16", 28, 1025, 1025, 128, True, cuda, seed=5, sm=-0.1, bnhd=True)
    run_shared_kv("fp16", 100, 250, 1600, 128, True, cuda, seed=6, sm=-0.1, bnhd=True)


def test_q_rows_beyond_32_bit_offsets(cuda):
    """Query rows 2^25 elements apart (64 MiB): more than a buffer offset
    reaches over a 32-row block, so Q takes the register path."""
    import torch

    n, stride = 40, 1 << 25
    q, k, v = wide_inputs("fp16", 1, 1, n, 70, 128, seed=9)
    store = torch.zeros((n - 1) * stride + 128, dtype=torch.float16, device=cuda)
    tq = store.as_strided((1, 1, n, 128), (0, 0, stride, 1))
    tq.copy_(torch.from_numpy(q))
    tk, tv = (torch.from_numpy(x).to(cuda).half() for x in (k, v))
    o = torch.full((1, 1, n, 128), float("nan"), dtype=torch.float16, device=cuda)
    p = capi.tensor_params_ex(tq, tk, tv, o, 0.1, True)
    capi.check(capi.fwd_ex(p, torch.cuda.current_stream(cuda).cuda_stream, -1))
    torch.cuda.synchronize(cuda)
    assert_close_oracle(o.float().cpu().numpy(), q, k, v, 0.1, True)
