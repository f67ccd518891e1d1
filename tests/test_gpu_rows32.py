"""GPU parity of the 32-row groups (few query blocks: the key tiles dealt to
4 or 8 waves) at both head dims and element types, through the dispatcher
(which at head dim 64 takes the streaming groups up to 64 keys), at the edges
of tiles, of the waves' shares and of the 8-wave rule (2048 keys).  Tolerances: gpu_util (against the fp32 oracle).
"""

import numpy as np
import pytest

import flashlite_amd as fl
from gpu_util import (LSE_MAX_ABS, LSE_MEAN_ABS, assert_close_oracle, run_wide, wide_inputs,
                      wide_tol)
from oracle import attention_fp32, attention_lse, error_stats

pytestmark = pytest.mark.gpu

KINDS = [("fp16", 64), ("fp16", 128), ("bf16", 64), ("bf16", 128)]
# N_q, N_k: single rows and keys, block edges, fewer tiles than waves, ragged
# tails, rows with no visible key (N_q > N_k), 8-wave groups.
SHAPES = [(1, 1), (1, 255), (31, 64), (32, 65), (33, 33), (64, 193), (40, 256), (100, 37),
          (65, 700), (5, 1000), (33, 2047), (32, 2048), (70, 2113),
          (1, 66), (100, 70), (95, 129)]


def check(kind, d, nq, nk, sm, causal, dev, scale=1.0, views=None, h=3):
    q, k, v = wide_inputs(kind, 1, h, nq, nk, d, seed=nq + 3 * nk + d, qk_scale=scale)
    out, lse = run_wide(kind, q, k, v, sm, causal, dev, lse=True, views=views)
    mx, mean = wide_tol(kind)
    assert_close_oracle(out, None, None, None, sm, causal, max_abs=mx, mean_abs=mean,
                        ref=attention_fp32(q, k, v, sm, causal), peaked=abs(sm) * scale >= 0.9,
                        mant_bits=7 if kind == "bf16" else 10)
    ref = attention_lse(q, k, sm, causal)
    fin = np.isfinite(ref)
    assert np.array_equal(fin, np.isfinite(lse)), "lse -inf pattern"
    if fin.any():
        lmx, lmean = error_stats(lse[fin], ref[fin])
        assert lmx <= LSE_MAX_ABS[kind] and lmean <= LSE_MEAN_ABS[kind]


@pytest.mark.parametrize("kind,d", KINDS)
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("nq,nk", SHAPES)
def test_shapes(cuda, kind, d, nq, nk, causal):
    check(kind, d, nq, nk, 0.125, causal, cuda)


@pytest.mark.parametrize("kind,d", KINDS)
@pytest.mark.parametrize("causal", [False, True])
def test_scales_and_layout(cuda, kind, d, causal):
    """Negative, unit-c and peaked scales (the stabiliser moves), and
    [B, N, H, D] storage."""
    bnhd = lambda *ts: [t.transpose(1, 2).contiguous().transpose(1, 2) for t in ts]  # noqa: E731
    check(kind, d, 70, 600, -0.1, causal, cuda)
    check(kind, d, 70, 600, float(np.log(2.0)) / 8, causal, cuda)
    check(kind, d, 70, 600, 1.0, causal, cuda, scale=1.5)
    check(kind, d, 50, 2100, 1.0, causal, cuda, scale=1.5)
    check(kind, d, 70, 600, 0.1, causal, cuda, views=bnhd)


@pytest.mark.parametrize("kind,d", KINDS)
def test_no_keys(cuda, kind, d):
    q, _, _ = wide_inputs(kind, 1, 2, 5, 1, d, seed=1)
    empty = np.zeros((1, 2, 0, d), dtype=np.float32)
    out, lse = run_wide(kind, q, empty, empty, 0.1, False, cuda, lse=True)
    assert (out == 0).all() and np.isneginf(lse).all()


@pytest.mark.parametrize("kind", ["fp16", "bf16"])
@pytest.mark.parametrize("h,nq,nk", [(512, 16, 455), (300, 100, 97), (100, 130, 200)])
def test_lse_sums_stay_fp32(cuda, kind, h, nq, nk):
    """Key ranges of at most 512 keys sum the unrounded p for the log-sum-exp
    whatever schedule serves the call without it: fp32 rounding of the scores
    and the sum (2^-24 of |lse| ~ 6 and of nk terms), against 2^-12 and more
    for sums of rounded p."""
    q, k, v = wide_inputs(kind, 1, h, nq, nk, 64, seed=h + nk)
    out, lse = run_wide(kind, q, k, v, 0.125, False, cuda, lse=True)
    mx, mean = wide_tol(kind)
    ref = attention_fp32(q, k, v, 0.125, False)
    assert_close_oracle(out, None, None, None, 0.125, False, max_abs=mx, mean_abs=mean, ref=ref)
    assert error_stats(lse, attention_lse(q, k, 0.125, False))[0] <= 1e-5
    out, _ = run_wide(kind, q, k, v, 0.125, False, cuda)
    assert_close_oracle(out, None, None, None, 0.125, False, max_abs=mx, mean_abs=mean, ref=ref)


@pytest.mark.parametrize("kind", ["fp16", "bf16"])
@pytest.mark.parametrize("h,nq,nk,causal", [
    (40, 193, 193, False), (64, 256, 256, True), (96, 129, 129, True), (128, 200, 200, False),
    (160, 192, 192, True), (300, 100, 97, False), (300, 5, 256, True), (600, 130, 130, True)])
def test_one_kernel_with_and_without_lse(cuda, kind, h, nq, nk, causal):
    """The output does not depend on whether the log-sum-exp is asked for: up
    to 256 keys both calls sum the fp32 p (test_lse_sums_stay_fp32), never
    p rounded to 16 bits."""
    import torch

    g = torch.Generator(device="cpu")
    g.manual_seed(h + nq + nk)
    dt = torch.bfloat16 if kind == "bf16" else torch.float16
    q = torch.randn((1, h, nq, 64), generator=g).to(cuda).to(dt)
    k, v = (torch.randn((1, h, nk, 64), generator=g).to(cuda).to(dt) for _ in range(2))
    out, _ = fl.forward_flash2_ex(q, k, v, 0.125, causal, return_lse=True)
    assert torch.equal(out, fl.forward_flash2_ex(q, k, v, 0.125, causal))


@pytest.mark.parametrize("kind", ["fp16", "bf16"])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("h,nq,nk", [(12, 700, 257), (16, 1024, 512), (264, 20, 300),
                                     (16, 700, 400), (16, 700, 200)])
def test_two_groups_per_cu(cuda, kind, causal, h, nq, nk):
    """129-512 keys over one to two 32-row blocks per CU (12 heads of 700 x 257:
    the key quarters): up to two tiles per wave, the second of which raises the
    stabiliser in about half the rows."""
    check(kind, 64, nq, nk, 0.125, causal, cuda, h=h)
    check(kind, 64, nq, nk, 1.0, causal, cuda, scale=1.5, h=h)
