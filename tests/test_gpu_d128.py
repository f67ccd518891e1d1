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
    assert torch.isfinite(o.float()).all(), "unwritten rows"
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


# What the dispatcher launches (asserted on an MI355X seen whole): shapes as
# (heads, N_q, N_k, causal).  Ragged and single-row ends, key ranges of one
# tile (the second stream of a split has none), rows with no visible key.
SHAPES = {
    "br32_rows": [(3, 1, 1, False), (3, 33, 31, True), (3, 65, 64, True), (4, 130, 1025, False),
                  (16, 512, 700, True), (3, 100, 37, True)],
    "br64_bc64_w2x2_slot": [(40, 300, 301, True), (60, 200, 97, False), (120, 65, 31, True),
                            (48, 260, 1000, True), (40, 513, 513, True), (64, 200, 130, False),
                            (256, 40, 4096, False)],
    "br64_bc64_w2x2_pair": [(24, 1025, 1025, True), (24, 1089, 1089, True),
                            (10, 2817, 2817, True)],
    "br128_bc64_w4x2_slot": [(70, 200, 1537, False), (100, 250, 1600, True), (70, 257, 1568, False),
                             (60, 257, 1101, False)],
    "br128_bc64_w4x2_pair": [(12, 4097, 4097, True)],
    "br256_bc64_w8_slot": [(100, 300, 100, False), (512, 33, 4099, True), (300, 40, 4096, False)],
    "br128_bc64_w4_slot": [(300, 100, 97, False), (300, 130, 65, True), (200, 300, 301, True),
                           (50, 450, 450, True)],
}
CASES = [(name, *s) for name, v in SHAPES.items() for s in v]


def assert_launch(name, kind, h, nq, nk, causal, dev):
    """`name` is what a call of this shape launches, where all CUs are seen."""
    import torch

    if torch.cuda.get_device_properties(dev).multi_processor_count != 256:
        return
    base = capi.make_params(1 << 16, 1 << 17, 1 << 18, 1 << 19, 1, h, nq, nk, 128, 0.1, causal)
    qs, ks = (h * nq * 128, nq * 128, 128), (h * nk * 128, nk * 128, 128)
    p = capi.make_params_ex(base, qs, ks, ks, qs)
    assert capi.launch_name(p, capi.DTYPE_BF16 if kind == "bf16" else capi.DTYPE_F16) == name


@pytest.mark.parametrize("kind", ["fp16", "bf16"])
@pytest.mark.parametrize("name,h,nq,nk,causal", CASES)
def test_dispatched_shapes(cuda, kind, name, h, nq, nk, causal):
    assert_launch(name, kind, h, nq, nk, causal, cuda)
    run_shared_kv(kind, h, nq, nk, 128, causal, cuda, seed=h + 7 * nq + nk)


# Scores far above the first tile's best hand the block to the checked pass.
@pytest.mark.parametrize("kind", ["fp16", "bf16"])
@pytest.mark.parametrize("name,i", [("br32_rows", 3), ("br64_bc64_w2x2_slot", 3),
                                    ("br64_bc64_w2x2_pair", 0), ("br128_bc64_w4x2_slot", 1),
                                    ("br128_bc64_w4_slot", 2)])
def test_peaked(cuda, kind, name, i):
    h, nq, nk, causal = SHAPES[name][i]
    assert_launch(name, kind, h, nq, nk, causal, cuda)
    run_shared_kv(kind, h, nq, nk, 128, causal, cuda, seed=h + nq, sm=1.0, qk_scale=2.0)


def test_projection_layout_and_negative_scale(cuda):
    run_shared_kv("bf16", 24, 1025, 1025, 128, True, cuda, seed=5, sm=-0.1, bnhd=True)
    run_shared_kv("bf16", 40, 300, 301, 128, True, cuda, seed=7, sm=-0.1, bnhd=True)
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
