"""The split-KV plan of fl_attn_fwd_ws as its workspace size (no GPU: the
library plans for 256 CUs)."""

import pytest

from flashlite_amd import capi


def need(dtype, d, heads, nq, nk, causal=False):
    base = capi.make_params(0x10000, 0x20000, 0x30000, 0x40000, 1, heads, nq, nk, d, 0.1, causal)
    qs, ks = (heads * nq * d, nq * d, d), (heads * nk * d, nk * d, d)
    return capi.workspace_bytes(capi.make_params_ex(base, qs, ks, ks, qs), dtype)


@pytest.mark.parametrize("dtype,d", [(capi.DTYPE_F16, 128), (capi.DTYPE_BF16, 64),
                                     (capi.DTYPE_BF16, 128)])
def test_wide_plan(dtype, d):
    row = 4 * (68 if d == 64 else 132)
    keys = 64 if d == 64 else 32
    for heads in (1, 2, 16, 32, 33, 48, 64, 100, 127, 128, 1024):
        for nq in (1, 7, 32, 33, 512):
            for nk in (0, 1, 31, 600, 1024, 1537, 3000, 4096, 16384, 100000):
                b = need(dtype, d, heads, nq, nk, causal=nq > 1)
                if nq > 32 or 2 * heads >= 256 or nk < 20 * keys:
                    assert b == 0
                    continue
                assert b % (heads * nq * row) == 0
                n, tiles = b // (heads * nq * row), -(-nk // keys)
                assert n == 0 or 4 <= n <= 256
                assert n * heads <= 512 and 4 * n <= tiles or n == 0 or n == 8


@pytest.mark.parametrize("dtype,d,heads,nq,nk,chunks", [
    (capi.DTYPE_F16, 128, 16, 1, 4096, 8), (capi.DTYPE_BF16, 64, 16, 1, 4096, 8),
    (capi.DTYPE_BF16, 128, 64, 1, 3000, 4), (capi.DTYPE_BF16, 64, 64, 1, 4096, 4),
    (capi.DTYPE_BF16, 64, 64, 1, 3000, 0), (capi.DTYPE_F16, 128, 2, 32, 16384, 32),
    (capi.DTYPE_BF16, 128, 1, 7, 100000, 195), (capi.DTYPE_F16, 128, 127, 1, 4096, 4)])
def test_wide_chunk_counts(dtype, d, heads, nq, nk, chunks):
    row = 4 * (68 if d == 64 else 132)
    assert need(dtype, d, heads, nq, nk) == chunks * heads * nq * row


def test_fp16_d64_follows_the_split_plan():
    for heads, nq, nk in [(16, 1, 4096), (16, 4, 8192), (1024, 1, 4096), (16, 4096, 4096), (8, 64, 8192)]:
        base = capi.make_params(0x10000, 0x20000, 0x30000, 0x40000, 1, heads, nq, nk, 64, 0.1, False)
        qs, ks = (heads * nq * 64, nq * 64, 64), (heads * nk * 64, nk * 64, 64)
        p = capi.make_params_ex(base, qs, ks, ks, qs)
        assert capi.workspace_bytes(p, capi.DTYPE_F16) == capi.splitkv_workspace_bytes(p, 0)


def test_wide_query_row_strides():
    # at head dim 64 a chunk's Q rows must lie within 32-bit byte offsets
    for d, splits in ((64, False), (128, True)):
        base = capi.make_params(0x10000, 0x20000, 0x30000, 0x40000, 1, 16, 16, 4096, d, 0.1, False)
        ks = (16 * 4096 * d, 4096 * d, d)
        for row, want in ((1 << 24, True), ((1 << 24) + 8, splits), (1 << 27, splits)):
            qs = (16 * d, d, row)
            p = capi.make_params_ex(base, qs, ks, ks, qs)
            assert (capi.workspace_bytes(p, capi.DTYPE_BF16) > 0) == want


def test_refusals():
    assert need(2, 64, 4, 1, 4096) == -1
    assert need(capi.DTYPE_BF16, 80, 4, 1, 4096) == -1
    assert capi.load().fl_attn_fwd_ws(None, 0, None, 0, None) == capi.FL_ERR_INVALID_ARGUMENT
