"""What the dispatcher launches (fl_attn_launch_name), without a GPU: the
library then plans for 256 CUs on 8 XCDs.
"""

import pytest

from flashlite_amd import capi

A = 0x10000
ROWS32, STREAM, QUARTER = "br32_rows", "br256_kv256_w8_stream", "br32_kv512_w4_quarters"
W4, W8 = "br128_bc64_w4_slot", "br256_bc64_w8_slot"
SPLIT64, SPLIT128 = "br64_bc64_w2x2_slot", "br128_bc64_w4x2_slot"
PAIR64, PAIR128 = "br64_bc64_w2x2_pair", "br128_bc64_w4x2_pair"


def params(heads, nq, nk, d=64, causal=False, row=None, lse=0, **kw):
    base = capi.make_params(A, 2 * A, 3 * A, 4 * A, 1, heads, nq, nk, d, 0.1, causal)
    qs, ks = (heads * nq * d, nq * d, row or d), (heads * nk * d, nk * d, d)
    return capi.make_params_ex(base, qs, ks, ks, qs, lse=lse)


def launched(*args, dtype=capi.DTYPE_F16, **kw):
    return capi.launch_name(params(*args, **kw), dtype)


def test_headline_and_small_calls():
    assert launched(16, 4096, 4096) == W8
    assert launched(16, 4096, 4096, causal=True) == PAIR128
    assert launched(16, 512, 512) == ROWS32
    assert launched(1, 128, 128) == ROWS32
    assert launched(1024, 256, 256, causal=True) == STREAM


def test_no_launch_and_refusals():
    assert launched(16, 0, 128) == ""
    assert launched(16, 128, 128, d=80) is None
    assert "head_dim" in capi.last_error()
    assert launched(16, 128, 128, dtype=2) is None
    assert capi.load().fl_attn_launch_name(None, 0) is None


@pytest.mark.parametrize("dtype", [capi.DTYPE_F16, capi.DTYPE_BF16])
def test_lse_does_not_change_the_kernel(dtype):
    for d in (64, 128):
        for heads in (1, 3, 8, 20, 40, 100, 256, 600):
            for nq, nk in ((1, 300), (40, 200), (100, 100), (200, 256), (400, 400), (130, 560),
                           (700, 700), (2048, 2048)):
                for causal in (False, True):
                    args = (heads, nq, nk, d, causal)
                    assert launched(*args, dtype=dtype) == launched(*args, lse=8 * A, dtype=dtype)
