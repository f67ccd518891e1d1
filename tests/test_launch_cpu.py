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


# (heads, N_q, N_k, head dim, causal) -> the kernel that measured fastest among
# those that lose no precision there; the figures are beside the rules.
CHOICES = [
    # head dim 64, up to 256 keys
    (30, 64, 64, 64, True, STREAM), (24, 172, 172, 64, True, ROWS32),
    (96, 120, 120, 64, True, STREAM), (64, 234, 234, 64, True, ROWS32),
    (256, 62, 211, 64, False, STREAM), (128, 256, 256, 64, False, STREAM),
    # 257-512 keys
    (18, 299, 299, 64, True, QUARTER), (8, 384, 384, 64, False, QUARTER),
    (25, 300, 300, 64, False, QUARTER), (256, 44, 309, 64, True, QUARTER),
    (32, 337, 337, 64, True, QUARTER), (32, 374, 374, 64, True, ROWS32),
    (32, 510, 510, 64, False, ROWS32), (300, 1, 400, 64, False, ROWS32),
    (64, 512, 512, 64, False, W4),
    # longer ranges
    (28, 276, 5678, 64, True, SPLIT64), (10, 772, 12304, 64, True, ROWS32),
    (128, 146, 3671, 64, True, SPLIT128), (10, 2107, 2107, 64, True, SPLIT128),
    (8, 3000, 3000, 64, True, SPLIT64), (16, 1999, 1999, 64, True, PAIR64),
    (14, 2225, 2225, 64, True, SPLIT128), (6, 3961, 3961, 64, True, PAIR64),
    (28, 515, 515, 64, False, W4), (16, 514, 514, 64, False, SPLIT64),
    (256, 76, 1469, 64, False, W4), (32, 3000, 3000, 64, False, W4),
    # head dim 128
    (18, 330, 330, 128, True, ROWS32), (28, 193, 5712, 128, False, SPLIT64),
    (192, 76, 76, 128, True, W4), (50, 338, 3640, 128, True, SPLIT128),
    (16, 1536, 1536, 128, True, SPLIT64), (12, 2591, 2591, 128, True, SPLIT128),
    (12, 3967, 3967, 128, True, PAIR128), (30, 2053, 2053, 128, True, W4),
    (16, 3000, 3000, 128, True, SPLIT128), (16, 8192, 8192, 128, False, W8),
]


@pytest.mark.parametrize("heads,nq,nk,d,causal,name", CHOICES)
def test_choices(heads, nq, nk, d, causal, name):
    assert launched(heads, nq, nk, d, causal) == name


def test_short_key_ranges_sum_unrounded_p():
    """Up to 512 keys (head dim 64) with at most two 32-row blocks per CU, and
    up to 256 for any count, only kernels whose row sums take the fp32 p."""
    for heads in (1, 7, 16, 25, 64, 100, 255, 256, 300, 511, 512, 1024):
        for nq in (1, 5, 32, 33, 64, 96, 100, 200, 256, 400, 512):
            for nk in (1, 64, 65, 128, 129, 193, 256, 257, 320, 352, 448, 512):
                if nk > 256 and heads * -(-nq // 32) > 512:
                    continue
                for causal in (False, True):
                    for dtype in (capi.DTYPE_F16, capi.DTYPE_BF16):
                        assert launched(heads, nq, nk, 64, causal, dtype=dtype) in (
                            ROWS32, STREAM, QUARTER)
