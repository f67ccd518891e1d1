"""Query rows further apart than 32-bit byte offsets reach over a 32-row
block (head dim 64): every schedule that stages Q through LDS reads them by
64-bit addresses.  100M elements between rows: 31 of them are 6.2 GB, so
offsets kept in 32 bits would wrap inside a block.
"""

import pytest

from flashlite_amd import capi
from gpu_util import (PAIR64_CFG, PAIR_CFG, QUARTER_CFG, SLOT_W4_CFG, SLOT_W8_CFG, SPLIT2_CFG,
                      SPLIT2W2_CFG, assert_close_oracle, wide_inputs, wide_tol)
from oracle import attention_fp32

pytestmark = pytest.mark.gpu

STRIDE = (1 << 26) + (1 << 25)
MAX_ROWS = 150


@pytest.fixture(scope="module")
def store():
    """Backing memory of the spread rows (never read as a whole)."""
    import torch

    yield torch.empty((MAX_ROWS - 1) * STRIDE + 300 * 64, dtype=torch.int16, device="cuda:0")
    torch.cuda.empty_cache()


def spread(store, x, dt):
    """x [1, H, N, 64] with STRIDE elements between rows, heads side by side."""
    import torch

    _, h, n, d = x.shape
    t = store.view(dt).as_strided((1, h, n, d), (0, d, STRIDE, 1))
    t.copy_(torch.from_numpy(x))
    return t


def run(kind, tq, k, v, causal, dev, config, splits=None):
    import torch

    dt = tq.dtype
    tk, tv = (torch.from_numpy(x).to(dev).to(dt) for x in (k, v))
    o = torch.full(tq.shape, float("nan"), dtype=dt, device=dev)
    p = capi.tensor_params_ex(tq, tk, tv, o, 0.125, causal)
    stream = torch.cuda.current_stream(dev).cuda_stream
    if splits:
        need = capi.splitkv_workspace_bytes(p, splits)
        ws = torch.empty(need // 4, dtype=torch.float32, device=dev)
        capi.check(capi.fwd_splitkv(p, ws.data_ptr(), need, stream, splits))
    else:
        capi.check((capi.fwd_bf16_ex if kind == "bf16" else capi.fwd_ex)(p, stream, config))
    torch.cuda.synchronize(dev)
    return o


def check(kind, h, nq, nk, causal, dev, store, config, splits=None, same=True):
    import torch

    dt = torch.bfloat16 if kind == "bf16" else torch.float16
    q, k, v = wide_inputs(kind, 1, h, nq, nk, 64, seed=nq + nk)
    far = run(kind, spread(store, q, dt), k, v, causal, dev, config, splits)
    if same:  # one kernel either way: the same bits
        near = run(kind, torch.from_numpy(q).to(dev).to(dt), k, v, causal, dev, config, splits)
        assert torch.equal(far, near)
    mx, mean = wide_tol(kind)
    assert_close_oracle(far.float().cpu().numpy(), None, None, None, 0.125, causal, max_abs=mx,
                        mean_abs=mean, ref=attention_fp32(q, k, v, 0.125, causal))


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("config", [SLOT_W8_CFG, SLOT_W4_CFG, SPLIT2_CFG, SPLIT2W2_CFG, PAIR_CFG,
                                    PAIR64_CFG, QUARTER_CFG])
@pytest.mark.parametrize("kind", ["fp16", "bf16"])
def test_configurations(cuda, store, kind, config, causal):
    """150 rows: two blocks of a pair, a ragged last block."""
    check(kind, 2, 150, 400, causal, cuda, store, config)


@pytest.mark.parametrize("causal", [False, True])
def test_two_block_quarters(cuda, store, causal):
    check("fp16", 135, 40, 300, causal, cuda, store, QUARTER_CFG)


@pytest.mark.parametrize("splits", [2, 5])
def test_chunks(cuda, store, splits):
    check("fp16", 2, 30, 2048, True, cuda, store, -1, splits)


# The dispatcher's kernels by heads (256 CUs) on both sides of 192, 256, 512
# and 576 keys.
@pytest.mark.parametrize("h,nq", [(2, 70), (100, 100), (200, 70), (260, 20), (300, 40)])
@pytest.mark.parametrize("nk", [100, 192, 193, 256, 257, 512, 513, 576, 577])
@pytest.mark.parametrize("kind", ["fp16", "bf16"])
def test_dispatched(cuda, store, kind, h, nq, nk):
    check(kind, h, nq, nk, nk % 2 == 1, cuda, store, -1, same=False)
