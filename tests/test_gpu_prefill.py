"""GPU parity of prefill-sized calls (many query tokens per sequence) against the float64
oracle: the orders in which row tiles are dealt over the XCDs, on the dense and the paged
pass.  Tolerances are the parity tests' own (attn_cases.tol)."""

from __future__ import annotations

import math

import pytest
import torch

import attn_cases as C
from oracle import mla_ref as R

pytestmark = pytest.mark.gpu

DEV = "cuda:0"
D = R.DSV3
SCALE = math.sqrt(D.qk_head)
BF, H16, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.fixture(scope="module")
def ext():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a ROCm GPU")
    import mla_custom_cuda
    return mla_custom_cuda


def gpu(t):
    return t.to(DEV)


def oracle(args, causal=True):
    qa, qr, ck, pe, wuv = (t.double() for t in args)
    return R.mla_attention_official(qa, qr, ck, pe, wuv, SCALE, causal=causal).float()


# one batch (every tile in the partial group), a partial group of three, a whole group and
# one left over; H = 40 leaves the last row tile partial
@pytest.mark.parametrize("dt", [BF, H16, F32], ids=["bf16", "f16", "f32"])
@pytest.mark.parametrize("B,Sq,Sk,H", [(1, 130, 300, 128), (3, 45, 77, 128), (9, 16, 150, 128),
                                       (9, 52, 100, 40)])
def test_causal_row_tiles_over_xcds(ext, dt, B, Sq, Sk, H):
    args = C.attn_inputs(B, Sq, Sk, H=H, seed=Sk + B, dt=dt)
    got = ext.mla_attention(*(gpu(t) for t in args), SCALE, True).float().cpu()
    ref = oracle(args)
    torch.testing.assert_close(got, ref, **C.tol(dt, ref))


@pytest.mark.parametrize("dt", [BF, F32], ids=["bf16", "f32"])
@pytest.mark.parametrize("lens", [[200, 77, 130], [64, 300, 16, 150, 65, 40, 90, 210, 128]])
def test_paged_row_tiles_over_xcds(ext, dt, lens):
    B, Sq, page, max_pages = len(lens), 16, 64, 5
    g = torch.Generator().manual_seed(sum(lens))
    qa, qr = (t.to(dt) for t in C.layer_queries(g, B, Sq))
    n_pages = B * max_pages + 3
    table = torch.randperm(n_pages, generator=g)[:B * max_pages].reshape(B, max_pages).int()
    ck = torch.randn(n_pages, page, D.kv_rank, generator=g).to(dt)
    pe = torch.randn(n_pages, page, D.rope, generator=g).to(dt)
    wuv = (torch.randn(D.n_heads, D.v, D.kv_rank, generator=g) / math.sqrt(D.kv_rank)).to(dt)
    sl = torch.tensor(lens, dtype=torch.int32)
    for causal in (True, False):
        got = ext.mla_attention_paged(gpu(qa), gpu(qr), gpu(ck), gpu(pe), gpu(table), gpu(sl),
                                      gpu(wuv), SCALE, causal).float().cpu()
        ref = R.mla_attention_paged(qa.double(), qr.double(), ck.double(), pe.double(), table, sl,
                                    wuv.double(), SCALE, causal=causal).float()
        torch.testing.assert_close(got, ref, **C.tol(dt, ref))
