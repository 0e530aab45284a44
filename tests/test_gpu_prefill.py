"""GPU parity of prefill-sized calls (many query tokens per sequence) against the float64
oracle: the orders in which row tiles are dealt over the XCDs, on the dense and the paged
pass, and the 16-bit products on both engines.  Tolerances are the parity tests' own (attn_cases.tol)."""

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


@pytest.mark.parametrize("B,H", [(3, 128), (64, 128), (140, 128), (40, 43)])
def test_paged_f32_decode_by_live_workgroups(ext, B, H):
    """fp32 decode over a work list whose workgroups with an item start all at once (queries
    loaded directly) or follow one another on a CU (B = 140: through the ring)."""
    page, max_pages = 64, 3
    g = torch.Generator().manual_seed(B)
    qa, qr = C.layer_queries(g, B, 1, H)
    table = torch.randperm(B * max_pages, generator=g).reshape(B, max_pages).int()
    ck = torch.randn(B * max_pages, page, D.kv_rank, generator=g)
    pe = torch.randn(B * max_pages, page, D.rope, generator=g)
    wuv = torch.randn(H, D.v, D.kv_rank, generator=g) / math.sqrt(D.kv_rank)
    sl = torch.randint(1, page * max_pages + 1, (B,), generator=g, dtype=torch.int32)
    got = ext.mla_attention_paged(*(gpu(t) for t in (qa, qr, ck, pe, table, sl, wuv)), SCALE).cpu()
    ref = R.mla_attention_paged(qa.double(), qr.double(), ck.double(), pe.double(), table, sl,
                                wuv.double(), SCALE).float()
    torch.testing.assert_close(got, ref, **C.tol(F32, ref))


# ---- the large-tile GEMM engine

def gemm_inputs(M, N, K, dt):
    g = torch.Generator().manual_seed(M + N + K)
    A = torch.randn(M, K, generator=g).to(dt)
    W = (torch.randn(K, N, generator=g) / math.sqrt(K)).to(dt)
    return A, W


@pytest.mark.parametrize("dt", [BF, H16], ids=["bf16", "f16"])
@pytest.mark.parametrize("M,N,K,plan", [
    (256, 256, 1024, "256,256,1"),   # one whole tile
    (257, 264, 96, "256,256,1"),     # a row and a chunk of columns past it, fewer slices than stages
    (40, 200, 32, "256,128,1"),      # one slice, rows and columns off the tile
    (700, 576, 416, "256,128,3"),    # slices 6, 6, 1 of 32 over the splits
    (1332, 1536, 512, "128,128,2"),  # many row tiles, the last of 52 rows
    (130, 392, 224, "128,128,1"),
    (2100, 512, 64, "256,256,1"),    # past one group of eight row tiles
    (4200, 4104, 64, "256,256,1"),   # 289 tiles on 256 workgroups, the last columns' chunk alone
    (2000, 9000, 160, "256,128,1"),  # 568 tiles, slices fewer than stages
    (3300, 4104, 32, "128,128,2"),   # 858 tiles on 512 workgroups (one slice: one split)
])
def test_large_tile_gemm(ext, monkeypatch, dt, M, N, K, plan):
    """Forced large-tile plans against the float64 product of the same 16-bit values (fp32
    sums of K terms of unit total variance: 1e-4 as for the other engines)."""
    A, W = gemm_inputs(M, N, K, dt)
    monkeypatch.setenv("MLA_BGEMM_PLAN", f"{M},{N},{K},1={plan}")
    got = ext.gemm(gpu(A), gpu(W)).cpu()
    ref = (A.double() @ W.double()).float()
    torch.testing.assert_close(got, ref, rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("M", [1, 100, 128, 129, 300, 520])
@pytest.mark.parametrize("N,K", [(576, 7168), (1536, 640), (200, 192)])
def test_16bit_products_by_rule(ext, M, N, K):
    """The plans that the rules pick on both sides of the engines' line (128 rows), short
    products on the tiled engine among them (N = 200), against float64 (see above)."""
    A, W = gemm_inputs(M, N, K, BF)
    got = ext.gemm(gpu(A), gpu(W)).cpu()
    torch.testing.assert_close(got, (A.double() @ W.double()).float(), rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("dt", [BF, H16], ids=["bf16", "f16"])
@pytest.mark.parametrize("M,N,K", [(40, 128, 512), (129, 64, 512), (333, 576, 512), (512, 128, 1536),
                                   (3072, 128, 256), (1540, 2112, 128), (768, 576, 1536)])
def test_16bit_products_short_of_the_large_tiles(ext, dt, M, N, K):
    """Both sides of the line to the tiled engine, against float64 (see above)."""
    A, W = gemm_inputs(M, N, K, dt)
    got = ext.gemm(gpu(A), gpu(W)).cpu()
    torch.testing.assert_close(got, (A.double() @ W.double()).float(), rtol=1e-4, atol=1e-4)


@pytest.mark.parametrize("dt", [BF, H16], ids=["bf16", "f16"])
@pytest.mark.parametrize("B,Sq,per_seq", [(5, 26, True), (3, 87, False), (150, 2, True),
                                           (265, 2, True)])
def test_q_absorbed_many_rows(ext, monkeypatch, dt, B, Sq, per_seq):
    """2a2 on the large tiles with 2b in its epilogue, and 2c from its 16-bit q_nope on them:
    the same bits as 2a2, the 2b launch and 2c on the tiled engine from fp32 q_raw
    (MLA_QUP_FUSE=0: the same 2a1 and 2a2 sums), and the fp32 oracle's result."""
    inp = R.make_inputs(B, Sq, max(Sq, 64), seed=B + Sq, dtype=dt)
    W_uk, _ = R.split_wkv_b(inp["wkv_b"], D.nope)
    pos = inp["positions"]
    if per_seq:
        pos = torch.arange(Sq)[None] + 4900 - 31 * torch.arange(B)[:, None]
    args = [gpu(inp[k]) for k in ("x", "W_q_a", "q_norm_w", "W_q_b")] + [gpu(W_uk.contiguous()),
                                                                        gpu(pos)]
    qa, qr = (t.cpu() for t in ext.q_absorbed(*args, D.nope, D.rope, 1e-6))
    monkeypatch.setenv("MLA_QUP_FUSE", "0")
    qa0, qr0 = (t.cpu() for t in ext.q_absorbed(*args, D.nope, D.rope, 1e-6))
    assert torch.equal(qa, qa0) and torch.equal(qr, qr0)
    f = {k: inp[k].float() for k in ("x", "W_q_a", "q_norm_w", "W_q_b")}
    pick = [0, B // 2, B - 1]
    if per_seq:
        ra, rr = R.prepare_q_ragged(f["x"][pick], f["W_q_a"], f["q_norm_w"], f["W_q_b"],
                                    W_uk.float(), pos[pick], D.nope, D.rope)
    else:
        ra, rr = R.prepare_q_mla_absorbed(f["x"][pick], f["W_q_a"], f["q_norm_w"], f["W_q_b"],
                                          W_uk.float(), pos, D.nope, D.rope)
    torch.testing.assert_close(qa[pick].float(), ra, **C.tol(dt, ra))
    torch.testing.assert_close(qr[pick].float(), rr, **C.tol(dt, rr))


@pytest.mark.parametrize("dt", [BF, H16], ids=["bf16", "f16"])
@pytest.mark.parametrize("B,Sq", [(260, 1), (2, 130), (300, 2), (7, 100)])
def test_out_projection_many_rows(ext, monkeypatch, dt, B, Sq):
    """3d on the large tiles (NT, G = heads) gives the tiled engine's bits (MLA_WGEMM=0)."""
    args = [gpu(t) for t in C.attn_inputs(B, Sq, 140, seed=B, dt=dt)]
    got = ext.mla_attention(*args, SCALE, Sq > 1).cpu()
    monkeypatch.setenv("MLA_WGEMM", "0")
    assert torch.equal(got, ext.mla_attention(*args, SCALE, Sq > 1).cpu())


# ---- the large tiles' 16-bit results and groups

def o_proj_inputs(rows, H, hidden, dt):
    g = torch.Generator().manual_seed(rows + hidden)
    attn = torch.randn(rows, 1, H, D.v, generator=g).to(dt)
    W_o = (torch.randn(H * D.v, hidden, generator=g) / math.sqrt(H * D.v)).to(dt)
    return attn, W_o


@pytest.mark.parametrize("dt", [BF, H16], ids=["bf16", "f16"])
@pytest.mark.parametrize("rows,H,hidden,plan", [
    (129, 8, 264, "256,256,1"), (300, 8, 264, "256,128,1"), (130, 8, 136, "128,128,1"),
    (1332, 8, 1160, "256,256,1"),    # columns a chunk past the tile, rows off it
    (2100, 4, 392, "256,128,1"),     # more tiles than one group of eight row tiles
    (300, 8, 264, "128,128,2"),      # fp32 partials, rounded by the reduction
    (1332, 128, 7168, ""), (300, 128, 7168, ""), (129, 128, 7168, ""),   # the rule's own plans
])
def test_large_tile_16bit_results(ext, monkeypatch, dt, rows, H, hidden, plan):
    """The output projection rounds fp32 sums once to the storage format: within half a unit in
    the last place of the float64 result of the same 16-bit values (bf16: 8 significant bits, a
    unit of 2^-7, half 2^-8 of the value; fp16: 11 bits, 2^-11), and the fp32 sums' own error
    (1e-4, as for the fp32 results above)."""
    attn, W_o = o_proj_inputs(rows, H, hidden, dt)
    if plan:
        monkeypatch.setenv("MLA_BGEMM_PLAN", f"{rows},{hidden},{H * D.v},1={plan}")
    got = ext.o_proj(gpu(attn), gpu(W_o)).cpu().double()[:, 0]
    if rows * hidden * H > 1e8:
        pick = torch.tensor([0, 1, rows // 2, rows - 2, rows - 1])
        got, attn = got[pick], attn[pick]
    ref = attn.double().reshape(attn.shape[0], -1) @ W_o.double()
    torch.testing.assert_close(got, ref, rtol=2.0 ** (-8 if dt == BF else -11), atol=1e-4)


@pytest.mark.parametrize("dt", [BF, H16], ids=["bf16", "f16"])
@pytest.mark.parametrize("H,B,tile", [(12, 2100, "256,256"), (12, 2100, "256,128"),
                                      (128, 1100, "128,128"), (5, 1100, "128,128")])
def test_grouped_large_tiles_many_rows(ext, monkeypatch, dt, H, B, tile):
    """3d with more than eight row tiles, whose groups start at different heads (also where
    their number is no multiple of eight): the tiled engine's bits."""
    args = [gpu(t) for t in C.attn_inputs(B, 1, 70, H=H, seed=B + H, dt=dt)]
    monkeypatch.setenv("MLA_BGEMM_PLAN", f"{B},{D.v},{D.kv_rank},{H}={tile},1")
    got = ext.mla_attention(*args, SCALE).cpu()
    monkeypatch.delenv("MLA_BGEMM_PLAN")
    monkeypatch.setenv("MLA_WGEMM", "0")
    assert torch.equal(got, ext.mla_attention(*args, SCALE).cpu())


@pytest.mark.parametrize("M,N,K", [(300, 576, 7168), (129, 1536, 7168), (520, 1536, 2048)])
def test_f16_products_by_rule(ext, M, N, K):
    A, W = gemm_inputs(M, N, K, H16)
    got = ext.gemm(gpu(A), gpu(W)).cpu()
    torch.testing.assert_close(got, (A.double() @ W.double()).float(), rtol=1e-4, atol=1e-4)
