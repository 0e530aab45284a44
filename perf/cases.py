"""The work a serving program has this library do, as a list of timed cases.

Everything goes through `mla_custom_cuda`, at the DeepSeek-V3 dimensions that the library's
benchmark and tests use.  A case names an operation:

  q_path     q_absorbed: hidden states -> absorbed queries
  attention  mla_attention / mla_attention_fp8kv over a dense cache
  paged      mla_attention_paged / mla_attention_paged_fp8kv over a ragged, paged cache
  layer      q_absorbed, then mla_attention (the benchmark's layer)
  block      kv_append, q_absorbed, mla_attention, o_proj: one layer's attention block as a
             model runs it; with "page", the paged forms of the same calls

and the sizes: B sequences of Sq new tokens each, over Sk cached keys (the new ones among
them; the longest sequence's where lengths are ragged).  Sq > 1 is causal.
"""

from __future__ import annotations

import math
import os
import random
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "mla-cuda_amd")
if PKG not in sys.path:
    sys.path.insert(0, PKG)

import mla_custom_cuda as mla  # noqa: E402
from mla_inputs import DEEPSEEK_V3 as D  # noqa: E402

DEVICE = "cuda:0"
EPS = 1e-6
SCALE = math.sqrt(D.qk_head)
DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}
PAGE = 64


def case(name, op, dtype, B, Sq, Sk, cache="", page=0):
    """cache: "" for the inputs' type, "fp8" for e4m3 codes; page: keys a page, 0 for dense."""
    return {"name": name, "op": op, "dtype": dtype, "B": B, "Sq": Sq, "Sk": Sk,
            "cache": cache, "page": page}


def listed():
    return [
        # one user's decode step early in a chat: launches and latency
        case("layer_decode_one_f32", "layer", "float32", 1, 1, 512),
        # the headline decode shape, in the reference's own type
        case("layer_decode_serving_f32", "layer", "float32", 128, 1, 4989),
        # the same batch in the type that serving runs in
        case("layer_decode_serving_bf16", "layer", "bfloat16", 128, 1, 4989),
        # a lightly loaded server's whole attention block: weights are most of the bytes
        case("block_decode_small_bf16", "block", "bfloat16", 8, 1, 4989),
        # checking four speculated tokens a sequence, in the other 16-bit type
        case("layer_verify_f16", "layer", "float16", 64, 4, 768),
        # one user with a very long document
        case("attention_decode_long_bf16", "attention", "bfloat16", 1, 1, 65536),
        # the query projections of a prefill chunk
        case("q_path_prefill_bf16", "q_path", "bfloat16", 1, 2048, 2048),
        # the attention of a longer prefill chunk
        case("attention_prefill_bf16", "attention", "bfloat16", 1, 4096, 4096),
        # a batch of chat prompts, in the reference's own type
        case("layer_prefill_chat_f32", "layer", "float32", 8, 512, 512),
        # continuous batching: sequences of all lengths, an odd number of them
        case("paged_decode_bf16", "paged", "bfloat16", 61, 1, 4989, page=PAGE),
        # the same with the cache kept in 8 bits, where long contexts fit more users
        case("paged_decode_fp8", "paged", "bfloat16", 128, 1, 8192, cache="fp8", page=PAGE),
        # chunked prefill into a paged cache beside what is already there, of ragged size
        case("block_chunk_paged_bf16", "block", "bfloat16", 4, 333, 2011, page=PAGE),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _cost(c):
    """A rough time, to keep drawn cases within the listed ones' cost."""
    w = work(c)
    return w["flops"] / (1.2e14 if c["dtype"] == "float32" else 1e15) + w["bytes"] / 4e12


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        op = rng.choice(["q_path", "attention", "paged", "layer", "layer", "block"])
        dtype = rng.choice(["float32", "bfloat16", "bfloat16", "float16"])
        kind = rng.choice(["decode", "decode", "verify", "prefill"])
        if kind == "decode":
            B, Sq, Sk = _log_int(rng, 1, 256), 1, _log_int(rng, 64, 65536)
        elif kind == "verify":
            B, Sq, Sk = _log_int(rng, 1, 128), rng.randint(2, 8), _log_int(rng, 64, 16384)
        else:
            B, Sq = _log_int(rng, 1, 8), _log_int(rng, 64, 4096)
            Sk = Sq + rng.choice([0, _log_int(rng, 64, 8192)])
        cache, page = "", 0
        if op == "paged" or (op == "block" and rng.random() < 0.5):
            page = PAGE
        if op in ("attention", "paged") and dtype == "bfloat16" and rng.random() < 0.5:
            cache = "fp8"
        c = case("", op, dtype, B, Sq, Sk, cache, page)
        del c["name"]
        if _cost(c) <= most and B * Sk * 576 * 4 <= 12e9:
            return c


def lengths(c):
    """Keys of each sequence, the new tokens included: all Sk in a dense cache; in a paged one
    spread evenly up to Sk, the longest Sk."""
    if not c["page"]:
        return [c["Sk"]] * c["B"]
    r = random.Random(c["B"] * 1000003 + c["Sk"])
    return [c["Sk"]] + [r.randint(c["Sq"], c["Sk"]) for _ in range(c["B"] - 1)]


def prepare(c, seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    dt, B, Sq, Sk = DTYPES[c["dtype"]], c["B"], c["Sq"], c["Sk"]

    def normal(*shape, std=1.0, to=dt):
        t = torch.randn(*shape, generator=g, dtype=torch.float32, device=DEVICE)
        return (t.mul_(std) if std != 1.0 else t).to(to)

    def gain(n):
        return (1.0 + 0.1 * torch.randn(n, generator=g, device=DEVICE)).to(dt)

    s = {"case": dict(c)}
    if c["op"] in ("q_path", "layer", "block"):
        s["x"] = normal(B, Sq, D.hidden)
        s["W_q_a"] = normal(D.hidden, D.q_lora, std=D.hidden ** -0.5)
        s["q_norm_w"] = gain(D.q_lora)
        s["W_q_b"] = normal(D.q_lora, D.n_heads * D.qk_head, std=D.q_lora ** -0.5)
        s["W_uk"] = normal(D.n_heads, D.nope, D.kv_rank, std=D.kv_rank ** -0.5)
    else:  # the queries' spread that the projections give
        s["q_absorbed"] = normal(B, Sq, D.n_heads, D.kv_rank, std=math.sqrt(D.nope / D.kv_rank))
        s["q_rope"] = normal(B, Sq, D.n_heads, D.rope)
    if c["op"] == "block":
        s["W_kv_a"] = normal(D.hidden, D.kv_rank + D.rope, std=D.hidden ** -0.5)
        s["kv_norm_w"] = gain(D.kv_rank)
        s["W_o"] = normal(D.n_heads * D.v, D.hidden, std=(D.n_heads * D.v) ** -0.5)

    lens = lengths(c)
    if c["page"]:
        order = torch.randperm(B, generator=g, device=DEVICE).tolist()
        lens = [lens[i] for i in order]
        need = [-(-n // PAGE) for n in lens]
        pool = torch.randperm(sum(need) + 5, generator=g, device=DEVICE).int()
        table = torch.zeros(B, -(-Sk // PAGE), dtype=torch.int32, device=DEVICE)
        at = 0
        for b, n in enumerate(need):
            table[b, :n] = pool[at:at + n]
            at += n
        s["block_table"] = table
        s["seq_lens"] = torch.tensor(lens, dtype=torch.int32, device=DEVICE)
        s["positions"] = torch.tensor([[n - Sq + i for i in range(Sq)] for n in lens],
                                      dtype=torch.int64, device=DEVICE)
        rows = (sum(need) + 5, PAGE)
    else:
        s["positions"] = torch.arange(Sk - Sq, Sk, dtype=torch.int64, device=DEVICE)
        rows = (B, Sk)

    if c["op"] != "q_path":
        s["W_uv"] = normal(D.n_heads, D.v, D.kv_rank, std=D.kv_rank ** -0.5)
        if c["cache"] == "fp8":
            s["kv_scale"] = 6.0 / 448.0
            quantise = lambda t: t.div_(s["kv_scale"]).clamp_(-448.0, 448.0).to(torch.float8_e4m3fn)  # noqa: E731
            s["c_kv"] = quantise(normal(*rows, D.kv_rank, to=torch.float32))
            s["pe"] = quantise(normal(*rows, D.rope, to=torch.float32))
        else:
            s["c_kv"] = normal(*rows, D.kv_rank)
            s["pe"] = normal(*rows, D.rope)
    return s


def run(s):
    c = s["case"]
    causal = c["Sq"] > 1
    if c["op"] == "block":
        if c["page"]:
            mla.kv_append_paged(s["x"], s["W_kv_a"], s["kv_norm_w"], s["positions"],
                                s["block_table"], s["c_kv"], s["pe"], EPS)
        else:
            mla.kv_append(s["x"], s["W_kv_a"], s["kv_norm_w"], s["positions"], s["c_kv"],
                          s["pe"], c["Sk"] - c["Sq"], EPS)
    if c["op"] in ("q_path", "layer", "block"):
        qa, qr = mla.q_absorbed(s["x"], s["W_q_a"], s["q_norm_w"], s["W_q_b"], s["W_uk"],
                                s["positions"], D.nope, D.rope, EPS)
        if c["op"] == "q_path":
            return {"q_absorbed": qa, "q_rope": qr}
    else:
        qa, qr = s["q_absorbed"], s["q_rope"]
    if c["page"] and c["cache"] == "fp8":
        attn = mla.mla_attention_paged_fp8kv(qa, qr, s["c_kv"], s["pe"], s["block_table"],
                                             s["seq_lens"], s["kv_scale"], s["W_uv"], SCALE,
                                             causal)
    elif c["page"]:
        attn = mla.mla_attention_paged(qa, qr, s["c_kv"], s["pe"], s["block_table"],
                                       s["seq_lens"], s["W_uv"], SCALE, causal)
    elif c["cache"] == "fp8":
        attn = mla.mla_attention_fp8kv(qa, qr, s["c_kv"], s["pe"], s["kv_scale"], s["W_uv"],
                                       SCALE, causal)
    else:
        attn = mla.mla_attention(qa, qr, s["c_kv"], s["pe"], s["W_uv"], SCALE, causal)
    if c["op"] == "block":
        return {"attn": attn, "out": mla.o_proj(attn, s["W_o"]), "c_kv": s["c_kv"],
                "pe": s["pe"]}
    if c["op"] == "layer":
        return {"q_absorbed": qa, "q_rope": qr, "attn": attn}
    return attn


def work(c):
    size = 4 if c["dtype"] == "float32" else 2
    key = D.kv_rank + D.rope
    T, H, Sq = c["B"] * c["Sq"], D.n_heads, c["Sq"]
    lens = lengths(c)
    nbytes, flops = 0, 0
    q_bytes = T * H * key * size
    if c["op"] in ("q_path", "layer", "block"):
        q_weights = (D.hidden * D.q_lora + D.q_lora * H * D.qk_head + H * D.nope * D.kv_rank)
        nbytes += (q_weights + T * D.hidden) * size
        flops += 2 * T * q_weights
    if c["op"] != "block":  # the absorbed queries are an input or an output of the pass
        nbytes += q_bytes
    if c["op"] == "q_path":
        return {"bytes": nbytes, "flops": flops}
    keys = sum(lens)
    pairs = Sq * keys - c["B"] * (Sq * (Sq - 1) // 2)  # (query, visible key)
    nbytes += keys * key * (1 if c["cache"] == "fp8" else size)
    nbytes += (H * D.v * D.kv_rank + T * H * D.v) * size
    flops += 2 * pairs * H * (key + D.kv_rank) + 2 * T * H * D.v * D.kv_rank
    if c["op"] == "block":
        more = D.hidden * key + H * D.v * D.hidden
        nbytes += (more + T * (key + D.hidden)) * size
        flops += 2 * T * more
    return {"bytes": nbytes, "flops": flops}


def tolerance(c):
    # About four times the distance from 64 bits that each kind of pass shows.
    if c["dtype"] == "float32":
        return {"rel": 1e-5, "max": 4e-4}
    if c["dtype"] == "float16":
        return {"rel": 2e-3, "max": 6e-2}
    return {"rel": 1.6e-2, "max": 3e-1}


def _rms(t, w):
    return t * torch.rsqrt(t.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rotate(t, positions):
    """Interleaved pairs of t [B, Sq, n, rope] rotated by the tokens' positions, with the
    float32 frequencies and angles that the operation is defined by."""
    inv = 1.0 / 10000 ** (torch.arange(0, D.rope, 2, dtype=torch.float32) / D.rope)
    pos = positions if positions.dim() == 2 else positions[None]
    a = (pos[..., None].float() * inv.to(pos.device)).double()[:, :, None]
    even, odd = t[..., 0::2], t[..., 1::2]
    return torch.stack((even * a.cos() - odd * a.sin(), even * a.sin() + odd * a.cos()),
                       -1).flatten(-2)


def exact(c, seed):
    s = prepare(c, seed)
    B, Sq, H = c["B"], c["Sq"], D.n_heads
    T = B * Sq
    out = {}
    if c["op"] == "block":
        kv = s["x"].double().view(T, -1) @ s["W_kv_a"].double()
        lat = _rms(kv[:, :D.kv_rank], s["kv_norm_w"]).view(B, Sq, -1)
        rot = _rotate(kv[:, D.kv_rank:].view(B, Sq, 1, -1), s["positions"]).view(B, Sq, -1)
        ck, pe = s["c_kv"].double(), s["pe"].double()
        if c["page"]:
            page = s["block_table"].long().gather(1, s["positions"] // PAGE)
            ck[page, s["positions"] % PAGE] = lat
            pe[page, s["positions"] % PAGE] = rot
        else:
            ck[:, c["Sk"] - Sq:] = lat
            pe[:, c["Sk"] - Sq:] = rot
        out["c_kv"], out["pe"] = ck, pe
    elif c["op"] != "q_path":
        ck, pe = s["c_kv"], s["pe"]
    if c["op"] in ("q_path", "layer", "block"):
        lat = _rms(s["x"].double().view(T, -1) @ s["W_q_a"].double(), s["q_norm_w"])
        q = (lat @ s["W_q_b"].double()).view(B, Sq, H, D.qk_head)
        nope = q[..., :D.nope].reshape(T, H, D.nope).transpose(0, 1).contiguous()
        qa = torch.matmul(nope, s["W_uk"].double()).transpose(0, 1).reshape(B, Sq, H, D.kv_rank)
        qr = _rotate(q[..., D.nope:], s["positions"])
        if c["op"] != "block":
            out["q_absorbed"], out["q_rope"] = qa, qr
        if c["op"] == "q_path":
            return out
    else:
        qa, qr = s["q_absorbed"].double(), s["q_rope"].double()

    attn = torch.empty(B, Sq, H, D.v, dtype=torch.float64, device=DEVICE)
    w_uv = s["W_uv"].double().transpose(1, 2).contiguous()
    lens = s["seq_lens"].tolist() if c["page"] else lengths(c)
    for b, n in enumerate(lens):
        if c["page"]:
            k = torch.arange(n, device=DEVICE)
            row = s["block_table"][b].long()[k // PAGE], k % PAGE
            v, r = ck[row] if c["cache"] != "fp8" else ck.view(torch.uint8)[row].view(ck.dtype), \
                pe[row] if c["cache"] != "fp8" else pe.view(torch.uint8)[row].view(pe.dtype)
        else:
            v, r = ck[b], pe[b]
        if c["cache"] == "fp8":
            v, r = v.float().double() * s["kv_scale"], r.float().double() * s["kv_scale"]
        v, r = v.double(), r.double()
        keys = torch.cat((v, r), -1).t().contiguous()
        step = max(1, (1 << 27) // (H * n))
        for i in range(0, Sq, step):
            rows = min(step, Sq - i)
            q = torch.cat((qa[b, i:i + rows], qr[b, i:i + rows]), -1).view(rows * H, -1)
            p = (q @ keys).div_(SCALE).view(rows, H, n)
            if Sq > 1:
                hidden = (torch.arange(n, device=DEVICE)[None]
                          > torch.arange(n - Sq + i, n - Sq + i + rows, device=DEVICE)[:, None])
                p.masked_fill_(hidden[:, None], float("-inf"))
            ctx = (torch.softmax(p, -1).view(rows * H, n) @ v).view(rows, H, -1)
            attn[b, i:i + rows] = torch.matmul(ctx.transpose(0, 1).contiguous(),
                                               w_uv).transpose(0, 1)
    if c["op"] == "block":
        out["out"] = (attn.view(T, -1) @ s["W_o"].double()).view(B, Sq, -1)
    if c["op"] in ("layer", "block"):
        out["attn"] = attn
        return out
    return attn
