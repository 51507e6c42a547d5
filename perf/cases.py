"""The work that programs have this library do, as cases that can be timed and
compared: Q8_0 products from one row to a prompt, the MLP block, paged
attention of a decode step and of a prompt, logits with sampling, and a whole
request to a model.  Shapes are those of the library's own configurations (the
0.5B-, 1.5B- and 7B-shaped models), and `draw` gives others of the same
ranges.  Every case goes through the public Context / Model entry points.

Outputs of the canonical schedule are defined to the bit (include/lgx.h), so
their tolerance is "exact"; the binary16 flash attention of the fast prefill
has a measured one.
"""
from __future__ import annotations

import math

import torch

import logicaffeine_amd as lgx

# (hidden, intermediate) of the 0.5B-, 1.5B- and 7B-shaped models
MLPS = {"0.5b": (896, 4864), "1.5b": (1536, 8960), "7b": (3584, 18944)}
# (query heads, KV heads, head dim) of the same
HEADS = {"0.5b": (14, 2, 64), "1.5b": (12, 2, 128), "7b": (28, 4, 128)}
VOCAB = 151936
SIGMA = 0.02                      # of the weights' scales (times 1/127) and the embedding
PAGE = 16

_ctx = None


def _context() -> lgx.Context:
    """One library context for the process, as a serving program keeps it."""
    global _ctx
    if _ctx is None:
        _ctx = lgx.Context(torch.cuda.current_device())
    return _ctx


def listed() -> list:
    return [
        # one token of one user, the smallest product of a decode step
        dict(name="gemv-4864x896", kind="gemm", n=4864, k=896, m=1),
        # one token of one user through an MLP block (weights from memory)
        dict(name="mlp-1.5b-m1", kind="mlp", shape="1.5b", m=1),
        # a small batch of users decoding together
        dict(name="mlp-1.5b-m8", kind="mlp", shape="1.5b", m=8),
        # a full decode batch on the largest product of a 7B-shaped layer
        dict(name="gemm-7b-gateup-m64", kind="gemm", n=37888, k=3584, m=64),
        # a prompt of odd length through the long-K product
        dict(name="gemm-7b-down-m2047", kind="gemm", n=3584, k=18944, m=2047),
        # decode attention: one user far into a long context
        dict(name="attn-decode-7b-b1-l8191", kind="attn", shape="7b", B=1, L=8191, ragged=False),
        # a full batch with the ragged lengths that a server sees
        dict(name="attn-decode-7b-b64-l4096", kind="attn", shape="7b", B=64, L=4096, ragged=True),
        # the small model's heads (d = 64), equal lengths
        dict(name="attn-decode-0.5b-b32-l2048", kind="attn", shape="0.5b", B=32, L=2048,
             ragged=False),
        # a chunk of prompts attending to what is cached, canonical schedule
        dict(name="attn-prefill-7b-b8-p128-l2000", kind="prefill", shape="7b", B=8, P=128, L=2000,
             fast=False),
        # the same kind of chunk in the fast mode, longer
        dict(name="attn-prefill-fast-7b-b16-p256-l4000", kind="prefill", shape="7b", B=16, P=256,
             L=4000, fast=True),
        # logits of a decode batch and the sampled tokens
        dict(name="sample-0.5b-m32", kind="sample", h=896, vocab=VOCAB, m=32),
        # whole requests of a small server's users: prompts, then greedy tokens
        dict(name="request-0.5b-b16-p193-n32", kind="request", B=16, P=193, N=32),
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    """An integer of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["gemm", "gemm", "mlp", "attn", "attn", "prefill", "sample", "request"])
    if kind == "gemm":
        # rows and columns of any layer shape: multiples of 16 and 64
        n = 16 * _log_int(rng, 32, 2368)
        k = 64 * _log_int(rng, 8, 296)
        m = _log_int(rng, 1, 2047)
        top = 2047 * 3584 * 18944
        if n * k * m > top:
            m = max(1, top // (n * k))
        return dict(kind=kind, n=n, k=k, m=m)
    if kind == "mlp":
        return dict(kind=kind, shape=rng.choice(sorted(MLPS)), m=_log_int(rng, 1, 300))
    if kind == "attn":
        B = _log_int(rng, 1, 64)
        return dict(kind=kind, shape=rng.choice(sorted(HEADS)), B=B,
                    L=min(_log_int(rng, 17, 32768), 64 * 4096 // B), ragged=rng.random() < 0.5)
    if kind == "prefill":
        B = _log_int(rng, 1, 16)
        P = _log_int(rng, 2, 256)
        fast = rng.random() < 0.5
        # B P L up to that of the listed chunk of the same mode
        top = 16 * 256 * 4000 if fast else 8 * 128 * 2000
        L = max(P, min(_log_int(rng, P, 4000), top // (B * P)))
        while B * P * L > top:
            B = max(1, B // 2)
        return dict(kind=kind, shape=rng.choice(sorted(HEADS)), B=B, P=P, L=L, fast=fast)
    if kind == "sample":
        return dict(kind=kind, h=rng.choice([896, 896, 1536]), vocab=rng.randint(32000, VOCAB),
                    m=_log_int(rng, 1, 32))
    return dict(kind=kind, B=_log_int(rng, 1, 16), P=_log_int(rng, 12, 193), N=_log_int(rng, 2, 32))


# ---- inputs ---------------------------------------------------------------

def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device="cuda").manual_seed(seed)


def _weights(g, n: int, k: int):
    """Row-major Q8_0 weights: quants, and scales as binary16."""
    qs = torch.randint(-127, 128, (n, k), dtype=torch.int8, device="cuda", generator=g)
    d = torch.randn(n, k // 32, device="cuda", generator=g).abs_().mul_(SIGMA / 127).half()
    return qs, d


def _rows(g, m: int, k: int):
    return torch.randn(m, k, device="cuda", generator=g)


def _gemm_inputs(case, seed):
    g = _gen(seed)
    return _weights(g, case["n"], case["k"]), _rows(g, case["m"], case["k"])


def _mlp_inputs(case, seed):
    h, inter = MLPS[case["shape"]]
    g = _gen(seed)
    return _weights(g, 2 * inter, h), _weights(g, h, inter), _rows(g, case["m"], h)


def _lens(case, seed):
    """Tokens of each sequence (for a prompt chunk: its own rows among them)."""
    B, L = case["B"], case["L"]
    lo = case["P"] if case["kind"] == "prefill" else (max(1, L // 16) if case["ragged"] else L)
    cpu = torch.Generator().manual_seed(seed)
    n = torch.randint(lo, L + 1, (B,), generator=cpu, dtype=torch.int32)
    n[0] = L
    return n


def _attn_inputs(case, seed):
    hq, hkv, d = HEADS[case["shape"]]
    B, maxp = case["B"], -(-case["L"] // PAGE)
    g = _gen(seed)
    rows = B * case.get("P", 1)
    q = torch.randn(rows, hq, d, device="cuda", generator=g)
    pages = torch.empty(2, B * maxp, hkv, PAGE, d, dtype=torch.float16, device="cuda")
    pages.normal_(generator=g)
    table = torch.randperm(B * maxp, device="cuda", generator=g).to(torch.int32).view(B, maxp)
    return q, pages[0], pages[1], table, _lens(case, seed)


def _sample_inputs(case, seed):
    g = _gen(seed)
    emb = torch.empty(case["vocab"], case["h"], dtype=torch.float16, device="cuda")
    emb.normal_(0.0, SIGMA, generator=g)
    pos = torch.randint(0, 4096, (case["m"],), device="cuda", generator=g, dtype=torch.int32)
    return emb, _rows(g, case["m"], case["h"]), pos


def _model_config(case) -> dict:
    """The 0.5B-shaped model, room for the request."""
    hidden, inter = MLPS["0.5b"]
    hq, hkv, d = HEADS["0.5b"]
    return dict(n_layers=24, hidden=hidden, inter=inter, n_heads=hq, n_kv=hkv, head_dim=d,
                vocab=VOCAB, tied=1, max_batch=case["B"], max_seq=512, eps=1e-6, theta=1e6,
                emb_sigma=0.002)


def prepare(case, seed):
    ctx, kind = _context(), case["kind"]
    state = dict(case=case, ctx=ctx)
    if kind == "gemm":
        (qs, d), state["x"] = _gemm_inputs(case, seed)
        state["W"] = ctx.q8_matrix(qs, d.view(torch.int16))
    elif kind == "mlp":
        gu, dn, state["x"] = _mlp_inputs(case, seed)
        state["Wgu"] = ctx.q8_matrix(gu[0], gu[1].view(torch.int16))
        state["Wdn"] = ctx.q8_matrix(dn[0], dn[1].view(torch.int16))
    elif kind in ("attn", "prefill"):
        q, kp, vp, state["table"], lens = _attn_inputs(case, seed)
        state.update(q=q, kp=kp.view(torch.int16), vp=vp.view(torch.int16),
                     lens=(lens - case.get("P", 0)).cuda())
    elif kind == "sample":
        emb, state["x"], state["pos"] = _sample_inputs(case, seed)
        state["t64"] = ctx.f16_repack_t64(emb.view(torch.int16))
        state["seed"] = seed
    else:
        state["model"] = lgx.Model(ctx, _model_config(case), seed)
        state["prompt"] = torch.randint(0, VOCAB, (case["B"], case["P"]), dtype=torch.int32,
                                        device="cuda", generator=_gen(seed))
        state["tok"] = torch.empty(case["B"], dtype=torch.int32, device="cuda")
    return state


# ---- the calls ------------------------------------------------------------

def run(state):
    case, ctx = state["case"], state["ctx"]
    kind = case["kind"]
    if kind == "gemm":
        if case["m"] == 1:
            return ctx.q8q8_gemv_quantize(state["W"], state["x"])
        xq, xd = ctx.quantize_q8_0(state["x"])
        return ctx.q8_gemm(state["W"], xq, xd)
    if kind == "mlp":
        gu, = ctx.q8_gemm_quantize_group([state["Wgu"]], [state["x"]])
        _, aq, ad = ctx.swiglu_quant(gu.view(case["m"], -1), y=False)
        return ctx.q8_gemm(state["Wdn"], aq, ad)
    if kind == "attn":
        return ctx.gqa_decode_attn(state["q"], state["kp"], state["vp"], state["table"],
                                   state["lens"], case["L"])
    if kind == "prefill":
        return ctx.gqa_prefill_attn(state["q"], state["kp"], state["vp"], state["table"],
                                    state["lens"], case["P"], case["L"], fast=case["fast"])
    if kind == "sample":
        logits = ctx.lm_head_f16_t64(state["x"], state["t64"], case["vocab"])
        tokens = ctx.sample(logits, state["pos"], top_k=20, top_p=0.8, temperature=0.7,
                            seed=state["seed"])
        return dict(logits=logits, tokens=tokens)
    m, tok = state["model"], state["tok"]
    m.reset()
    m.prefill(state["prompt"], tok)
    history = torch.empty(case["N"], case["B"], dtype=torch.int32, device=tok.device)
    m.generate(tok, case["N"], history)
    return dict(history=history, logits=m.logits(case["B"]))


# ---- what a pass cannot do without ----------------------------------------

def _q8_bytes(n: int, k: int) -> int:
    return n * k + 2 * n * (k // 32)


def _mean_len(case) -> float:
    if case["kind"] == "prefill":
        return (case["P"] + case["L"]) / 2
    return (max(1, case["L"] // 16) + case["L"]) / 2 if case["ragged"] else case["L"]


def work(case) -> dict:
    kind = case["kind"]
    if kind == "gemm":
        n, k, m = case["n"], case["k"], case["m"]
        return dict(bytes=_q8_bytes(n, k) + 4 * m * (n + k), flops=2 * m * n * k)
    if kind == "mlp":
        (h, inter), m = MLPS[case["shape"]], case["m"]
        return dict(bytes=_q8_bytes(2 * inter, h) + _q8_bytes(h, inter) + 8 * m * h,
                    flops=6 * m * h * inter)
    if kind in ("attn", "prefill"):
        hq, hkv, d = HEADS[case["shape"]]
        P, B, L = case.get("P", 1), case["B"], _mean_len(case)
        attended = L if kind == "attn" else L - (P - 1) / 2
        return dict(bytes=int(B * L * hkv * d * 4 + 8 * B * P * hq * d),
                    flops=int(4 * d * hq * B * P * attended))
    if kind == "sample":
        m, h, v = case["m"], case["h"], case["vocab"]
        return dict(bytes=2 * v * h + 4 * m * (h + v), flops=2 * m * h * v)
    c = _model_config(case)
    B, P, N = case["B"], case["P"], case["N"]
    h, inter, d = c["hidden"], c["inter"], c["head_dim"]
    qkv = (c["n_heads"] + 2 * c["n_kv"]) * d
    macs = h * qkv + h * c["n_heads"] * d + 3 * h * inter
    layer = (_q8_bytes(qkv, h) + _q8_bytes(h, c["n_heads"] * d) + _q8_bytes(2 * inter, h)
             + _q8_bytes(h, inter))
    # the prompt's rows in one pass over the weights, then one pass a token;
    # every step also picks a token from the embedding and reads the cache
    kv = 4 * d * c["n_kv"] * c["n_layers"]
    total = ((1 + N) * (c["n_layers"] * layer + 2 * VOCAB * h)
             + B * kv * (P + sum(P + 1 + i for i in range(N))) + 4 * B * VOCAB)
    rows = B * (P + N)
    attended = B * (P * (P + 1) / 2 + sum(P + 1 + i for i in range(N)))
    flops = (2 * rows * c["n_layers"] * macs + 2 * B * (1 + N) * VOCAB * h
             + 4 * d * c["n_heads"] * c["n_layers"] * attended)
    return dict(bytes=int(total), flops=int(flops))


def tolerance(case):
    if case["kind"] == "prefill" and case["fast"]:
        # binary16 queries and probabilities: 2.6e-4 off the 64-bit result
        return dict(rel=1e-3)
    return "exact"


# ---- the same in 64 bits --------------------------------------------------

def _q8_rows(x):
    """Q8_0 of rows, dequantised: d = amax / 127 stored as binary16, quants
    rounded half away from zero."""
    b = x.double().view(x.shape[0], -1, 32)
    d = b.abs().amax(-1, keepdim=True) / 127
    r = torch.where(d > 0, b / d, torch.zeros_like(b))
    q = (r.abs() + 0.5).floor().copysign(r).clamp_(-127, 127)
    return (q * d.half().double()).view(x.shape[0], -1)


def _dequant(w):
    qs, d = w
    return (qs.double().view(qs.shape[0], -1, 32) * d.double().unsqueeze(-1)).view(qs.shape)


def _dense_rows(pages, table, b: int, n: int):
    """The first n cached rows of sequence b: [heads][n][d] in 64 bits."""
    rows = pages[table[b, :-(-n // PAGE)].long()].double()
    return rows.transpose(0, 1).flatten(1, 2)[:, :n]


def exact(case, seed):
    kind = case["kind"]
    if kind == "gemm":
        w, x = _gemm_inputs(case, seed)
        y = _q8_rows(x) @ _dequant(w).T
        return y[0] if case["m"] == 1 else y
    if kind == "mlp":
        gu, dn, x = _mlp_inputs(case, seed)
        a = _q8_rows(x) @ _dequant(gu).T
        gate, up = a.chunk(2, -1)
        return _q8_rows(gate / (1 + torch.exp(-gate)) * up) @ _dequant(dn).T
    if kind in ("attn", "prefill"):
        hq, hkv, d = HEADS[case["shape"]]
        q, kp, vp, table, lens = _attn_inputs(case, seed)
        P = case.get("P", 1)
        q = q.double().view(case["B"], P, hkv, hq // hkv, d)
        out = torch.empty(case["B"], P, hq, d, dtype=torch.float64, device=q.device)
        for b, n in enumerate(lens.tolist()):
            k, v = (_dense_rows(p, table, b, n) for p in (kp, vp))
            s = torch.matmul(q[b].permute(1, 0, 2, 3).flatten(1, 2),
                             k.transpose(1, 2).contiguous()) / math.sqrt(d)
            s = s.view(hkv, P, hq // hkv, n)
            # row j of the chunk is position n - P + j
            late = torch.arange(n, device=s.device) > torch.arange(n - P, n, device=s.device)[:, None]
            s.masked_fill_(late[None, :, None, :], -math.inf)
            o = torch.matmul(torch.softmax(s, -1).flatten(1, 2), v).view(hkv, P, hq // hkv, d)
            out[b] = o.permute(1, 0, 2, 3).reshape(P, hq, d)
        return out.view(-1, hq, d)
    if kind == "sample":
        emb, x, _ = _sample_inputs(case, seed)
        return dict(logits=x.double() @ emb.double().T, tokens=None)
    return None
