"""Parity of the paged GQA decode attention kernels with the CPU oracle.

The canonical schedule (256-token chunks, sequential score and PV chains,
halving-tree sums, log-sum-exp merge in chunk order) is followed by both, so
outputs are compared bit-for-bit; the float64 golden fixture checks the
north star's 2e-3 tolerance."""
import numpy as np
import pytest

import logicaffeine_amd as lgx

pytestmark = pytest.mark.gpu


def host(t):
    return t.cpu().numpy()


def make_cache(B, hkv, d, lens, seed):
    rng = np.random.default_rng(seed)
    maxp = max(1, -(-max(lens) // 16))
    npages = B * maxp
    k = rng.standard_normal((npages, hkv, 16, d)).astype(np.float16).view(np.uint16)
    v = rng.standard_normal((npages, hkv, 16, d)).astype(np.float16).view(np.uint16)
    pt = rng.permutation(npages).astype(np.int32).reshape(B, maxp)
    return k, v, pt, maxp


def run(ctx, q, k, v, pt, lens, max_seq_len=None):
    lens = np.asarray(lens, np.int32)
    msl = int(max_seq_len or max(1, lens.max()))
    return host(ctx.gqa_decode_attn(ctx.to_device(q), ctx.to_device(k), ctx.to_device(v),
                                    ctx.to_device(pt), ctx.to_device(lens), msl))


def test_golden_fixture(ctx, orc, golden):
    out = run(ctx, golden["attn_q"], golden["attn_k"], golden["attn_v"], golden["attn_pt"],
              golden["attn_lens"])
    ref = orc.gqa_decode_attn(golden["attn_q"], golden["attn_k"], golden["attn_v"],
                              golden["attn_pt"], golden["attn_lens"])
    assert np.array_equal(out, ref)
    f64 = golden["attn_out"]
    assert np.all(np.abs(out - f64) <= 2e-3 * (np.abs(f64) + 1e-2))


@pytest.mark.parametrize("L", [512, 4096, 32768])
def test_config2_uniform_bit_exact(ctx, orc, L):
    B, hq, hkv, d = 16, 12, 2, 128
    lens = [L] * B
    k, v, pt, _ = make_cache(B, hkv, d, lens, seed=L)
    q = orc.gen_normal_f32(2, 10 + L, (B, hq, d))
    out = run(ctx, q, k, v, pt, lens)
    assert np.array_equal(out, orc.gqa_decode_attn(q, k, v, pt, np.asarray(lens, np.int32)))


def test_config2_ragged_long_bit_exact(ctx, orc):
    """Config 2's ragged variant at its batch of 16: lengths uniform in
    [256, 32768], the first at the maximum."""
    B, hq, hkv, d = 16, 12, 2, 128
    lens = list(orc.gen_below_i32(2, 30, 32768 - 256 + 1, (B,)) + 256)
    lens[0] = 32768
    k, v, pt, _ = make_cache(B, hkv, d, lens, seed=3)
    q = orc.gen_normal_f32(2, 31, (B, hq, d))
    out = run(ctx, q, k, v, pt, lens)
    assert np.array_equal(out, orc.gqa_decode_attn(q, k, v, pt, np.asarray(lens, np.int32)))


@pytest.mark.parametrize("d,hq", [(64, 14), (128, 12)])
def test_very_long_context_merge_bit_exact(ctx, orc, d, hq):
    """Contexts past 64 Ki tokens (more than 256 chunks: the merge runs
    several LDS tiles, and more chunks than threads), next to a short one
    and an empty one in the same call."""
    B, hkv = 3, 2
    lens = [70000, 3000, 0]
    k, v, pt, _ = make_cache(B, hkv, d, lens, seed=d + 7)
    q = orc.gen_normal_f32(2, 40 + d, (B, hq, d))
    out = run(ctx, q, k, v, pt, lens)
    assert np.array_equal(out, orc.gqa_decode_attn(q, k, v, pt, np.asarray(lens, np.int32)))
    assert np.all(out[2] == 0.0)


@pytest.mark.parametrize("hq,hkv,d", [(2 * g, 2, d) for d in (64, 128) for g in range(1, 9)]
                         + [(28, 4, 128), (8, 8, 64), (8, 1, 128)])
def test_head_layouts_bit_exact(ctx, orc, hq, hkv, d):
    B = 5
    lens = [1, 16, 255, 257, 1500]
    k, v, pt, _ = make_cache(B, hkv, d, lens, seed=hq * d)
    q = orc.gen_normal_f32(3, hq + d, (B, hq, d))
    out = run(ctx, q, k, v, pt, lens)
    assert np.array_equal(out, orc.gqa_decode_attn(q, k, v, pt, np.asarray(lens, np.int32)))
    # single cached token: the output is that token's V row exactly
    for h in range(hq):
        assert np.array_equal(out[0, h], orc.f16_to_f32(v[pt[0, 0], h // (hq // hkv), 0]))


def test_lengths_clamped_to_max_seq_len(ctx, orc):
    B, hq, hkv, d = 3, 6, 2, 64
    lens = np.array([700, 100, 0], np.int32)
    k, v, pt, maxp = make_cache(B, hkv, d, [700, 700, 700], seed=9)
    q = orc.gen_normal_f32(3, 77, (B, hq, d))
    out = run(ctx, q, k, v, pt, lens, max_seq_len=300)
    ref = orc.gqa_decode_attn(q, k, v, pt, np.minimum(lens, 300))
    assert np.array_equal(out, ref)
    assert np.all(out[2] == 0.0)                      # empty sequence


def test_attention_argument_errors(ctx, orc):
    t = ctx.torch
    q = t.zeros((1, 6, 96), dtype=t.float32, device=ctx.dev)
    pages = t.zeros((4, 2, 16, 96), dtype=t.int16, device=ctx.dev)
    pt = t.zeros((1, 4), dtype=t.int32, device=ctx.dev)
    sl = t.ones(1, dtype=t.int32, device=ctx.dev)
    with pytest.raises(lgx.LgxError) as ei:
        ctx.gqa_decode_attn(q, pages, pages, pt, sl, 16)
    assert ei.value.status_name == "LGX_UNSUPPORTED"
    q = t.zeros((1, 6, 64), dtype=t.float32, device=ctx.dev)
    pages = t.zeros((4, 2, 16, 64), dtype=t.int16, device=ctx.dev)
    with pytest.raises(lgx.LgxError) as ei:
        ctx.gqa_decode_attn(q, pages, pages, pt, sl, 65)
    assert ei.value.status_name == "LGX_OUT_OF_BOUNDS"
    q3 = t.zeros((1, 6, 64), dtype=t.float32, device=ctx.dev)
    pages3 = t.zeros((4, 4, 16, 64), dtype=t.int16, device=ctx.dev)
    with pytest.raises(lgx.LgxError) as ei:                 # 6 / 4 heads
        ctx.gqa_decode_attn(q3, pages3, pages3, pt, sl, 16)
    assert ei.value.status_name == "LGX_INVALID_ARGUMENT"


# ---- prefill: several causal query rows per sequence ----

def prefill_ref(orc, q, k, v, pt, ctx_len, P):
    """Oracle: row b*P + j is a decode query of sequence b at length
    ctx_len[b] + j + 1 (the page table row repeated per query row)."""
    B = len(ctx_len)
    lens = np.array([ctx_len[b] + j + 1 for b in range(B) for j in range(P)], np.int32)
    ptr = np.repeat(pt, P, axis=0)
    return orc.gqa_decode_attn(q, k, v, ptr, lens)


@pytest.mark.parametrize("hq,hkv,d,ctx_len,P", [
    (14, 2, 64, [0, 37], 40),            # fresh sequence + short context, ragged row block
    (28, 4, 128, [0, 200], 72),          # rows cross the first chunk boundary
    (12, 2, 128, [500, 0, 255], 9),      # GQ 6; P not a multiple of the row block
    (8, 8, 64, [3], 257),                # GQ 1, rows spanning two chunks
    (8, 1, 128, [1000], 20),             # GQ 8
])
def test_prefill_attn_bit_exact(ctx, orc, hq, hkv, d, ctx_len, P):
    """Every prefill row equals the decode schedule at its own length."""
    B = len(ctx_len)
    lens_end = [c + P for c in ctx_len]
    k, v, pt, maxp = make_cache(B, hkv, d, lens_end, seed=hq * d + P)
    q = orc.gen_normal_f32(4, hq + d + P, (B * P, hq, d))
    msl = maxp * 16
    out = host(ctx.gqa_prefill_attn(ctx.to_device(q), ctx.to_device(k), ctx.to_device(v),
                                    ctx.to_device(pt), ctx.to_device(np.asarray(ctx_len, np.int32)),
                                    P, msl))
    assert np.array_equal(out, prefill_ref(orc, q, k, v, pt, ctx_len, P))


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("g", range(1, 9))
def test_prefill_attn_head_groups_bit_exact(ctx, orc, g, d):
    """Every head-group size the prefill kernels are built for, with one
    fresh and one cached sequence whose rows cross a chunk boundary."""
    hkv, ctx_len, P = 2, [0, 230], 35
    B, hq = len(ctx_len), 2 * g
    k, v, pt, maxp = make_cache(B, hkv, d, [c + P for c in ctx_len], seed=g * d)
    q = orc.gen_normal_f32(5, g + d, (B * P, hq, d))
    out = host(ctx.gqa_prefill_attn(ctx.to_device(q), ctx.to_device(k), ctx.to_device(v),
                                    ctx.to_device(pt), ctx.to_device(np.asarray(ctx_len, np.int32)),
                                    P, maxp * 16))
    assert np.array_equal(out, prefill_ref(orc, q, k, v, pt, ctx_len, P))


@pytest.mark.parametrize("hq,hkv,d,P", [(14, 2, 64, 21), (28, 4, 128, 5), (2, 2, 128, 33), (9, 3, 64, 1)])
def test_prefill_attn_values_some_rows_do_not_attend_to(ctx, orc, hq, hkv, d, P):
    """Infinite and NaN V rows inside the last rows' reach: rows before them
    keep their finite bits, rows from them on get the oracle's infinities and
    NaN (the 0 weight of a row that ends earlier must not meet such a value).
    One, two and three blocks of query rows, one with a cut at max_seq_len."""
    ctx_len = [0, 250, 37]
    B = len(ctx_len)
    k, v, pt, maxp = make_cache(B, hkv, d, [c + P for c in ctx_len], seed=3 * d + P)
    for b, c in enumerate(ctx_len):
        for pos, val in ((c + P // 2, np.inf), (c + P - 1, np.nan)):
            v[pt[b, pos // 16], :, pos % 16, 3::7] = np.float16(val).view(np.uint16)
    q = orc.gen_normal_f32(6, d + P, (B * P, hq, d))
    msl = 250 + P - 1 if P > 1 else 251        # the second sequence's last row is clamped
    out = host(ctx.gqa_prefill_attn(ctx.to_device(q), ctx.to_device(k), ctx.to_device(v),
                                    ctx.to_device(pt), ctx.to_device(np.asarray(ctx_len, np.int32)),
                                    P, msl))
    lens = np.minimum([c + j + 1 for c in ctx_len for j in range(P)], msl).astype(np.int32)
    ref = orc.gqa_decode_attn(q, k, v, np.repeat(pt, P, axis=0), lens)
    assert np.isfinite(ref).any() and not np.isfinite(ref).all()
    assert np.array_equal(out, ref, equal_nan=True)


@pytest.mark.parametrize("rows", [16, 32])
@pytest.mark.parametrize("d", [64, 128])
def test_prefill_attn_both_block_sizes_bit_exact(monkeypatch, orc, rows, d):
    """16 and 32 (query row, head) pairs per workgroup, every head group: one
    block exactly full, one row more, a block cut by the chunk's end, NaN in a
    V row that only the last query rows attend to."""
    monkeypatch.setenv("LGX_PFA_ROWS", str(rows))
    c = lgx.Context(0)
    try:
        for g in range(1, 9):
            for P in (rows // g, rows // g + 1, 2 * (rows // g) + 1):
                ctx_len = [0, 256 - P // 2, 700]
                k, v, pt, maxp = make_cache(3, 2, d, [n + P for n in ctx_len], seed=g * d + P)
                v[pt[1, (255 + P // 2) // 16], :, (255 + P // 2) % 16, 1::5] = 0x7E00
                q = orc.gen_normal_f32(7, g + d + P, (3 * P, 2 * g, d))
                out = host(c.gqa_prefill_attn(c.to_device(q), c.to_device(k), c.to_device(v), c.to_device(pt),
                                              c.to_device(np.asarray(ctx_len, np.int32)), P, maxp * 16))
                assert np.array_equal(out, prefill_ref(orc, q, k, v, pt, ctx_len, P), equal_nan=True), (g, P)
    finally:
        c.close()


@pytest.mark.parametrize("hkv,g,d,P", [(1, 7, 64, 3), (2, 2, 128, 9), (3, 1, 64, 2), (4, 6, 128, 17), (1, 8, 128, 13),
                                       (5, 3, 64, 4), (1, 4, 64, 33)])
def test_prefill_attn_few_runs_bit_exact(ctx, orc, hkv, g, d, P):
    """One sequence: one to five runs of query blocks per chunk, several
    chunks in a grid row (1, 2, 3 and 4 runs), a first and a last chunk cut."""
    for ctx_len in (1, 250, 1500):
        k, v, pt, maxp = make_cache(1, hkv, d, [ctx_len + P], seed=g * d + hkv + ctx_len)
        q = orc.gen_normal_f32(6, 40 + P + ctx_len, (P, hkv * g, d))
        out = host(ctx.gqa_prefill_attn(ctx.to_device(q), ctx.to_device(k), ctx.to_device(v),
                                        ctx.to_device(pt), ctx.to_device(np.asarray([ctx_len], np.int32)),
                                        P, maxp * 16))
        assert np.array_equal(out, prefill_ref(orc, q, k, v, pt, [ctx_len], P)), ctx_len


def test_prefill_attn_more_chunks_than_a_grid_dimension(ctx, orc):
    """32769 chunks of 6 KV heads (a context of 8.4 million tokens on 64 pages
    in turn): the grid's chunks continue in z."""
    hq, hkv, d, P, ctx_len = 6, 6, 64, 2, 32768 * 256 + 38    # runs of one block: fold 1
    rng = np.random.default_rng(5)
    k, v, _, _ = make_cache(1, hkv, d, [64 * 16], seed=21)
    pt = rng.integers(0, 64, (1, -(-(ctx_len + P) // 16))).astype(np.int32)
    q = orc.gen_normal_f32(4, 31, (P, hq, d))
    out = host(ctx.gqa_prefill_attn(ctx.to_device(q), ctx.to_device(k), ctx.to_device(v),
                                    ctx.to_device(pt), ctx.to_device(np.asarray([ctx_len], np.int32)),
                                    P, ctx_len + P))
    assert np.array_equal(out, prefill_ref(orc, q, k, v, pt, [ctx_len], P))


def extreme_inputs(orc, hq, hkv, d, lens, rows, seed):
    """Cache and query rows that reach every part of binary32 in the two
    chains: binary16-subnormal K and V values and zeros among normal ones,
    query rows so small that products are subnormal or vanish, one large row
    whose scores lie from just below the -87.33 cutoff up to 0 (the
    probabilities near 2^-126 times subnormal V), an infinite and a NaN row."""
    k, v, pt, _ = make_cache(len(lens), hkv, d, lens, seed)
    rng = np.random.default_rng(seed)
    for a in (k, v):
        m = rng.random(a.shape)
        a[m < 0.3] &= 0x83ff                             # subnormal, both signs
        a[m < 0.1] &= 0x8000                             # zeros
    q = orc.gen_normal_f32(8, seed, (rows, hq, d))
    scale = np.float32([1.0, 1e-38, 1e-40, 1e-33])
    q *= scale[rng.integers(0, 4, (rows, hq, 1))]
    # dimension 0 alone decides the scores of these rows: 0 at the first cached
    # token, whose V is 0, and -86.9 to -87.4 elsewhere
    q[1::5] = 0.0
    q[1::5, :, 0] = np.sqrt(d) / 8
    for b, n in enumerate(lens):
        k0 = -(np.float32(695.0) + 4 * rng.random((n, hkv), dtype=np.float32))
        for t in range(n):
            k[pt[b, t // 16], :, t % 16, 0] = k0[t].astype(np.float16).view(np.uint16)
        k[pt[b, 0], :, 0, 0] = 0
        v[pt[b, 0], :, 0] = 0
    q[3, 0, 1] = np.inf
    q[3, -1, 2] = np.nan
    return q, k, v, pt


def assert_bits(out, ref):
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(out), nan)
    assert np.array_equal(out.view(np.uint32)[~nan], ref.view(np.uint32)[~nan])


@pytest.mark.parametrize("hq,hkv,d", [(2, 2, 64), (8, 2, 64), (7, 1, 64), (16, 2, 64), (2, 2, 128), (3, 1, 128),
                                      (8, 2, 128), (7, 1, 128), (8, 1, 128)])
def test_decode_attn_subnormal_infinite_and_nan_operands(ctx, orc, hq, hkv, d):
    """The matrix-instruction chains (and the fmaf forms of few heads) round
    every step like fmaf also where operands, products or sums are subnormal,
    infinite or NaN: chunk tails of 1 to 15 tokens, one and two V stages."""
    lens = [1, 7, 31, 128, 143, 255, 300, 529, 64, 17]
    q, k, v, pt = extreme_inputs(orc, hq, hkv, d, lens, len(lens), seed=hq + d)
    ref = orc.gqa_decode_attn(q, k, v, pt, np.asarray(lens, np.int32))
    fin = np.abs(ref[np.isfinite(ref)])
    assert ((fin > 0) & (fin < 1.17e-38)).any() and np.isnan(ref[3]).any()
    assert_bits(run(ctx, q, k, v, pt, lens), ref)


@pytest.mark.parametrize("rows", [16, 32])
@pytest.mark.parametrize("hq,hkv,d,P", [(2, 2, 64, 40), (7, 1, 64, 9), (8, 1, 128, 9), (2, 2, 128, 35), (6, 2, 128, 21)])
def test_prefill_attn_subnormal_infinite_and_nan_operands(monkeypatch, orc, rows, hq, hkv, d, P):
    """The same through both block sizes of the exact prefill attention, whose
    last token groups hold rows of different lengths."""
    monkeypatch.setenv("LGX_PFA_ROWS", str(rows))
    ctx_len = [0, 250, 19]
    lens = [n + P for n in ctx_len]
    q, k, v, pt = extreme_inputs(orc, hq, hkv, d, lens, 3 * P, seed=hq + d + P)
    ref = prefill_ref(orc, q, k, v, pt, ctx_len, P)
    fin = np.abs(ref[np.isfinite(ref)])
    assert ((fin > 0) & (fin < 1.17e-38)).any() and np.isnan(ref[3]).any()
    c = lgx.Context(0)
    try:
        assert_bits(host(c.gqa_prefill_attn(c.to_device(q), c.to_device(k), c.to_device(v), c.to_device(pt),
                                            c.to_device(np.asarray(ctx_len, np.int32)), P, max(lens))), ref)
    finally:
        c.close()


def test_prefill_attn_config4_shape_sampled(ctx, orc):
    """Config-4 head layout at a 4096-token context: 64 new rows after 4032
    cached tokens (17 chunks), checked on a sample of rows."""
    B, hq, hkv, d, P = 2, 28, 4, 128, 64
    ctx_len = [4032, 1111]
    k, v, pt, maxp = make_cache(B, hkv, d, [c + P for c in ctx_len], seed=77)
    q = orc.gen_normal_f32(4, 99, (B * P, hq, d))
    out = host(ctx.gqa_prefill_attn(ctx.to_device(q), ctx.to_device(k), ctx.to_device(v),
                                    ctx.to_device(pt), ctx.to_device(np.asarray(ctx_len, np.int32)),
                                    P, maxp * 16))
    rows = [0, 1, 31, 63, 64, 100, 127]
    lens = np.array([ctx_len[r // P] + r % P + 1 for r in rows], np.int32)
    ref = orc.gqa_decode_attn(q[rows], k, v, pt[[r // P for r in rows]], lens)
    assert np.array_equal(out[rows], ref)


def test_repeated_calls_changing_lengths_bit_exact(ctx, orc):
    """Call after call with changing lengths (empty, one chunk, many chunks,
    ragged) on one ctx (its workspace reused), for d = 64 and 128: the
    oracle's bits each time, zeros for empty sequences."""
    for d, hq, hkv in ((64, 14, 2), (128, 28, 4)):
        for rep, lens in enumerate(([0, 1, 256, 257, 3000], [2049, 0, 5, 511, 4097],
                                    [7, 7, 7, 7, 7])):
            B = len(lens)
            k, v, pt, _ = make_cache(B, hkv, d, [4097] * B, seed=d + rep)
            q = orc.gen_normal_f32(5, 10 * d + rep, (B, hq, d))
            out = run(ctx, q, k, v, pt, lens, max_seq_len=4097)
            ref = orc.gqa_decode_attn(q, k, v, pt, np.asarray(lens, np.int32))
            assert np.array_equal(out, ref), (d, rep)
            assert np.all(out[np.asarray(lens) == 0] == 0.0)
