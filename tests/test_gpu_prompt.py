"""Kernels that prompt-sized steps take, at the edges of their tiles and spans."""
import numpy as np
import pytest

import oracle
from numerics import assert_bf16_close

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hb(bridge):
    import hip_bridge.quant  # noqa: F401

    return bridge


def test_pack_tables_prompt_rows(hb):
    """Rows longer than the workgroup beside empty and one-token rows, first and last too."""
    from hip_bridge import DeviceBuffer

    rng = np.random.default_rng(12)
    row_tokens = np.array([0, 1, 2500, 0, 0, 1023, 1, 1025, 0], np.int32)
    rows, max_pages, page = len(row_tokens), 200, 16
    positions = rng.integers(0, max_pages * page - 2500, rows).astype(np.int32)
    bt = rng.permutation(rows * max_pages).reshape(rows, max_pages).astype(np.int32)
    n = int(row_tokens.sum())
    d = [DeviceBuffer.from_array(a) for a in (row_tokens, positions, bt)]
    out = {k: DeviceBuffer(4 * m) for k, m in (("cu_seqlens", rows + 1), ("token_row", n), ("token_pos", n),
                                              ("kv_slot", n), ("context", rows), ("status", 1))}
    print("case: pack prompt rows", flush=True)
    hb.pack_tables(d[0], d[1], d[2], max_pages, rows, page, *out.values())
    hb.synchronize()
    want = oracle.pack_tables(row_tokens, positions, bt, page)
    assert out["status"].download(np.int32, 1)[0] == 0
    for k in ("cu_seqlens", "token_row", "token_pos", "kv_slot", "context"):
        assert np.array_equal(out[k].download(np.int32, len(want[k])), want[k]), k


# tokens around the 16-token span and the 64-token span group; histories in the
# first span's rows, across its end, in a later span, and past the row's tokens
@pytest.mark.parametrize("in_place", [True, False])
@pytest.mark.parametrize("heads", [(16, 32), (2, 4)])
def test_gdn_prep_spans_equal_the_row_walk(hb, heads, in_place):
    """The span form gives the bits of the form that walks a row (which input
    rows with an odd stride still take): outputs and the rewritten window."""
    from hip_bridge import DeviceBuffer

    hk, hv = heads
    dk, conv, most = 128, 4, 300
    C = 2 * hk * dk + hv * dk
    T = np.array([1, 15, 16, 17, 64, 65, 300, 0, 80, 130], np.int32)
    hist = np.array([0, 300, 16, 14, 20, 64, 17, 5, 80, 62], np.int32)
    rows, n = len(T), int(T.sum())
    rng = np.random.default_rng(hk + in_place)
    bits = lambda *shape: hb.quant.bf16_bits(rng.standard_normal(shape, dtype=np.float32))  # noqa: E731
    slots = rows if in_place else 2 * rows
    win = bits(slots, conv - 1 + most, C)
    src = np.arange(rows, dtype=np.int32)
    dst = src if in_place else src + rows
    wide = np.zeros((n, C + 1), np.uint16)
    wide[:, :C] = bits(n, C)
    ab = bits(n, 2 * hv)
    cu = np.concatenate([[0], np.cumsum(T)]).astype(np.int32)
    conv_w = (rng.standard_normal((C, conv)) * 0.5).astype(np.float32)
    alog, dt = rng.uniform(0, 1, hv).astype(np.float32), rng.standard_normal(hv).astype(np.float32) * 0.1
    got = []
    for ld in (C, C + 1):
        d = [DeviceBuffer.from_array(a) for a in (np.ascontiguousarray(wide[:, :ld]), ab, conv_w, alog, dt, win, hist,
                                                  src, dst, cu)]
        out = [DeviceBuffer(n * w * 4) for w in (hk * dk, hk * dk, hv * dk, hv, hv)]
        print(f"case: gdn prep heads={heads} in_place={in_place} ld={ld}", flush=True)
        hb.call("hb_gdn_prep", d[0], ld, d[1], hb._p(d[1].ptr + 2 * hv), 2 * hv, d[2], d[3], d[4], d[5], d[6], d[7],
                d[8], d[9], rows, hk, hv, dk, dk, conv, most, *out, None)
        hb.synchronize()
        got.append([o.download(np.uint32, n * w) for o, w in zip(out, (hk * dk, hk * dk, hv * dk, hv, hv))]
                   + [d[5].download(np.uint16, win.shape)])
    for name, a, b in zip(("q", "k", "v", "decay", "beta", "window"), *got):
        assert np.array_equal(a, b), f"{name}: {int(np.sum(a != b))} values differ"


# prompt rows beside decode rows, at the prompt kernel's edges: 64 tokens (its
# least), 16-token blocks and 32-key tiles full and one over, keys before the
# prompt, rows on both sides of the rule that leaves few tokens over many keys to
# the splits, a row without keys, a lone row (no split launches), head groupings of
# 1 and 8
@pytest.mark.parametrize("T,ctx", [
    ([64, 1, 63, 130, 4], [64, 500, 70, 333, 4]),
    ([97, 80, 64], [97, 607, 32 * 5]),
    ([64, 64, 390, 383], [512, 513, 3200, 3100]),
    ([64, 2, 64], [0, 300, 65]),
    ([129], [129]),
    ([65], [1000]),
])
@pytest.mark.parametrize("hq,hkv", [(16, 2), (2, 2)])
def test_paged_attention_prompt_rows(hb, T, ctx, hq, hkv):
    from hip_bridge import DeviceBuffer

    dim, page, split = 256, 16, 256
    rng = np.random.default_rng(sum(T) + hq)
    rows, tokens, most, width = len(T), sum(T), max(T), max(ctx)
    max_pages = (width + page - 1) // page
    bt = rng.permutation(rows * max_pages).reshape(rows, max_pages).astype(np.int32)
    bits = lambda *shape, std=1.0: hb.quant.bf16_bits(rng.standard_normal(shape, dtype=np.float32) * np.float32(std))  # noqa: E731
    kc, vc = bits(rows * max_pages, hkv, page, dim), bits(rows * max_pages, hkv, page, dim)
    q, qg = bits(tokens, hq, dim, std=3.0), bits(tokens, hq, 2 * dim)
    cu = np.concatenate([[0], np.cumsum(T)]).astype(np.int32)
    full = np.maximum(ctx, T).astype(np.int32)  # the oracle's context of a row without keys, whose output is zeros
    obt = bt if full.max() <= max_pages * page else np.tile(bt, 2)
    val = hb.quant.bf16_value
    want = oracle.paged_attention(val(q), val(kc), val(vc), obt, cu, full, 1 / 16, gate=val(qg)[:, :, dim:].copy())
    for r in range(rows):
        if ctx[r] == 0:
            want[cu[r]:cu[r + 1]] = 0.0
    up = DeviceBuffer.from_array
    nwo = hb.attn_workspace_floats(rows, hkv, dim, most, hq // hkv, width, split)
    dev = [up(a) for a in (q, kc, np.ascontiguousarray(vc.transpose(0, 1, 3, 2)), bt, cu, np.asarray(ctx, np.int32),
                           np.repeat(np.arange(rows, dtype=np.int32), T), qg)]
    wo, wml, out = DeviceBuffer(4 * nwo), DeviceBuffer(4 * nwo // dim * 2 + 256), DeviceBuffer(tokens * hq * dim * 2)
    print(f"case: prompt attention T={T} ctx={ctx} heads {hq}/{hkv}", flush=True)
    hb.paged_attention(dev[0], dev[1], dev[2], dev[3], max_pages, dev[4], dev[5], dev[6], dev[7], hq * 2 * dim, rows,
                       tokens, most, width, hq, hkv, dim, 1 / 16, split, wo, wml, out)
    hb.synchronize()
    got = val(out.download(np.uint16, (tokens, hq, dim)))
    for r in range(rows):  # each row by its own scale
        sl = slice(cu[r], cu[r + 1])
        if ctx[r] == 0:
            assert not got[sl].any(), f"row {r} has no keys"
        else:
            assert_bf16_close(got[sl], want[sl], f"row {r}: {T[r]} tokens, context {ctx[r]}")


def test_paged_attention_prompt_sink(hb):
    """One key far above all later ones (by about 2^170 in weight): the later
    keys' reference may not lift it out of range, and the rows see it alone."""
    from hip_bridge import DeviceBuffer

    dim, page, T, split = 256, 16, 1100, 256
    rng = np.random.default_rng(3)
    pages = (T + page - 1) // page
    k = np.zeros((pages, 1, page, dim), np.float32)
    k[..., 0] = -1.0
    k[0, 0, 0, 0] = 1.0
    v = rng.standard_normal((pages, 1, page, dim)).astype(np.float32)
    q = np.zeros((T, 1, dim), np.float32)
    q[..., 0] = 60.0  # scores +60 and -60 at scale 1
    bits, up = hb.quant.bf16_bits, DeviceBuffer.from_array
    qg = np.zeros((T, 1, 2 * dim), np.float32)  # gate 1/2
    nwo = hb.attn_workspace_floats(1, 1, dim, T, 1, T, split)
    wo, wml, out = DeviceBuffer(4 * nwo), DeviceBuffer(4 * nwo // dim * 2 + 256), DeviceBuffer(T * dim * 2)
    print("case: prompt attention with a sink key", flush=True)
    hb.paged_attention(up(bits(q)), up(bits(k)), up(np.ascontiguousarray(bits(v).transpose(0, 1, 3, 2))),
                       up(np.arange(pages, dtype=np.int32)[None]), pages, up(np.array([0, T], np.int32)),
                       up(np.array([T], np.int32)), up(np.zeros(T, np.int32)), up(bits(qg)), 2 * dim, 1, T, T, T, 1, 1,
                       dim, 1.0, split, wo, wml, out)
    hb.synchronize()
    got = hb.quant.bf16_value(out.download(np.uint16, (T, dim)))
    want = np.repeat(0.5 * hb.quant.bf16_value(bits(v))[0, 0, :1], T, 0)
    assert_bf16_close(got, want, "sink")


# one token more than the streamed projection takes, last blocks of 1, 33, 96 and
# 65 tokens, K of a single group pair, of no whole number of 16 groups, and of the
# output projections (fewer than 160 blocks stay with the older kernels, whose
# codes' offset is 128 and whose bound is not this one)
@pytest.mark.parametrize("M,N,K", [(257, 13824, 128), (321, 10240, 2048), (1920, 2048, 4096), (833, 4608, 1152)])
def test_qmm_blocks(hb, M, N, K):
    """The block form (more than 256 tokens, 160 blocks) in every output mode, rows wider than
    N, against float64. f32 outputs: each of the K / 64 <= 64 group terms is
    rounded at 2^-24 of a partial sum of at most some 16 times the output's rms
    (the codes' offset of 16 against their spread of 4.6): 64 * 2^-24 * 4 = 1.5e-5
    of the rms at the worst; bf16: 2^-8 of the value more."""
    from hip_bridge import DeviceBuffer

    rng = np.random.default_rng(M + K)
    x, packed, s, b = hb.quant.qgemv_workload(M, N, K, seed=M + N)
    tw = hb.TiledWeight(packed, s, b)
    val = hb.quant.bf16_value
    codes = ((packed[:, :, None] >> (4 * np.arange(8, dtype=np.uint32))) & 15).reshape(N, K).astype(np.float64)
    w = codes * np.repeat(val(s).astype(np.float64), 64, 1) + np.repeat(val(b).astype(np.float64), 64, 1)
    want = val(x).astype(np.float64) @ w.T
    rms = np.sqrt(np.mean(want * want))
    ldy = N + 32
    init = rng.standard_normal((M, ldy)).astype(np.float32)
    dx = DeviceBuffer.from_array(x)
    for mode in (0, 1, 2):
        print(f"case: block qmm {M}x{N}x{K} mode {mode}", flush=True)
        dy = DeviceBuffer.from_array(init)
        hb.qmm(dx, tw.w, tw.sb, None, dy, M, N, K, ldy=ldy, out_mode=mode)
        hb.synchronize()
        if mode == 0:
            got = val(dy.download(np.uint16, (M, ldy)))[:, :N].astype(np.float64)
            assert np.all(np.abs(got - want) <= 2.0**-8 * np.abs(want) + 1.5e-5 * rms), np.abs(got - want).max() / rms
            continue
        got = dy.download(np.float32, (M, ldy))
        assert np.array_equal(got[:, N:], init[:, N:]), "columns past N untouched"
        base = init[:, :N].astype(np.float64) if mode == 2 else 0.0
        err = np.abs(got[:, :N] - (want + base)).max() / rms
        print(f"  max error / rms {err:.2e}")
        assert err < 1.5e-5


# 301 tokens: about 75, 38 and 9 rows per expert (tiles of three, two and one
# 32-row products), a shared expert of three full tiles and one of 13 rows
@pytest.mark.parametrize("experts", [8, 16, 64])
def test_engine_prompt_matches_oracle(bridge, experts):
    """A prompt step past the streaming kernels' 256 tokens, layer by layer
    against the oracle: the MoE block form beside prompt attention and the
    chunked recurrence, then one decode step on the state it left."""
    from hip_bridge.engine import Engine, tiny_config
    from layer_check import Row, check_layers
    from oracle.model import HybridModel

    cfg = tiny_config(layers=2, interval=2, experts=experts)
    e = Engine(cfg, 2, 512, 260, 301, seed=experts, mtp=False)
    try:
        e.trace(True)
        model = HybridModel(cfg.dims(), e.export)
        model.tie_window = 2e-3
        rng = np.random.default_rng(experts)
        seqs = [rng.integers(0, cfg.vocab, n).astype(np.uint32) for n in (260, 41)]
        print(f"case: engine prompt of 301 tokens, {experts} experts", flush=True)
        e.forward([260, 41], [0, 0], [0, 1], np.concatenate(seqs), logit_rows=[259, 300])
        trace, mid, logits = e.read("trace", 301), e.read("mid_trace", 301), e.read("logits", 2)
        rows = []
        for r, (a, b) in enumerate(((0, 260), (260, 301))):
            row = Row(cfg.layers, cfg.hidden)
            row.extend(trace[:, a:b], mid[:, a:b])
            check_layers(model, row, b - a, seqs[r], f"row {r}")
            assert_bf16_close(logits[r], model.head(row.x[cfg.layers][-1:])[1][0], f"logits row {r}")
            rows.append(row)
        nxt = rng.integers(0, cfg.vocab, 2).astype(np.uint32)
        e.forward([1, 1], [260, 41], [0, 1], nxt, hist_off=[260, 41], logit_rows=[0, 1])
        trace, mid = e.read("trace", 2), e.read("mid_trace", 2)
        for r in range(2):
            rows[r].extend(trace[:, r:r + 1], mid[:, r:r + 1])
            check_layers(model, rows[r], 1, np.append(seqs[r], nxt[r]), f"decode after row {r}")
    finally:
        e.close()


@pytest.mark.parametrize("last", [40, 304])
def test_engine_step_of_two_moe_chunks(bridge, last):
    """More tokens than one MoE chunk takes (4096), the rest in the decode form or
    the block form: every row as in a step of its own. A token whose routing is
    nearly tied may go to another expert there; 1 in 100 is allowed for."""
    from hip_bridge.engine import Engine, tiny_config

    cfg = tiny_config(layers=1, interval=2, context=2048)
    lens = [1400, 1400, 1296 - 8, last + 8]
    e = Engine(cfg, 4, 2048, 1400, sum(lens), seed=5, mtp=False)
    try:
        rng = np.random.default_rng(last)
        seqs = [rng.integers(0, cfg.vocab, n).astype(np.uint32) for n in lens]
        print(f"case: engine step of {sum(lens)} tokens", flush=True)
        e.forward(lens, [0] * 4, [0, 1, 2, 3], np.concatenate(seqs))
        got = e.read("hidden", sum(lens)).copy()
        at = 0
        for r, s in enumerate(seqs):
            e.forward([len(s)], [0], [r], s)
            want = e.read("hidden", len(s))
            rms = np.sqrt(np.mean(want * want))
            off = (np.abs(got[at:at + len(s)] - want).max(1) > 2e-2 * (np.abs(want).max(1) + rms)).mean()
            assert off <= 0.01, f"row {r}: {off:.3f} of the tokens differ"
            at += len(s)
    finally:
        e.close()


@pytest.mark.parametrize("vocab", [8193, 16384, 64 * 8192 + 1, 151936])
def test_argmax_chunk_edges(hb, vocab):
    """The two-level selection at its chunk edges: winner and runner-up on either
    side of one, ties across waves and chunks, a row of equal values, a row of
    -inf, a NaN, and more chunks than a wave has lanes."""
    from hip_bridge import DeviceBuffer

    rng = np.random.default_rng(vocab)
    rows, ld = 7, vocab + 3
    x = rng.standard_normal((rows, ld)).astype(np.float32)
    x[0, 8191], x[0, 8192] = 9.0, 8.5
    x[1, vocab - 1] = x[1, 63] = x[1, 64] = 9.0
    x[2] = 1.25
    x[3] = -np.inf
    x[4, vocab - 1] = np.nan
    x[5, 0], x[5, vocab - 1] = 7.5, 9.0
    x[:, vocab:] = 1e30  # past the vocabulary
    dx = DeviceBuffer.from_array(x)
    ws = DeviceBuffer(int(hb.load().hb_argmax_workspace_bytes(rows, vocab)))
    w, m, s = (DeviceBuffer(4 * rows) for _ in range(3))
    print(f"case: argmax vocab {vocab}", flush=True)
    hb.call("hb_argmax_margin", dx, ld, rows, vocab, w, m, s, ws, None)
    hb.synchronize()
    win, margin, status = w.download(np.uint32, rows), m.download(np.float32, rows), s.download(np.int32, rows)
    for r in range(rows):
        # total order: NaN above all; equal values, -inf among them, by the lower index
        best = int(np.argmax(x[r, :vocab])) if r not in (3, 4) else {3: 0, 4: vocab - 1}[r]
        want = best, np.nan if r in (3, 4) else x[r, best] - np.delete(x[r, :vocab], best).max()
        assert win[r] == want[0], (r, win[r], want)
        assert margin[r] == want[1] or (np.isnan(margin[r]) and np.isnan(want[1])), (r, margin[r], want)
        assert bool(status[r]) == (not np.all(np.isfinite(x[r, :vocab]))), r
