"""Operator forms at the sizes where their launches change shape: run and
vector edges of the convolution, candidate lists with ties and few tokens,
batches of the direct GEMM, block counts of the GEMV's passes,
wavefront tails of the X4 preparation,
ragged attention grids, the greedy head's counts.
Each against the oracle's token-by-token or single-value form, within the
rounding of one fp32 chain (2^-24 per term) unless exact."""
import numpy as np
import pytest

from tests.operand_util import At

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,ch,kern,begin,end,extra", [
    (1, 64, 4, 0, 64, 0), (2, 64, 4, 0, 64, 4), (3, 68, 4, 4, 68, 0), (7, 64, 4, 0, 64, 0), (8, 64, 4, 0, 63, 0),
    (9, 66, 4, 0, 66, 0), (24, 64, 4, 8, 60, 12), (257, 72, 4, 0, 72, 0), (5, 40, 1, 0, 40, 0), (10, 40, 2, 0, 40, 0),
    (17, 44, 9, 0, 44, 0), (4, 44, 9, 1, 43, 1), (19, 40, 10, 0, 40, 0)])
@pytest.mark.parametrize("in_place", [False, True])
def test_conv1d_runs(q, ctx, orc, batch, ch, kern, begin, end, extra, in_place):
    rng = np.random.default_rng(batch * 100 + ch + kern)
    hist, ring = kern - 1, (kern - 1) // 2
    state = rng.standard_normal((max(hist, 1), ch)).astype(np.float32)
    x = rng.standard_normal((batch, ch + (0 if in_place else extra))).astype(np.float32)
    w = (rng.standard_normal((kern, ch)) * 0.5).astype(np.float32)
    dstate, dx = ctx.array(state), ctx.array(x)
    dout = dx if in_place else ctx.array(np.full((batch, ch), 7.0, np.float32))
    before = x[:, :ch].copy() if in_place else np.full((batch, ch), 7.0, np.float32)
    print(f"conv1d batch {batch} channels [{begin}, {end}) of {ch} kernel {kern} in place {in_place}", flush=True)
    q.causal_conv1d_silu_f32(ctx, dstate, ring if hist else 0, dx, ctx.array(w), dout, ch, kern, batch=batch,
                             input_stride=x.shape[1], channel_begin=begin, channel_end=end)
    # the causal sum over [ring oldest first | inputs] in float64
    order = [(ring + k) % hist for k in range(hist)] if hist else []
    seq = np.concatenate([state[order] if hist else np.zeros((0, ch)), x[:, :ch]]).astype(np.float64)
    s = sum(seq[k:k + batch] * w[k].astype(np.float64) for k in range(kern))
    want = before.astype(np.float64)
    want[:, begin:end] = (s / (1.0 + np.exp(-s)))[:, begin:end]
    # kern products of magnitude below about 8 in fp32, silu's slope below 1.1
    np.testing.assert_allclose(dout.download(), want, rtol=1e-5, atol=kern * 8 * 2.0 ** -23)
    want_state = state.copy()
    for p in range(batch):
        if hist:
            want_state[(ring + p) % hist, begin:end] = x[p, begin:end]
    np.testing.assert_array_equal(dstate.download(), want_state)


@pytest.mark.parametrize("kern", [1, 2, 3, 4, 5, 9, 10])
@pytest.mark.parametrize("batch,ch", [(1, 64), (7, 68), (12, 64), (13, 64), (40, 66), (130, 64)])
def test_conv1d_bits_do_not_depend_on_the_form(q, ctx, batch, ch, kern):
    """The sum of a token is one fma chain (its own tap's product, then the
    history oldest first) in every form: four channels per thread or one, taps
    in registers or re-read, and the walk through the ring of an in-place call."""
    rng = np.random.default_rng(batch + ch + kern)
    hist = kern - 1
    state = rng.standard_normal((max(hist, 1), ch)).astype(np.float32)
    x = rng.standard_normal((batch, ch)).astype(np.float32)
    w = ctx.array((rng.standard_normal((kern, ch)) * 0.5).astype(np.float32))

    def call(place, begin, end):
        ds, dx = ctx.array(state), ctx.array(x)
        out = dx if place else ctx.array(np.zeros((batch, ch), np.float32))
        q.causal_conv1d_silu_f32(ctx, ds, hist // 2 if hist else 0, dx, w, out, ch, kern, batch=batch,
                                 channel_begin=begin, channel_end=end)
        return out.download().view(np.uint32)[:, begin:end], ds.download()

    print(f"conv1d forms batch {batch} channels {ch} kernel {kern}", flush=True)
    want, ring = call(True, 0, ch)
    for begin, end in ((0, ch), (1, ch - 1)):
        got, after = call(False, begin, end)
        np.testing.assert_array_equal(got, want[:, begin:end])
        np.testing.assert_array_equal(after[:, begin:end], ring[:, begin:end])


def _candidate_model(q, ctx, vocab):
    from tests.model_util import build_small_model, small_dims, upload_model
    d, sched = small_dims()
    d["vocab"] = vocab
    model = upload_model(q, ctx, d, sched, build_small_model(d, sched, seed=vocab))
    return d, model, q.Runtime(model, max_slots=1, max_batch=1, max_context=64, page_tokens=16, use_graphs=False)


def _check_candidates(rt, d, slot, k, ties, rng):
    vocab = d["vocab"]
    hidden = np.zeros(d["hidden"], np.float32) if ties else rng.standard_normal(d["hidden"]).astype(np.float32)
    print(f"candidates vocab {vocab} k {k} ties {ties}", flush=True)
    cand, raw = rt.head_candidates(slot, hidden, k, 1.25, penalty=1.3, raw_logits=True)
    v = raw.copy()
    hit = rt.slot_counts(slot) > 0
    v[hit] = np.where(v[hit] > 0, v[hit] / np.float32(1.3), v[hit] * np.float32(1.3))
    v = (v * np.float32(1.25)).astype(np.float32)
    # the kernel's order puts +0 above -0
    key = np.where(v == 0, np.where(np.signbit(v), -1e-45, 0.0), v.astype(np.float64))
    order = np.lexsort((np.arange(vocab), -key))[:k]
    np.testing.assert_array_equal(cand["token"][:k], order)
    np.testing.assert_array_equal(cand["value"][:k].view(np.uint32), v[order].view(np.uint32))
    assert np.all(cand["token"][k:] == -1) and np.all(np.isneginf(cand["value"][k:]))
    return raw, order


@pytest.mark.parametrize("vocab,k", [(64, 64), (264, 1), (264, 64), (8192, 20), (8192, 64)])
@pytest.mark.parametrize("ties", [False, True])
def test_candidates_against_sort(q, ctx, vocab, k, ties):
    """The candidate list equals a descending sort of the raw logits (lower
    token first among equals): few tokens per slice, all logits equal (a zero
    hidden row), penalized tokens, k up to 64."""
    d, model, rt = _candidate_model(q, ctx, vocab)
    slot = rt.slot_alloc(np.arange(0, vocab, 3, dtype=np.int32)[:40])
    _check_candidates(rt, d, slot, k, ties, np.random.default_rng(k))
    rt.close()
    model.close()


@pytest.mark.parametrize("vocab", [20008, 248320])
def test_candidates_of_many_tokens_per_slice(q, ctx, vocab):
    """The same where a thread of a slice holds several tokens: 313 a slice
    with a ragged last one, and the 3880 of the models' vocabulary (all 16 a
    thread takes); every third token counted, so that penalties fall on every
    place of a slice and move some of the best."""
    d, model, rt = _candidate_model(q, ctx, vocab)
    slot = rt.slot_alloc(np.arange(0, vocab, 3, dtype=np.int32))
    rng = np.random.default_rng(vocab)
    for k in (1, 20, 64):
        _check_candidates(rt, d, slot, k, True, rng)
        raw, order = _check_candidates(rt, d, slot, k, False, rng)
        if k == 64:
            assert set(order) != set(np.argsort(-raw)[:k])  # some of the best raw logits were counted
    rt.close()
    model.close()


@pytest.mark.parametrize("rows,blocks", [(8, 1), (8, 8), (24, 9), (40, 3), (72, 33), (136, 112), (16, 260)])
@pytest.mark.parametrize("tokens", [5, 8, 15, 16, 17, 36, 64, 68])
def test_direct_gemm_forms(q, ctx, orc, rows, blocks, tokens):
    """X4 and X1 activations, row and token tails, one split to more than 16:
    every output within the rounding of its chain of the float64 product, and
    the same bits whatever the layout and the batch (the chain of an output
    depends on rows and blocks only); rows past the stride's end untouched."""
    rng = np.random.default_rng(rows * 1000 + blocks * 10 + tokens)
    cols = 32 * blocks
    dm = ctx.array(orc.dot4_pack(orc.random_q4_blocks(rng, rows, cols), rows, blocks))
    codes = rng.integers(-127, 128, size=(tokens, blocks, 32)).astype(np.int8)
    scales = rng.uniform(0.001, 0.02, size=(tokens, blocks)).astype(np.float32)

    def x1_blocks(c, s):
        b = np.zeros((len(c), blocks), np.dtype([("s", "<f4"), ("sum", "<i2"), ("q", "i1", 32), ("pad", "<i2")]))
        b["s"], b["sum"], b["q"] = s, c.sum(-1), c
        return b

    def x4_blocks(c, s):
        b = np.zeros((len(c) // 4, blocks), np.dtype([("s", "<f4", 4), ("sum", "<i2", 4), ("q", "i1", (4, 32))]))
        b["s"] = s.reshape(-1, 4, blocks).transpose(0, 2, 1)
        b["q"] = c.reshape(-1, 4, blocks, 32).transpose(0, 2, 1, 3)
        b["sum"] = b["q"].sum(-1)
        return b

    def run(call, blk, n, stride):
        out = ctx.array(np.full((n, stride), 7.0, np.float32))
        call(ctx, dm, ctx.array(blk.view(np.uint8)), out, rows, n, blocks, stride)
        got = out.download()
        assert np.all(got[:, rows:] == 7.0)
        return got[:, :rows]

    print(f"direct GEMM {rows} rows {blocks} blocks {tokens} tokens", flush=True)
    got = run(q.q4_dot4_matmul_x1, x1_blocks(codes, scales), tokens, rows + 3)
    # terms dot * d * s per block: the kernels' exact integer dots, in float64
    pad = (-tokens) % 4
    c4, s4 = np.concatenate([codes, codes[:pad]]), np.concatenate([scales, scales[:pad]])
    dots = ctx.array(shape=(tokens + pad, rows, blocks), dtype=np.int32)
    q.q4_dot4_block_dots(ctx, dm, ctx.array(x4_blocks(c4, s4).view(np.uint8)), dots, rows, tokens + pad, blocks)
    tiles = dm.download().view(np.uint8).reshape(rows // 8, blocks, 144)
    d = np.ascontiguousarray(tiles[..., :16]).view(np.float16).reshape(rows // 8, blocks, 8).transpose(0, 2, 1)
    terms = dots.download()[:tokens] * d.reshape(rows, blocks).astype(np.float64) * scales[:, None, :].astype(np.float64)
    bound = (blocks + 2) * 2.0 ** -24 * 2 * np.abs(terms).sum(-1)  # a rounding per product and per addition
    assert np.all(np.abs(got - terms.sum(-1)) <= bound)
    x4 = run(q.q4_dot4_matmul, x4_blocks(c4, s4), tokens + pad, rows + 4)
    np.testing.assert_array_equal(x4[:tokens].view(np.uint32), got.view(np.uint32))
    few = run(q.q4_dot4_matmul_x1, x1_blocks(codes[:5], scales[:5]), 5, rows)
    np.testing.assert_array_equal(few.view(np.uint32), got[:5].view(np.uint32))


@pytest.mark.parametrize("offset", [0, 160, 1024])
@pytest.mark.parametrize("rows,blocks,tokens,x1", [(40, 9, 8, False), (40, 9, 7, True), (72, 3, 64, False),
                                                   (24, 17, 68, False), (24, 2, 67, True)])
def test_outputs_over_activations(q, ctx, orc, rows, blocks, tokens, x1, offset):
    """Outputs that share memory with the activations they come from (at its
    start, ahead of it and within it) are those of separate buffers: such a
    call reads every activation before its first output is written."""
    rng = np.random.default_rng(rows + blocks + tokens)
    dm = ctx.array(orc.dot4_pack(orc.random_q4_blocks(rng, rows, 32 * blocks), rows, blocks))
    x = rng.standard_normal((tokens, 32 * blocks)).astype(np.float32)
    act = np.stack([orc.q8_quantize_1(r) for r in x]) if x1 else orc.q8_quantize_4(x)
    act = np.ascontiguousarray(act).view(np.uint8).ravel()
    call = q.q4_dot4_matmul_x1 if x1 else q.q4_dot4_matmul
    stride = rows + 4
    out_bytes = tokens * stride * 4
    apart = ctx.array(shape=(tokens, stride), dtype=np.float32)
    print(f"outputs over activations {rows} rows {blocks} blocks {tokens} tokens at {offset}", flush=True)
    call(ctx, dm, ctx.array(act), apart, rows, tokens, blocks, stride)
    want = apart.download()[:, :rows]
    # (the no-allocation form works in chunks of 64 vectors, so more than one chunk must not overlap)
    calls = [call] if x1 or tokens > 64 else [call, q.q4_dot4_matmul_noalloc]
    for a_at, o_at in ((0, offset), (offset, 0)):
        for f in calls:
            host = np.zeros(offset + max(act.size, out_bytes), np.uint8)
            host[a_at:a_at + act.size] = act
            both = ctx.array(host)
            f(ctx, dm, At(both, a_at), At(both, o_at), rows, tokens, blocks, stride)
            got = both.download()[o_at:o_at + out_bytes].view(np.float32).reshape(tokens, stride)[:, :rows]
            np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("rows,blocks,tokens", [
    (4096, 121, 16), (4096, 122, 16), (4104, 30, 20), (24, 31, 36),  # X1 direct or split (2000 blocks a unit)
    (1024, 8, 420), (1024, 8, 900), (2560, 4, 160),                  # X1 direct or dense (80 rows a unit)
    (8224, 64, 68), (8224, 65, 68), (4096, 80, 200),                 # X4 direct or dense (256 rows, 64 blocks)
    (8224, 106, 40), (8224, 107, 40), (8224, 257, 36), (2560, 352, 64), (2560, 353, 64)])  # X4 direct or split
def test_forms_on_both_sides_of_the_lines(q, ctx, orc, rows, blocks, tokens):
    """One set of codes through every form that takes it: X1 and X4 outputs in
    buffers of their own (the direct GEMM, or the split launches or the dense
    GEMM beyond its lines) and over their activations (never direct) have the
    same bits."""
    rng = np.random.default_rng(rows + blocks + tokens)
    dm = ctx.array(orc.dot4_pack(orc.random_q4_blocks(rng, rows, 32 * blocks), rows, blocks))
    codes = rng.integers(-127, 128, size=(tokens, blocks, 32)).astype(np.int8)
    scales = rng.uniform(0.001, 0.02, size=(tokens, blocks)).astype(np.float32)
    x1 = np.zeros((tokens, blocks), np.dtype([("s", "<f4"), ("sum", "<i2"), ("q", "i1", 32), ("pad", "<i2")]))
    x1["s"], x1["sum"], x1["q"] = scales, codes.sum(-1), codes
    x4 = np.zeros((tokens // 4, blocks), np.dtype([("s", "<f4", 4), ("sum", "<i2", 4), ("q", "i1", (4, 32))]))
    x4["s"] = scales.reshape(-1, 4, blocks).transpose(0, 2, 1)
    x4["q"] = codes.reshape(-1, 4, blocks, 32).transpose(0, 2, 1, 3)
    x4["sum"] = x4["q"].sum(-1)
    print(f"forms {rows} rows {blocks} blocks {tokens} tokens", flush=True)
    want = None
    for call, act in ((q.q4_dot4_matmul, x4), (q.q4_dot4_matmul_x1, x1)):
        act = act.view(np.uint8).ravel()
        apart = ctx.array(shape=(tokens, rows), dtype=np.float32)
        call(ctx, dm, ctx.array(act), apart, rows, tokens, blocks, rows)
        both = ctx.array(np.concatenate([act, np.zeros(max(0, tokens * rows * 4 - act.size), np.uint8)]))
        call(ctx, dm, both, both, rows, tokens, blocks, rows)
        over = both.download()[:tokens * rows * 4].view(np.uint32).reshape(tokens, rows)
        want = over if want is None else want
        np.testing.assert_array_equal(apart.download().view(np.uint32), want)
        np.testing.assert_array_equal(over, want)


@pytest.mark.parametrize("blocks", [1, 31, 32, 33, 64, 65, 97, 128, 129, 257, 288, 289, 577])
def test_gemv_passes(q, ctx, orc, blocks):
    """Every step count and pass boundary of the GEMV, one to four vectors:
    the bits of the exact-mode GEMM (one block-order chain per output)."""
    rng = np.random.default_rng(blocks)
    rows, cols = 24, 32 * blocks
    dm = ctx.array(orc.dot4_pack(orc.random_q4_blocks(rng, rows, cols), rows, blocks))
    x4 = np.zeros((1, blocks), np.dtype([("s", "<f4", 4), ("sum", "<i2", 4), ("q", "i1", (4, 32))]))
    x4["s"] = rng.uniform(0.001, 0.02, size=(1, blocks, 4))
    x4["q"] = rng.integers(-127, 128, size=(1, blocks, 4, 32))
    x4["sum"] = x4["q"].astype(np.int32).sum(-1)
    x1 = np.zeros((4, blocks), np.dtype([("s", "<f4"), ("sum", "<i2"), ("q", "i1", 32), ("pad", "<i2")]))
    x1["s"], x1["sum"], x1["q"] = x4["s"][0].T, x4["sum"][0].T, x4["q"][0].transpose(1, 0, 2)
    d4, d1, out = ctx.array(x4.view(np.uint8)), ctx.array(x1.view(np.uint8)), ctx.array(shape=(4, rows), dtype=np.float32)
    print(f"GEMV {blocks} blocks", flush=True)
    q.q4_dot4_matmul(ctx, dm, d4, out, rows, 4, blocks, rows, exact=True)
    want = out.download().view(np.uint32)
    q.q4_dot4_matmul(ctx, dm, d4, out, rows, 4, blocks, rows)
    np.testing.assert_array_equal(out.download().view(np.uint32), want)
    for n in (1, 2, 3, 4):
        dst = ctx.array(shape=(n, rows), dtype=np.float32)
        q.q4_dot4_matmul_x1(ctx, dm, d1, dst, rows, n, blocks, rows)
        np.testing.assert_array_equal(dst.download().view(np.uint32), want[:n])


@pytest.mark.parametrize("tokens,cols", [(4, 128), (8, 384), (12, 640), (5468, 384)])
@pytest.mark.parametrize("h128", [True, False])
def test_x4_preparation_equals_rows(q, ctx, tokens, cols, h128):
    """X4 blocks (one wavefront per four tokens and 128 columns, alone or four
    to a workgroup with a tail) hold the bytes of the rows prepared one by one."""
    rng = np.random.default_rng(tokens + cols)
    x = rng.standard_normal((tokens, cols)).astype(np.float32)
    x[1] = 0.0
    nb = cols // 32
    x4t = np.dtype([("s", "<f4", 4), ("sum", "<i2", 4), ("q", "i1", (4, 32))])
    x1t = np.dtype([("s", "<f4"), ("sum", "<i2"), ("q", "i1", 32), ("pad", "<i2")])
    d4 = ctx.array(shape=(tokens // 4, nb, 152), dtype=np.uint8)
    print(f"X4 preparation {tokens} x {cols} h128 {h128}", flush=True)
    if h128:
        q.q4_h128_prepare_activations_4(ctx, ctx.array(x), d4, tokens, cols)
    else:
        q.q8_0_quantize_vectors_4(ctx, ctx.array(x), d4, tokens, nb)
    got = d4.download().view(x4t).reshape(tokens // 4, nb)
    for r in sorted({0, 1, 2, 3, tokens // 2, tokens - 2, tokens - 1}):
        d1 = ctx.array(shape=(nb, 40), dtype=np.uint8)
        if h128:
            q.q4_h128_prepare_activation_1(ctx, ctx.array(x[r:r + 1]), d1, cols)
        else:
            q.q8_0_quantize_vector_1(ctx, ctx.array(x[r:r + 1]), d1, nb)
        one = d1.download().view(x1t).reshape(nb)
        for f in ("s", "sum", "q"):
            np.testing.assert_array_equal(got[r // 4][f][:, r % 4], one[f])


@pytest.mark.parametrize("batch,page_tokens,lens", [
    (2, 16, (1, 700)), (2, 16, (1, 7000)), (3, 4, (130, 1, 64)), (64, 16, None), (65, 16, None), (130, 8, None),
    (256, 16, None), (257, 16, None)])
def test_ragged_attention_equals_rows_alone(q, ctx, batch, page_tokens, lens):
    """Rows of unequal contexts in one call (the grid of exactly their chunks,
    in groups of 256 rows, or the full grid where that saves too little) give
    the bits of each row called alone."""
    rng = np.random.default_rng(batch)
    heads, kv, hd = 4, 2, 256
    lens = np.asarray(lens if lens is not None else rng.integers(1, 500, size=batch), np.int32)
    lens[-1] = max(lens[-1], 641)  # one long row: the others leave most of the full grid idle
    need = (lens + page_tokens - 1) // page_tokens
    pool = rng.standard_normal((2, int(need.sum()), page_tokens, kv, hd)).astype(np.float16).view(np.uint16)
    table = np.zeros((batch, need.max()), np.int32)
    perm, at = rng.permutation(int(need.sum())), 0
    for r in range(batch):
        table[r, :need[r]] = perm[at:at + need[r]]
        at += need[r]
    qv, gates = rng.standard_normal((2, batch, heads * hd)).astype(np.float32)
    dk, dv = ctx.array(pool[0]), ctx.array(pool[1])

    def call(rows):
        out = ctx.array(shape=(len(rows), heads * hd), dtype=np.float32)
        q.attention_decode_paged(ctx, ctx.array(qv[rows]), ctx.array(gates[rows]), dk, dv, ctx.array(table[rows]),
                                 table.shape[1], ctx.array(lens[rows]), page_tokens, out, len(rows), heads, kv, hd,
                                 1.0 / 16.0)
        return out.download().view(np.uint32)

    print(f"ragged attention batch {batch} page {page_tokens}", flush=True)
    together = call(np.arange(batch))
    for r in sorted({0, 1, batch // 2, min(63, batch - 1), min(64, batch - 1), min(255, batch - 1), batch - 1}):
        np.testing.assert_array_equal(call(np.array([r]))[0], together[r])
    with pytest.raises(q.Q35Error):
        lens[0] = table.shape[1] * page_tokens + 1
        call(np.arange(batch))


@pytest.mark.parametrize("blocks", [1, 12, 13, 16, 33])
@pytest.mark.parametrize("rows,vectors", [(8, 4), (72, 12), (200, 16), (520, 20), (1000, 36)])
def test_head_counts_of_the_best_rows(q, ctx, orc, rows, blocks, vectors):
    """Greedy head with the best rows of each token counted, so that a count
    read for another row or token changes the winner: fewer than four chunks
    of four blocks (counts read at a group's end) and more (read ahead), one
    and several token tiles, ragged row groups. Exact index and value."""
    rng = np.random.default_rng(rows * 100 + blocks)
    packed = orc.dot4_pack(orc.random_q4_blocks(rng, rows, blocks * 32), rows, blocks)
    act = orc.q8_quantize_4(rng.standard_normal((vectors, blocks * 32)).astype(np.float32))
    adj = orc.dot4_matmul(packed, act, rows, vectors, blocks).copy()
    pen = np.where(np.arange(vectors) % 4 == 3, 1.0, 1.5).astype(np.float32)
    counts = np.zeros((vectors, rows), np.int32)
    for v in range(vectors):
        counts[v, np.argsort(adj[v])[-1 - v % 4:]] = 1 + v
        m = (counts[v] > 0) & (pen[v] > 1)
        adj[v, m] = np.where(adj[v, m] > 0, adj[v, m] / pen[v], adj[v, m] * pen[v])
    want = adj.argmax(1)
    idx = ctx.array(shape=(vectors,), dtype=np.int32)
    val = ctx.array(shape=(vectors,), dtype=np.float32)
    q.q4_dot4_argmax_batch(ctx, ctx.array(packed), ctx.array(act), ctx.array(counts), ctx.array(pen), rows, vectors,
                           blocks, idx, val)
    np.testing.assert_array_equal(idx.download(), want)
    np.testing.assert_array_equal(val.download(), adj[np.arange(vectors), want])


@pytest.mark.parametrize("g16", [False, True])
@pytest.mark.parametrize("rows", [5, 20])
def test_greedy_steps_with_and_without_penalties(q, ctx, rows, g16):
    """Steps of one shape whose rows have no, some or only penalties, in turn
    and with captured graphs: each gives the tokens that its logits and counts
    give, so a step with a penalty never replays the graph without counts."""
    from tests.model_util import build_small_model, small_dims, upload_model
    d, _ = small_dims()
    d = dict(d, hidden=1024, intermediate=512, n_layers=2)
    sched = np.array([1, 0], np.uint8)
    model = upload_model(q, ctx, d, sched, build_small_model(d, sched, seed=23, head_g16=g16))
    rt = q.Runtime(model, max_slots=rows, max_batch=32, max_context=16, page_tokens=16, use_graphs=True)
    rng = np.random.default_rng(rows)
    # most of the vocabulary counted in every slot, so that a penalty moves most maxima
    slots = [rt.slot_alloc(rng.permutation(d["vocab"])[d["vocab"] // 16:].astype(np.int32)) for _ in range(rows)]
    table = np.array([[rt.page_alloc()] for _ in range(rows)], np.int32)
    toks = rng.integers(0, d["vocab"], size=rows).astype(np.int32)
    one, some, most = np.ones(rows, np.float32), np.ones(rows, np.float32), np.full(rows, 4.0, np.float32)
    some[::3] = 4.0
    print(f"greedy steps rows {rows} G16 {g16}", flush=True)
    # position 0 again each time: the step reads the state it found the first time
    want = {}
    for name, pen in (("one", one), ("some", some), ("most", most)):
        want[name] = rt.step(slots, [0] * rows, toks, table, penalties=pen, logits=True)[0]
    assert np.any(want["one"] != want["some"]) and np.any(want["some"] != want["most"])
    for name, pen in (("one", one), ("some", some), ("one", one), ("most", most), ("one", one), ("some", some)):
        np.testing.assert_array_equal(rt.step(slots, [0] * rows, toks, table, penalties=pen), want[name])
    rt.close()
    model.close()
