"""Forms of one operator whose dispatch chooses the faster: the chosen one is
timed against a call that the other form takes, or that does the same work in
another layout. Bounds lie well above the run to run spread (about 3%)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _us(ctx, *calls, repeats=50):
    """Microseconds of each call: best of seven rounds of `repeats`, the calls
    in turn so that a change of the machine's pace meets all of them."""
    for call in calls:
        for _ in range(10):
            call()
    best = [np.inf] * len(calls)
    for _ in range(7):
        for i, call in enumerate(calls):
            ctx.timer_begin()
            for _ in range(repeats):
                call()
            best[i] = min(best[i], ctx.timer_end() * 1e3 / repeats)
    return best


@pytest.mark.parametrize("rows,blocks,tokens", [(32768, 80, 64), (18432, 80, 16), (2560, 80, 256)])
def test_x1_rows_cost_about_what_x4_rows_do(q, ctx, rows, blocks, tokens):
    """X1 rows lie apart in memory: reading them in place took 3.0, 2.1 and 3.0
    times as long as X4 rows at these sizes; through the layout launch it is
    1.1 to 1.5 times."""
    rng = np.random.default_rng(0)
    dm = ctx.array(rng.integers(0, 60, size=(rows // 8, blocks, 144), dtype=np.uint8))
    x1 = ctx.array(np.zeros((tokens, blocks, 40), np.uint8))
    x4 = ctx.array(np.zeros((tokens // 4, blocks, 152), np.uint8))
    out = ctx.array(shape=(tokens, rows), dtype=np.float32)
    print(f"X1 against X4 {rows} rows {blocks} blocks {tokens} tokens", flush=True)
    t1, t4 = _us(ctx, lambda: q.q4_dot4_matmul_x1(ctx, dm, x1, out, rows, tokens, blocks, rows),
                 lambda: q.q4_dot4_matmul(ctx, dm, x4, out, rows, tokens, blocks, rows))
    assert t1 < 1.85 * t4, (t1, t4)


@pytest.mark.parametrize("kernel,tokens,channels", [(9, 8, 6144), (7, 6, 6144), (5, 8, 1000)])
def test_few_tokens_of_a_general_convolution(q, ctx, kernel, tokens, channels):
    """Few tokens of kernels other than 4 walk the ring, as an in-place call
    always does; in runs of tokens they took 1.38, 1.37 and 1.16 times as long."""
    rng = np.random.default_rng(0)
    state = ctx.array(rng.standard_normal((kernel - 1, channels)).astype(np.float32))
    x = ctx.array(rng.standard_normal((tokens, channels)).astype(np.float32))
    w = ctx.array((0.1 * rng.standard_normal((kernel, channels))).astype(np.float32))
    out = ctx.array(shape=(tokens, channels), dtype=np.float32)
    print(f"conv kernel {kernel} {tokens} tokens of {channels} channels", flush=True)
    apart, place = _us(ctx,
                       lambda: q.causal_conv1d_silu_f32(ctx, state, 0, x, w, out, channels, kernel, batch=tokens),
                       lambda: q.causal_conv1d_silu_f32(ctx, state, 0, x, w, x, channels, kernel, batch=tokens))
    assert apart < 1.1 * place, (apart, place)


@pytest.mark.parametrize("rows,blocks", [(512, 128), (1024, 120)])
def test_gemv_chain_reads_ahead(q, ctx, rows, blocks):
    """Four steps of the one-vector GEMV against three: a third more blocks
    took 1.4 to 1.5 times as long where the chain waited for every pair of
    terms that it reads; reading eight at once it is 1.0 to 1.1 times."""
    rng = np.random.default_rng(0)
    out = ctx.array(shape=(1, rows), dtype=np.float32)
    calls = []
    for nb in (96, blocks):
        dm = ctx.array(rng.integers(0, 60, size=(rows // 8, nb, 144), dtype=np.uint8))
        x1 = ctx.array(np.zeros((1, nb, 40), np.uint8))
        calls.append(lambda dm=dm, x1=x1, nb=nb: q.q4_dot4_matmul_x1(ctx, dm, x1, out, rows, 1, nb, rows))
    print(f"GEMV {rows} rows 96 and {blocks} blocks", flush=True)
    three, four = _us(ctx, *calls, repeats=400)
    assert four < 1.25 * three, (three, four)


def test_one_more_row_of_ragged_attention(q, ctx):
    """65 rows of unequal contexts against 64: the one row took a launch of its
    own and 1.23 times as long in groups of 64 rows; in one launch 1.02 times."""
    rng = np.random.default_rng(5)
    heads, kv, page = 8, 2, 16
    calls = []
    for rows in (64, 65):
        lens = rng.integers(62, 501, size=rows).astype(np.int32)
        lens[0] = 500
        need = (lens + page - 1) // page
        table = np.zeros((rows, need.max()), np.int32)
        at = 0
        for r in range(rows):
            table[r, :need[r]] = np.arange(at, at + need[r])
            at += need[r]
        pool = ctx.array(np.zeros((at, page, kv, 256), np.uint16))
        qv = ctx.array(np.zeros((rows, heads * 256), np.float32))
        dt, dl = ctx.array(table), ctx.array(lens)
        out = ctx.array(shape=(rows, heads * 256), dtype=np.float32)
        args = (qv, qv, pool, pool, dt, table.shape[1], dl, page, out, rows, heads, kv, 256, 1.0 / 16.0)
        calls.append(lambda args=args: q.attention_decode_paged(ctx, *args))
    print("attention 64 and 65 rows", flush=True)
    us64, us65 = _us(ctx, *calls)
    assert us65 < 1.13 * us64, (us64, us65)
