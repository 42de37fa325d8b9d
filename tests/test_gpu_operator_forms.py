"""Operator forms at the sizes where their launches change shape: run and
vector edges of the convolution.
Each against the oracle's token-by-token or single-value form, within the
rounding of one fp32 chain (2^-24 per term) unless exact."""
import numpy as np
import pytest

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
