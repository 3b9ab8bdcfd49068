"""The f16 arm's many-row projections on the matrix units against the vector
kernels, bit for bit: prompts of several rows a stream (and cohorts of 6 and
more streams at the logits head) take the matrix form, the same tokens one
position at a time on one stream take the vector form, and both compute
dot_f16c's association, so the logits must be identical.  Rows past 16 and 256
cover several row tiles and prefill chunks, widths 384 / 640 / 1280 the partial
weight batches."""
import numpy as np
import pytest

from franken_whisper_amd import abi, native, synth
from tests.helpers import assert_bitexact

pytestmark = pytest.mark.gpu

T = 96


@pytest.fixture(scope="module")
def decs():
    ctx = native.Context(0)
    made = {}

    def get(d):
        if d not in made:
            cfg = synth.Config(f"rows-{d}", 51864, T, d, d // 64, 1, 448, d, d // 64, 1, 16)
            made[d] = (cfg, native.Decoder(ctx, synth.Model(cfg, seed=3, encoder=False), abi.DEC_F16))
        return (ctx,) + made[d]

    yield get
    for _, e in made.values():
        e.close()
    ctx.close()


@pytest.mark.parametrize("d,S,n", [(1280, 1, 16), (1280, 1, 40), (1280, 1, 263), (1280, 5, 9), (1280, 6, 1),
                                   (1280, 10, 4), (1280, 16, 3), (1280, 17, 1), (384, 1, 107), (384, 9, 13),
                                   (384, 16, 33), (640, 1, 65), (640, 7, 31)])
def test_rows_match_single_rows(decs, d, S, n):
    ctx, cfg, dec = decs(d)
    states = synth.encoder_states(7, S, T, d)
    tokens = np.random.default_rng(n).integers(0, cfg.n_vocab, (S, n)).astype(np.int32)
    print("width", d, "streams", S, "positions", n, flush=True)
    st = dec.state(S, T)
    st.set_cross(ctx.array(states))
    out = ctx.empty((S, cfg.n_vocab), np.float32)
    am = st.step(tokens, out)
    got = out.download()
    st.close()
    one = ctx.empty((1, cfg.n_vocab), np.float32)
    for s in sorted({0, S // 2, S - 1}):
        ref = dec.state(1, T)
        ref.set_cross(ctx.array(np.ascontiguousarray(states[s:s + 1])))
        for t in range(n):
            a = ref.step(tokens[s:s + 1, t:t + 1], one)
        assert_bitexact(got[s], one.download()[0], f"stream {s}")
        assert a[0] == am[s]
        ref.close()


@pytest.mark.parametrize("V", [4096, 8192, 16383, 16384])
@pytest.mark.parametrize("d,S", [(128, 10), (384, 16)])
def test_small_vocabulary_argmax(d, S, V):
    """A logits head of fewer than 16,384 rows: the cohort's argmax keys are
    written at every step (the maximum moves from step to step), the tokens and
    logits are those of one stream at a time."""
    ctx = native.Context(0)
    cfg = synth.Config(f"vocab-{V}-{d}", V, T, d, d // 64, 1, 448, d, d // 64, 1, 16)
    m = synth.Model(cfg, seed=3, encoder=False)
    dec = native.Decoder(ctx, m, abi.DEC_F16)
    states = synth.encoder_states(7, S, T, d)
    tokens = np.random.default_rng(V).integers(0, V, (S, 6)).astype(np.int32)
    print("width", d, "streams", S, "vocabulary", V, flush=True)
    st, out, one = dec.state(S, T), ctx.empty((S, V), np.float32), ctx.empty((1, V), np.float32)
    st.set_cross(ctx.array(states))
    cuts = [(0, 3), (3, 4), (4, 5), (5, 6)]  # a prompt, then single positions
    got = []
    for a, b in cuts:
        am = st.step(tokens[:, a:b], out)
        got.append((am, out.download()))
        np.testing.assert_array_equal(am, got[-1][1].argmax(1))
    assert len({tuple(am) for am, _ in got}) == len(cuts)
    st.close()
    for s in (0, S - 1):
        ref = dec.state(1, T)
        ref.set_cross(ctx.array(np.ascontiguousarray(states[s:s + 1])))
        for (a, b), (am, logits) in zip(cuts, got):
            assert ref.step(tokens[s:s + 1, a:b], one)[0] == am[s]
            assert_bitexact(logits[s], one.download()[0], f"stream {s} positions {a}..{b}")
        ref.close()
    dec.close()
    ctx.close()
