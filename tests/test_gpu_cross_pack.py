"""The slot-order copies of the cross K and V^T at encoder lengths that end in a
tail of fewer than 32 frames, an odd 32-chunk or a whole 64-group: the f16
arm's logits in exact mode (strict cross K/V) against the oracle bit for bit."""
import numpy as np
import pytest

from franken_whisper_amd import abi, native, synth
from oracle import oracle as O
from tests.helpers import assert_bitexact

pytestmark = pytest.mark.gpu

CFG = synth.Config("cross-pack", 51864, 320, 128, 2, 1, 64, 128, 2, 1, 16)


@pytest.fixture(scope="module")
def pair():
    ctx = native.Context(0)
    m = synth.Model(CFG, seed=6, encoder=False)
    dec = native.Decoder(ctx, m, abi.DEC_F16)
    dec.set_exact(True)
    yield ctx, dec, O.Decoder(m, abi.DEC_F16)
    dec.close()
    ctx.close()


@pytest.mark.parametrize("T", [1, 31, 32, 33, 63, 64, 65, 95, 96, 97, 161, 255, 320])
def test_cross_lengths(pair, T):
    ctx, dec, odec = pair
    states = synth.encoder_states(T, 2, T, CFG.n_text_state)
    tokens = np.random.default_rng(T).integers(0, CFG.n_vocab, (2, 3)).astype(np.int32)
    print("frames", T, flush=True)
    st = dec.state(2, T)
    st.set_cross(ctx.array(states))
    out = ctx.empty((2, CFG.n_vocab), np.float32)
    st.step(tokens, out)
    got = out.download()
    st.close()
    for s in range(2):
        assert_bitexact(got[s], odec.state(states[s]).step(tokens[s]), f"stream {s}")


@pytest.mark.parametrize("S,T", [(40, 1), (40, 2), (33, 3), (40, 4), (9, 31), (5, 33), (7, 50), (16, 66), (3, 127), (3, 130),
                                 (5, 257), (7, 300), (2, 319), (40, 320)])
def test_cross_kv_of_a_cohort(S, T):
    """The fast cross K/V GEMM's tiles run over the streams' borders: every
    stream's K and V^T are the bits that it gets alone, and within f16 rounding
    of the strict ones (two f16 spacings of the largest value cover the f16
    pair's 2^-22 and a rounding to the other neighbour)."""
    ctx = native.Context(0)
    cfg = synth.Config("cross-cohort", 51864, 320, 384, 6, 1, 64, 384, 6, 2, 16)
    dec = native.Decoder(ctx, synth.Model(cfg, seed=6, encoder=False), abi.DEC_F16)
    states = synth.encoder_states(T, S, T, cfg.n_text_state)
    print("streams", S, "frames", T, flush=True)
    st, one = dec.state(S, T), dec.state(1, T)
    st.set_cross(ctx.array(states))
    for s in range(S):
        for exact in (False, True) if s in (0, S - 1) else (False,):
            dec.set_exact(exact)
            one.set_cross(ctx.array(np.ascontiguousarray(states[s:s + 1])))
            for what in (abi.DS_CROSS_K_F16, abi.DS_CROSS_VT_F16):
                got, want = st.read(what, s), one.read(what, 0)
                if not exact:
                    np.testing.assert_array_equal(got, want, err_msg=f"stream {s} buffer {what}")
                else:
                    g, w = got.view(np.float16).astype(np.float32), want.view(np.float16).astype(np.float32)
                    assert np.abs(g - w).max() <= 2 * np.spacing(np.abs(want.view(np.float16)).max())
    st.close()
    one.close()
    dec.close()
    ctx.close()
