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
