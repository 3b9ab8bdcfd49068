"""The f16-pair attention at the edges of its tiles: one 64-key tile, a last
tile of 1 or 63 keys, query blocks (256 and 512) that end inside a wave or
leave whole waves without a query.  One and two windows take the 128-query
blocks, 7 and more the 256-query ones, 40 windows of 257 to 512 rows the
512-query ones.

Fast mode against exact mode (bit-identical to the oracle): the pairs carry
|a| to 2^-22 relative and every sum stays in f32, so the bound is the fast
mode's max-abs 1e-3 (measured about 1e-6 here, where no quantizer follows)."""
import numpy as np
import pytest

from franken_whisper_amd import abi, native, synth
from tests.helpers import assert_bitexact, rel_maxabs

pytestmark = pytest.mark.gpu

CFG = synth.Config("attn-edges", 51864, 640, 384, 6, 2, 64, 384, 6, 1, 16)


@pytest.fixture(scope="module")
def enc():
    ctx = native.Context(0)
    e = native.Encoder(ctx, synth.Model(CFG, seed=5, decoder=False), abi.ENC_F32)
    yield ctx, e
    e.close()
    ctx.close()


def _forward(ctx, e, x, rows):
    out = ctx.empty((x.shape[0], rows, CFG.n_audio_state), np.float32)
    e.forward_time_major(ctx.array(np.ascontiguousarray(x)), x.shape[0], 2 * rows, out)
    return out.download()


@pytest.mark.parametrize("rows", [1, 2, 63, 64, 65, 127, 128, 129, 255, 256, 257, 320, 511, 512, 513, 640])
def test_attention_tile_edges(enc, rows):
    ctx, e = enc
    n = 40 if 256 < rows <= 512 else 2 if rows < 256 else 15  # 240 heads x 2 blocks of 256 queries or 1 of 512
    x = synth.mel_input(rows, n, 2 * rows, CFG.n_mels) * np.float32(0.5)
    print("rows", rows, "windows", n, flush=True)
    many = _forward(ctx, e, x, rows)
    e.set_exact(True)
    want = _forward(ctx, e, x[:2], rows)
    e.set_exact(False)
    assert rel_maxabs(many[:2], want) < 1e-3
    for w in (0, n - 1):
        one = _forward(ctx, e, x[w:w + 1], rows)
        assert_bitexact(one[0], many[w], f"{rows} rows: window {w} alone and among {n}")
    if rows < 256:  # 43 windows: 258 heads, past one round of 128-query blocks
        x = np.concatenate([x[:1]] * 43)
        for y in _forward(ctx, e, x, rows)[::14]:
            assert_bitexact(y, many[0], f"{rows} rows: among 43 windows")
