"""The f16-pair GEMMs at the edges of their tiles and of the GELU outputs' lo
planes: row counts around 64 / 128 / 256, windows that straddle row tiles (the
conv stem's padded layout), MLP and conv rows with values >= 10 (whose lo
halves are nonzero) in some 64 x 64 blocks only, and one encoder used with
other frame counts in between (nothing left over from a larger call).

Fast mode against exact mode (bit-identical to the oracle): pairs carry |a| to
2^-22 relative with f32 sums, so a GELU argument can round to the neighbouring
f16 table index and move one fc2 input by 2^-11 of it; bound 1e-3 max-abs, as
for the whole f32 plan.  With six fc1 values of about 300 a row's maximum is
about 300 * 0.03 * sqrt(6) = 22 (weights ~0.03): an index step there is at most
2^-11 * 10 * 0.03 / 22 = 7e-6 and a few together stay under 1e-4, while a lo
plane that is skipped or stale (2^-12 of 300 per value) would show as 1e-4 ..
6e-4.
The conv stem by itself (a model whose layers add nothing): the error of the
pairs and f32 sums alone, bound 2e-5 max-abs of LayerNorm outputs around 1: K =
1152 products at 2^-22 each and their sums give 1e-6; a conv2 value below 10 at the
neighbouring f16 index of the GELU is off by 2^-7 in a row whose spread is 400 at
these inputs, 5e-6 of a maximum of 4.  Without conv1's lo plane the same outputs are
off by 2e-4 (checked in the test, in 64 bits on the CPU)."""
import copy

import numpy as np
import pytest

from franken_whisper_amd import abi, native, synth
from tests.helpers import assert_bitexact, rel_maxabs

pytestmark = pytest.mark.gpu

CFG = synth.Config("gemm-edges", 51864, 640, 384, 6, 2, 64, 384, 6, 1, 16)


def _model(gain):
    """gain: the factor on a few MLP LayerNorm weights (fc1 values pass 10 in some blocks)."""
    m = copy.copy(synth.Model(CFG, seed=5, decoder=False))
    if gain:
        m.t = dict(m.t)
        for i in range(CFG.n_audio_layer):
            name = f"encoder.blocks.{i}.mlp.0.bias"
            b = m.t[name].copy()
            b[70:75] += np.float32(gain)  # one 64-column block of fc1 (two with the next at 1000)
            b[1000] += np.float32(gain)
            m.t[name] = b
    return m


@pytest.fixture(scope="module")
def encs():
    ctx = native.Context(0)
    made = {}

    def get(plan, gain):
        if (plan, gain) not in made:
            made[plan, gain] = native.Encoder(ctx, _model(gain), plan)
        return ctx, made[plan, gain]

    yield get
    for e in made.values():
        e.close()
    ctx.close()


@pytest.fixture(scope="module")
def stems():
    """Encoders whose layers leave the rows as conv2 wrote them, and the model."""
    ctx = native.Context(0)
    m = copy.copy(synth.Model(CFG, seed=5, decoder=False))
    m.t = dict(m.t)
    for i in range(CFG.n_audio_layer):
        for name in ("attn.out", "mlp.2"):
            for part in ("weight", "bias"):
                key = f"encoder.blocks.{i}.{name}.{part}"
                m.t[key] = np.zeros_like(m.t[key])
    made = {p: native.Encoder(ctx, m, p) for p in (abi.ENC_F32, abi.ENC_INT8)}
    yield ctx, m, made
    for e in made.values():
        e.close()
    ctx.close()


def _gelu(x):
    t = x.astype(np.float32).astype(np.float16).astype(np.float64)
    y = (0.5 * t * (1 + np.tanh(0.7978846 * t * (1 + 0.044715 * t * t)))).astype(np.float16).astype(np.float64)
    return np.where(x <= -10, 0.0, np.where(x >= 10, x, y))


def _stem64(m, x, lo):
    """ln_post of the conv stem of one window x [frames, mels] in 64 bits; lo: conv1's
    outputs as f32, else as their f16 hi halves.  Also how many of them are >= 10."""
    d, t = CFG.n_audio_state, x.shape[0]
    w1, w2 = (m.t[f"encoder.conv{i}.weight"].view(np.float16).astype(np.float64) for i in (1, 2))
    pad = np.pad(x.astype(np.float64), ((1, 1), (0, 0)))
    h = _gelu(sum(pad[k:k + t] @ w1[:, :, k].T for k in range(3)) + m.t["encoder.conv1.bias"])
    big = int((h >= 10).sum())
    h = h.astype(np.float32 if lo else np.float16).astype(np.float64)
    pad = np.pad(h, ((1, 1), (0, 0)))
    y = _gelu(sum(pad[k:k + t:2] @ w2[:, :, k].T for k in range(3)) + m.t["encoder.conv2.bias"])
    y = y + m.t["encoder.positional_embedding"].reshape(-1, d)[:t // 2]
    y = y - y.mean(1, keepdims=True)
    return y / np.sqrt((y * y).mean(1, keepdims=True) + 1e-5), big


@pytest.mark.parametrize("plan", [abi.ENC_F32, abi.ENC_INT8], ids=["f32", "int8"])
@pytest.mark.parametrize("rows,n", [(5, 7), (65, 9), (129, 4), (300, 3), (511, 3), (640, 4)])
def test_conv_lo_plane(stems, rows, n, plan):
    """conv1 outputs >= 10 (their lo halves are not zero), windows that end inside
    row tiles: every window against the stem in 64 bits."""
    ctx, m, made = stems
    x = synth.mel_input(rows, n, 2 * rows, CFG.n_mels) * np.float32(15000.0)
    got = _forward(ctx, made[plan], x, rows)
    for w in range(n):
        want, big = _stem64(m, x[w], True)
        err, lost = rel_maxabs(got[w], want.astype(np.float32)), rel_maxabs(_stem64(m, x[w], False)[0], want)
        print("rows", rows, "window", w, "large", big, "error", err, "without lo", lost, flush=True)
        assert big > rows * 2 * CFG.n_audio_state // 5 and lost > 5e-5
        assert err < 2e-5


def _forward(ctx, e, x, rows, exact=False):
    out = ctx.empty((x.shape[0], rows, CFG.n_audio_state), np.float32)
    e.set_exact(exact)
    e.forward_time_major(ctx.array(np.ascontiguousarray(x)), x.shape[0], 2 * rows, out)
    e.set_exact(False)
    return out.download()


@pytest.mark.parametrize("gain", [0, 11, 300], ids=["small", "values-10", "values-300"])
@pytest.mark.parametrize("rows,n", [(1, 1), (1, 5), (2, 3), (31, 3), (32, 2), (63, 2), (64, 4), (65, 5), (127, 2), (129, 3),
                                    (255, 2), (257, 3), (300, 40), (513, 2), (640, 8)])
def test_f32_plan_tile_edges(encs, rows, n, gain):
    ctx, e = encs(abi.ENC_F32, gain)
    x = synth.mel_input(rows, n, 2 * rows, CFG.n_mels) * np.float32(0.5)
    got = _forward(ctx, e, x, rows)
    want = _forward(ctx, e, x, rows, exact=True)
    err = rel_maxabs(got, want)
    print("rows", rows, "windows", n, "gain", gain, "error", err, flush=True)
    assert err < (1e-4 if gain == 300 else 1e-3)


@pytest.mark.parametrize("plan", [abi.ENC_F32, abi.ENC_INT8], ids=["f32", "int8"])
def test_calls_of_other_sizes_leave_nothing(encs, plan):
    """Large conv inputs (conv1 outputs >= 10, a nonzero lo plane), then shorter
    and smaller ones on the same buffers: the same bits as before."""
    ctx, e = encs(plan, 0)
    small = [(100, 3), (300, 2), (640, 1)]
    xs = [synth.mel_input(7 + r, n, 2 * r, CFG.n_mels) * np.float32(0.5) for r, n in small]
    first = [_forward(ctx, e, x, r) for x, (r, n) in zip(xs, small)]
    big = synth.mel_input(3, 4, 2 * 640, CFG.n_mels) * np.float32(400.0)
    got = _forward(ctx, e, big, 640)
    if plan == abi.ENC_F32:
        assert rel_maxabs(got, _forward(ctx, e, big, 640, exact=True)) < 1e-3
    for x, (r, n), want in zip(xs, small, first):
        assert_bitexact(_forward(ctx, e, x, r), want, f"{r} rows x {n} after larger calls")
