"""The int8 encoder GEMMs at the edges of their tiles (256 x 256, 256 x 128 and
128 x 128, the choice as on 256 CUs): the exact accumulators and the f32 rows
against the oracle bit for bit, the fused q/k/v split against the f16 pairs of
the oracle's values, fc1's index form; the residual epilogue through whole
forwards, window for window the bits of a window alone."""
import numpy as np
import pytest

from franken_whisper_amd import abi, native, synth
from oracle import oracle as O
from tests.helpers import assert_bitexact

pytestmark = pytest.mark.gpu

CFG = synth.Config("i8-edges", 51864, 1500, 384, 6, 1, 64, 384, 6, 1, 16)


@pytest.fixture(scope="module")
def pair():
    ctx = native.Context(0)
    m = synth.Model(CFG, seed=9, decoder=False)
    e = native.Encoder(ctx, m, abi.ENC_INT8)
    yield ctx, e, O.Encoder(m, abi.ENC_INT8)
    e.close()
    ctx.close()


@pytest.mark.parametrize("M", [1, 31, 32, 33, 127, 128, 129, 255, 256, 257, 700, 1500, 3000, 6001])
def test_gemm_rows(pair, M):
    ctx, e, oenc = pair
    d = CFG.n_audio_state
    rng = np.random.default_rng(M)
    for which in (0, 3, 4, 5):
        inp, out = (4 * d if which == 5 else d), (4 * d if which == 4 else d)
        x = (rng.standard_normal((M, inp)) * 1.3).astype(np.float32)
        acc, y = ctx.empty((M, out), np.int32), ctx.empty((M, out), np.float32)
        print("rows", M, "gemm", which, flush=True)
        e.gemm_i8(0, which, ctx.array(x), acc, y)
        want_acc, want_y = oenc.gemm(0, which, x)
        np.testing.assert_array_equal(acc.download(), want_acc)
        assert_bitexact(y.download(), want_y, f"rows {M} gemm {which}")


@pytest.mark.parametrize("B,T", [(1, 1), (3, 31), (2, 64), (1, 129), (5, 255), (2, 257), (1, 1500), (30, 300),
                                 (10, 257), (14, 259), (8, 639),  # 256 x 128
                                 (12, 513), (7, 1025), (9, 769), (16, 511)])  # 256 x 256
def test_qkv_windows(pair, B, T):
    ctx, e, oenc = pair
    d, H, Tp = CFG.n_audio_state, CFG.n_audio_head, (T + 63) // 64 * 64
    x = (np.random.default_rng(T).standard_normal((B * T, d)) * 1.3).astype(np.float32)
    qk, vt = B * H * T * 64, B * H * 64 * Tp
    out = ctx.empty((4 * qk + 2 * vt,), np.uint16)
    print("windows", B, "rows", T, flush=True)
    e.gemm_i8_fused(0, 0, ctx.array(x), B, T, out)
    got = out.download()
    t = np.arange(T)
    pos = (t & ~12) | ((t & 4) << 1) | ((t & 8) >> 1)
    for which in range(3):
        y = np.asarray(oenc.gemm(0, which, x)[1], np.float32)
        hi = y.astype(np.float16)
        lo = (y - hi.astype(np.float32)).astype(np.float16)
        for k, p in enumerate((hi, lo)):
            want = p.view(np.uint16).reshape(B, T, H, 64)
            if which < 2:
                plane = got[(2 * which + k) * qk:(2 * which + k + 1) * qk].reshape(B, H, T, 64)
                np.testing.assert_array_equal(plane, want.transpose(0, 2, 1, 3))
            else:
                plane = got[4 * qk + k * vt:4 * qk + (k + 1) * vt].reshape(B, H, 64, Tp)
                np.testing.assert_array_equal(plane[:, :, :, pos], want.transpose(0, 2, 3, 1))


@pytest.mark.parametrize("M", [1, 33, 129, 257, 1500, 6001])
def test_fc1_index(pair, M):
    ctx, e, oenc = pair
    d = CFG.n_audio_state
    x = (np.random.default_rng(M).standard_normal((M, d)) * 1.3).astype(np.float32)
    x[::5] *= 60.0  # rows whose fc1 values pass +-10
    idx, side = ctx.empty((M, 4 * d), np.uint16), ctx.empty((M, 4 * d), np.float32)
    print("fc1 index rows", M, flush=True)
    e.gemm_i8_fused(0, 4, ctx.array(x), 1, M, idx, side)
    y = oenc.gemm(0, 4, x)[1]
    inside = np.abs(y) < np.float32(9.98)
    gi = idx.download()
    np.testing.assert_array_equal(gi[inside], y[inside].astype(np.float16).view(np.uint16))
    assert np.all(gi[~inside] == 0xFFFF)
    assert_bitexact(side.download()[~inside], y[~inside], "fc1 side values")


@pytest.mark.parametrize("n,rows", [(5, 37), (3, 129), (14, 1499), (15, 1411)])
def test_residual_windows(pair, n, rows):
    """attn.out and fc2 add into the rows that they update: 128 x 128 tiles (few
    rows), 256 x 128 (21,000), with a last tile of a few rows."""
    ctx, e, _ = pair
    x = synth.mel_input(n, n, 2 * rows, CFG.n_mels) * np.float32(0.5)
    out, one = ctx.empty((n, rows, 384), np.float32), ctx.empty((1, rows, 384), np.float32)
    print("windows", n, "rows", rows, flush=True)
    e.forward_time_major(ctx.array(np.ascontiguousarray(x)), n, 2 * rows, out)
    got = out.download()
    for w in sorted({0, n // 2, n - 1}):
        e.forward_time_major(ctx.array(np.ascontiguousarray(x[w:w + 1])), 1, 2 * rows, one)
        assert_bitexact(got[w], one.download()[0], f"window {w} of {n}")


# Width 128: a tile of K = 128 has two steps, fewer than the stages in flight, and
# with more tiles than blocks a block's next tiles load their scales while it is
# still at the last ones'.  Row counts for which a CU (256 of them) takes two and
# three tiles.
NARROW = synth.Config("i8-narrow", 51864, 1500, 128, 2, 1, 64, 128, 2, 1, 16)


@pytest.fixture(scope="module")
def narrow():
    ctx = native.Context(0)
    m = synth.Model(NARROW, seed=9, decoder=False)
    e = native.Encoder(ctx, m, abi.ENC_INT8)
    yield ctx, e, O.Encoder(m, abi.ENC_INT8)
    e.close()
    ctx.close()


@pytest.mark.parametrize("M,which", [(66000, 0), (66000, 3), (33000, 4), (66000, 4), (66000, 5)])
def test_narrow_rows(narrow, M, which):
    ctx, e, oenc = narrow
    d = NARROW.n_audio_state
    inp, out = (4 * d if which == 5 else d), (4 * d if which == 4 else d)
    rng = np.random.default_rng(M + which)
    x = (rng.standard_normal((M, inp)) * rng.uniform(0.1, 3.0, (M, 1))).astype(np.float32)  # a scale of its own for every row
    acc, y = ctx.empty((M, out), np.int32), ctx.empty((M, out), np.float32)
    print("rows", M, "gemm", which, flush=True)
    e.gemm_i8(0, which, ctx.array(x), acc, y)
    want_acc, want_y = oenc.gemm(0, which, x)
    np.testing.assert_array_equal(acc.download(), want_acc)
    assert_bitexact(y.download(), want_y, f"rows {M} gemm {which}")


@pytest.mark.parametrize("exact", [False, True], ids=["fast", "exact"])
def test_narrow_windows(narrow, exact):
    """44 and 64 windows through every epilogue of the forward (q/k/v split or
    f32 rows, residual, index form): window for window the bits of a call with
    that window alone."""
    ctx, e, _ = narrow
    e.set_exact(exact)
    for n in (44,) if exact else (44, 64):
        x = synth.mel_input(n, n, 3000, NARROW.n_mels) * np.float32(0.5)
        out = ctx.empty((n, 1500, 128), np.float32)
        print("windows", n, "exact", exact, flush=True)
        e.forward_time_major(ctx.array(np.ascontiguousarray(x)), n, 3000, out)
        got, one = out.download(), ctx.empty((1, 1500, 128), np.float32)
        for w in (0, n // 3, n - 2, n - 1):
            e.forward_time_major(ctx.array(np.ascontiguousarray(x[w:w + 1])), 1, 3000, one)
            assert_bitexact(got[w], one.download()[0], f"window {w} of {n}")
    e.set_exact(False)
