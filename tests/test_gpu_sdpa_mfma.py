"""SDPA with several query rows per head on the matrix cores (attention.hip),
against the CPU oracle at the sizes where its tiles end.

Bar 1e-5 of max|oracle| for fp32 results: both sides sum a score's 128 products
in fp32, so a score of |s| <= 8 is off by up to about sqrt(128) * 2^-24 * 8 =
5e-6 on each side, which is the relative error of that key's weight. bf16
results add their own rounding, half a unit of an 8-bit significand: 2^-8.
"""
import numpy as np
import pytest

from janis_amd import synth
from janis_amd.engine import BF16, F16, F32
from tests.conftest import Graph, rel_ok, step

pytestmark = pytest.mark.gpu
D = 128


def _put(hip, a, dt):
    a = np.asarray(a, np.float32)
    if dt == BF16:
        return hip.FromBF16Bits(synth.f32_to_bf16_bits(a), *a.shape)
    if dt == F16:
        return hip.FromRaw(F16, a.astype(np.float16), *a.shape)
    return hip.FromFloats(a, *a.shape)


def _round(a, dt):
    if dt == BF16:
        return synth.bf16_bits_to_f32(synth.f32_to_bf16_bits(a))
    return a.astype(np.float16).astype(np.float32) if dt == F16 else a


def _case(B, Hq, Hk, Lq, Lk, q_dt, kv_dt, spread=1.5):
    rng = np.random.default_rng(Lq * 1009 + Lk * 7 + Hq)
    q = _round((spread * rng.standard_normal((B, Hq, Lq, D))).astype(np.float32), q_dt)
    k = _round((spread * rng.standard_normal((B, Hk, Lk, D))).astype(np.float32), kv_dt)
    v = _round(rng.standard_normal((B, Hk, Lk, D)).astype(np.float32), kv_dt)
    return q, k, v


def _cache(hip, a, dt, cap):
    """a's rows at the start of a [B, H, cap, D] buffer whose other rows are NaN."""
    B, H, L, _ = a.shape
    full = np.full((B, H, cap, D), np.nan, np.float32)
    full[:, :, :L] = a
    return _put(hip, full, dt)


# rows of a kv head (Hq / Hk * Lq) and keys around the wave's 32, the block's 128
# and the key tile's 64; several blocks; calls split over the keys (Lk >= 512
# with few rows); group sizes that are no power of two; a batch
@pytest.mark.parametrize("B,Hq,Hk,Lq,Lk,causal", [
    (1, 2, 2, 2, 2, True), (1, 1, 1, 32, 64, True), (1, 1, 1, 33, 65, True), (1, 4, 1, 32, 63, False),
    (2, 6, 2, 43, 129, True), (1, 8, 8, 127, 128, True), (1, 5, 1, 26, 191, False), (1, 16, 2, 7, 1025, True),
    (1, 8, 8, 3, 512, False), (1, 4, 4, 200, 700, True)])
@pytest.mark.parametrize("q_dt,kv_dt", [(F32, F16), (BF16, F16), (F32, BF16), (BF16, BF16)])
def test_sdpa_mfma(hip, oracle, B, Hq, Hk, Lq, Lk, causal, q_dt, kv_dt):
    q, k, v = _case(B, Hq, Hk, Lq, Lk, q_dt, kv_dt)
    kc, vc = _cache(hip, k, kv_dt, Lk + 5), _cache(hip, v, kv_dt, Lk + 5)
    step(f"jh_sdpa rows B={B} Hq={Hq} Hk={Hk} Lq={Lq} Lk={Lk} causal={causal} q={q_dt} kv={kv_dt}")
    want = oracle.sdpa(q, k, v, D ** -0.5, causal)
    for out_dt, bar in ((F32, 1e-5), (BF16, 2.0 ** -8 + 1e-5)):
        got = hip.Floats(hip.SDPA(_put(hip, q, q_dt), kc, vc, D ** -0.5, causal, kv_len=Lk, out_dtype=out_dt))
        ok, dd, sc = rel_ok(got, want, bar)
        assert ok, (out_dt, dd, sc)


@pytest.mark.parametrize("scale,bar", [(0.0, 1e-5), (1e-3, 1e-5), (-0.1, 1.4e-4), (3.0, 7e-4)])
def test_sdpa_mfma_scales(hip, oracle, scale, bar):
    """The scale's sign and size, rows of q of very different sizes (a row's own
    power of two for f16 keys) and scores far apart: scores of up to 100 (scale
    -0.1) and 500 (scale 3) are off by sqrt(128) * 2^-24 times that, 7e-5 and
    3.4e-4, on each side."""
    q, k, v = _case(1, 2, 1, 20, 90, F32, F16)
    q *= (10.0 ** np.linspace(-6, 1, 20, dtype=np.float32))[None, None, :, None] * (1.0 if scale < 1 else 0.1)
    step(f"jh_sdpa rows scale={scale}")
    got = hip.Floats(hip.SDPA(_put(hip, q, F32), _put(hip, k, F16), _put(hip, v, F16), scale, True))
    ok, dd, sc = rel_ok(got, oracle.sdpa(q, k, v, scale, True), bar)
    assert ok, (dd, sc)


@pytest.mark.parametrize("kv_dt", [F16, BF16])
@pytest.mark.parametrize("Lk", [100, 600])
def test_sdpa_mfma_values_not_finite(hip, oracle, Lk, kv_dt):
    """An infinity or NaN in a key or value row reaches the rows that attend to
    it and no other, also inside one tile and one split."""
    Lq = 40
    q, k, v = _case(1, 4, 2, Lq, Lk, F32, kv_dt)
    v[0, 0, Lk - 10, 3] = np.inf   # seen by the last 10 queries of kv head 0
    v[0, 1, Lk - 20, 7] = np.nan   # ... the last 20 of kv head 1
    k[0, 1, Lk - 5, 9] = np.nan    # ... the last 5: all their features
    step(f"jh_sdpa rows, values not finite, Lk={Lk}")
    got = hip.Floats(hip.SDPA(_put(hip, q, F32), _put(hip, k, kv_dt), _put(hip, v, kv_dt), D ** -0.5, True))
    with np.errstate(all="ignore"):
        want = oracle.sdpa(q, k, v, D ** -0.5, True)
    assert np.isposinf(want[0, :2, Lq - 10:, 3]).all() and np.isnan(want[0, 2:, Lq - 20:, 7]).all()
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    fine = np.isfinite(want)
    ok, dd, sc = rel_ok(got[fine], want[fine], 1e-5)
    assert ok, (dd, sc)


def test_sdpa_mfma_captured_without_workspace(oracle):
    """A call that would split its keys still captures on a context whose
    workspace was never sized (it runs unsplit), and replays to its result."""
    from janis_amd.engine import HipBackend

    b = HipBackend(0)
    q, k, v = _case(1, 4, 2, 9, 1500, F32, F16)
    Q, K, V = _put(b, q, F32), _put(b, k, F16), _put(b, v, F16)
    arena = b.make_arena(1 << 20)
    out = []
    with b.use_arena(arena):
        step("jh_sdpa rows captured first")
        g = Graph(b, lambda: out.append(b.SDPA(Q, K, V, D ** -0.5, True)))
    want = oracle.sdpa(q, k, v, D ** -0.5, True)
    for _ in range(3):
        g.replay()
        ok, dd, sc = rel_ok(b.Floats(out[-1]), want, 1e-5)
        assert ok, (dd, sc)
    b.Close()


@pytest.mark.parametrize("kv_dt", [F16, BF16])
@pytest.mark.parametrize("Lk", [200, 700])
@pytest.mark.parametrize("gap", [6, 12, 16, 20, 30, 45])
def test_sdpa_mfma_dominant_key(hip, gap, Lk, kv_dt):
    """One key holds all but 2^-gap of a row's weight and its values are zero (an
    attention sink): the result is the sum over the small probabilities, which
    keep fp32's relative precision. A score of gap * ln 2 nats and its difference
    to the maximum are rounded to fp32 (the dominant score is exact, the others
    are below 2): 2^-24 of gap each way of writing it, three roundings, and the
    exponential's and the sums' own 2^-22."""
    Lq = 40
    q, k, v = _case(1, 2, 1, Lq, Lk, F32, kv_dt, spread=0.2)
    at = Lk // 3
    q[..., 0] = 1.0
    k[..., 0] = 0.0
    k[0, 0, at] = 0.0
    k[0, 0, at, 0] = _round(np.float32([gap * np.log(2.0)]), kv_dt)[0]
    v[0, 0, at] = 0.0
    step(f"jh_sdpa rows, a dominant key, gap={gap} Lk={Lk} kv={kv_dt}")
    got = hip.Floats(hip.SDPA(_put(hip, q, F32), _put(hip, k, kv_dt), _put(hip, v, kv_dt), 1.0, False)).astype(np.float64)
    s = q[0].astype(np.float64) @ k[0, 0].astype(np.float64).T
    p = np.exp(s - s.max(-1, keepdims=True))
    want = (p @ v[0, 0].astype(np.float64)) / p.sum(-1, keepdims=True)
    err = np.linalg.norm(got[0] - want, axis=-1) / np.linalg.norm(want, axis=-1)
    assert err.max() <= 2.0 ** -22 + 3 * gap * 2.0 ** -24, err.max()


@pytest.mark.parametrize("q_dt,kv_dt", [(F32, F16), (BF16, F16), (F32, BF16), (BF16, BF16)])
@pytest.mark.parametrize("Lk,dead", [(100, 70), (700, 400)])
def test_sdpa_mfma_scores_of_minus_infinity(hip, oracle, Lk, dead, q_dt, kv_dt):
    """Keys whose scores are -inf have no weight, also where they fill whole key
    tiles and whole splits; a row with no other key is NaN."""
    q, k, v = _case(1, 4, 2, 20, Lk, q_dt, kv_dt)
    q[..., 0] = 1.0
    k[:, :, :dead, 0] = -np.inf
    k[:, 1, :, 0] = -np.inf
    step(f"jh_sdpa rows, scores of -inf, Lk={Lk} q={q_dt} kv={kv_dt}")
    got = hip.Floats(hip.SDPA(_put(hip, q, q_dt), _put(hip, k, kv_dt), _put(hip, v, kv_dt), D ** -0.5, True, out_dtype=F32))
    with np.errstate(all="ignore"):
        want = oracle.sdpa(q, k, v, D ** -0.5, True)
    assert np.isfinite(want[:, :2]).all() and np.isnan(want[:, 2:]).all()
    assert np.isnan(got[:, 2:]).all()
    ok, dd, sc = rel_ok(got[:, :2], want[:, :2], 1e-5)
    assert ok, (dd, sc)


@pytest.mark.parametrize("kv_dt", [F16, BF16])
@pytest.mark.parametrize("Lk", [70, 700])
@pytest.mark.parametrize("n", [1, 7, 8, 9, 33, 60])
def test_sdpa_mfma_rows_again(hip, oracle, n, Lk, kv_dt):
    """Rows that are not finite are computed again eight at a time: fewer, exactly
    eight, and more of them, with values that are not finite (one pass over the
    keys) and a query that is NaN (two)."""
    Lq = 60
    q, k, v = _case(1, 1, 1, Lq, Lk, F32, kv_dt)
    v[0, 0, Lk - n, 5] = -np.inf   # seen by the last n queries, in the tile of others
    v[0, 0, Lk - n, 64] = np.nan
    q[0, 0, 11, 3] = np.nan
    step(f"jh_sdpa rows computed again, n={n} Lk={Lk} kv={kv_dt}")
    got = hip.Floats(hip.SDPA(_put(hip, q, F32), _put(hip, k, kv_dt), _put(hip, v, kv_dt), D ** -0.5, True))
    with np.errstate(all="ignore"):
        want = oracle.sdpa(q, k, v, D ** -0.5, True)
    seen = [i for i in range(Lq - n, Lq) if i != 11]
    assert np.isneginf(want[0, 0, seen, 5]).all() and np.isnan(want[0, 0, 11]).all()
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    fine = np.isfinite(want)
    ok, dd, sc = rel_ok(got[fine], want[fine], 1e-5)
    assert ok, (dd, sc)


@pytest.mark.parametrize("scale", [0.0, -0.0, 1e-38, 1e-30])
def test_sdpa_mfma_scale_of_nothing(hip, oracle, scale):
    """Scores of up to 1e38 times a scale of zero, or next to it, are zero (1e-38
    of them at most 1, 1e-30 far from it: the smallest on the matrix cores)."""
    q, k, v = _case(1, 2, 1, 20, 90, BF16, BF16)
    q, k = _round(q * np.float32(1e18), BF16), _round(k * np.float32(1e18), BF16)
    step(f"jh_sdpa rows scale={scale} of scores of 1e38")
    got = hip.Floats(hip.SDPA(_put(hip, q, BF16), _put(hip, k, BF16), _put(hip, v, BF16), scale, True, out_dtype=F32))
    ok, dd, sc = rel_ok(got, oracle.sdpa(q, k, v, scale, True), 1e-5)
    assert ok, (dd, sc)


def test_sdpa_mfma_captured_with_some_workspace(oracle):
    """Captured on a context whose workspace holds some of the splits' partials,
    a call takes those: neither the bits of the unsplit sums nor an error."""
    from janis_amd.engine import HipBackend

    q, k, v = _case(1, 4, 2, 9, 1500, F32, F16)
    want = oracle.sdpa(q, k, v, D ** -0.5, True)
    got = []
    for keys in (None, 150):  # no workspace; one for 150 keys in parts of 64
        b = HipBackend(0)
        Q, K, V = _put(b, q, F32), _put(b, k, F16), _put(b, v, F16)
        if keys:
            b.SDPA(Q, _put(b, k[:, :, :keys], F16), _put(b, v[:, :, :keys], F16), D ** -0.5, True)
        arena, out = b.make_arena(1 << 20), []
        with b.use_arena(arena):
            step(f"jh_sdpa rows captured after {keys} keys")
            g = Graph(b, lambda: out.append(b.SDPA(Q, K, V, D ** -0.5, True)))
        for _ in range(3):
            g.replay()
            got.append(b.Floats(out[-1]))
            ok, dd, sc = rel_ok(got[-1], want, 1e-5)
            assert ok, (dd, sc)
        b.Close()
    assert not np.array_equal(got[0], got[-1])
