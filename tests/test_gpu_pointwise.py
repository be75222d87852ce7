"""Element-wise operators and strided copies where their 16-byte paths begin and
end: lengths and runs that are no multiple of 8, buffers off a 16-byte boundary,
dimensions that merge and that do not, every pair of float types."""
import ctypes

import numpy as np
import pytest

from janis_amd import _lib, synth
from janis_amd.engine import BF16, F16, F32, I32, U8
from tests.conftest import step

pytestmark = pytest.mark.gpu
SIZE = {F32: 4, F16: 2, BF16: 2, I32: 4, U8: 1}


def _bits(a, dt):
    """Float32 values as the bytes of dtype dt, and the values those hold."""
    a = np.asarray(a, np.float32)
    if dt == BF16:
        b = synth.f32_to_bf16_bits(a)
        return b, synth.bf16_bits_to_f32(b)
    if dt == F16:
        b = a.astype(np.float16)
        return b, b.astype(np.float32)
    return a, a


def _at(hip, raw, dt, shift):
    """raw on the device, `shift` elements past a 16-byte boundary."""
    pad = np.zeros(shift, raw.dtype)
    t = hip.FromRaw(dt, np.concatenate([pad, raw.reshape(-1)]), shift + raw.size)
    return t, t.ptr + shift * SIZE[dt]


# (Add and Mul move pieces of 8 from 2^19 elements on, SiLU from 5 * 2^18)
@pytest.mark.parametrize("n", [1, 7, 8, 2049, 12288, (1 << 19) + 5, (1 << 20) - 1, (1 << 20) + 3, (5 << 18) - 1,
                               (5 << 18) + 3])
@pytest.mark.parametrize("a_dt,b_dt,o_dt,shift", [(F32, F32, F32, 0), (BF16, BF16, BF16, 0), (F32, BF16, BF16, 0),
                                                  (BF16, F32, F32, 0), (F32, F32, F32, 1), (BF16, BF16, F32, 3)])
def test_elementwise_sizes(hip, oracle, n, a_dt, b_dt, o_dt, shift):
    rng = np.random.default_rng(n + shift)
    ra, a = _bits(rng.standard_normal(n) * 30, a_dt)
    rb, b = _bits(rng.standard_normal(n), b_dt)
    if n > 7 and a_dt == F32:
        ra[:7] = a[:7] = [np.nan, np.inf, -np.inf, 104.5, -104.5, 1e-30, -88.9]
    (ta, pa), (tb, pb) = _at(hip, ra, a_dt, shift), _at(hip, rb, b_dt, shift)
    for op, want in ((_lib.JH_OP_ADD, a + b), (_lib.JH_OP_MUL, a * b), (_lib.JH_OP_SILU, oracle.silu(a)),
                     (_lib.JH_OP_SILU_MUL, oracle.silu(a) * b)):
        to, po = _at(hip, np.zeros(n, _bits(0, o_dt)[0].dtype), o_dt, shift)
        step(f"jh_elementwise op={op} n={n} {a_dt},{b_dt}->{o_dt} shift={shift}")
        _lib.check(hip._ctx, hip._L.jh_elementwise(hip._ctx, op, pa, a_dt, pb, b_dt, n, po, o_dt))
        got = hip.Floats(to)[shift:]
        with np.errstate(all="ignore"):
            if op in (_lib.JH_OP_ADD, _lib.JH_OP_MUL):
                np.testing.assert_array_equal(got, _bits(want, o_dt)[1])
                continue
            # the exponential is right to 2^-46 before it is rounded, as the
            # oracle's is: at most a unit of fp32 where it lies on a tie, then the
            # same sum and quotient, the product by b and the rounding of the result
            assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
            f = np.isfinite(want)
            # (below the smallest normal value, half a unit of the subnormal ones: 2^-134
            # in bf16; products that small occur among 2^20 values)
            bar, tiny = {F32: (2.0 ** -22, 1e-44), BF16: (2.0 ** -8, 2.0 ** -134)}[o_dt]
            assert (np.abs(got[f] - want[f]) <= bar * np.abs(want[f]) + tiny).all()


@pytest.mark.parametrize("shape,perm,cut", [
    ((1, 37, 6, 128), (0, 2, 1, 3), None),      # heads and tokens exchanged
    ((2, 3, 5, 16), (2, 0, 1, 3), None),        # two outer dimensions that do not merge
    ((3, 4, 5, 2, 8), (4, 3, 2, 1, 0), None),   # nothing contiguous
    ((4, 6, 24), (0, 1, 2), (1, 1, 5)),         # rows 1..4 of a longer axis
    ((5, 4, 12), (1, 0, 2), None),              # runs of 12
    ((64,), (0,), None), ((7,), (0,), None)])
@pytest.mark.parametrize("s_dt,d_dt,shift", [(F32, F32, 0), (BF16, BF16, 0), (F32, F16, 0), (BF16, F16, 0), (F16, F32, 0),
                                             (F32, BF16, 0), (BF16, BF16, 1), (F32, F32, 2)])
def test_copy_shapes(hip, shape, perm, cut, s_dt, d_dt, shift):
    rng = np.random.default_rng(len(shape) + shape[0])
    raw, val = _bits(rng.standard_normal(shape) * 3, s_dt)
    t, p = _at(hip, raw, s_dt, shift)
    st = np.array(val.strides) // 4
    view, off = val, 0
    if cut:
        ax, lo, hi = cut
        view = np.take(val, range(lo, hi), ax)
        off = lo * int(st[ax])
    shp, ss = [view.shape[i] for i in perm], [int(st[i]) for i in perm]
    want = _bits(np.transpose(view, perm), d_dt)[1]
    out, po = _at(hip, np.zeros(want.size, _bits(0, d_dt)[0].dtype), d_dt, shift)
    step(f"jh_copy_strided {shape} perm={perm} cut={cut} {s_dt}->{d_dt} shift={shift}")
    c = ctypes.c_int64 * len(shp)
    _lib.check(hip._ctx, hip._L.jh_copy_strided(hip._ctx, p + off * SIZE[s_dt], s_dt, len(shp), c(*shp), c(*ss), po, d_dt,
                                                None))
    np.testing.assert_array_equal(hip.Floats(out)[shift:], want.reshape(-1))


def test_copy_broadcast_and_reverse(hip):
    """Zero and negative strides, and a destination with strides of its own."""
    a = np.arange(4 * 16, dtype=np.float32).reshape(4, 16)
    t = hip.FromFloats(a)
    c = ctypes.c_int64 * 3
    out = hip.FromFloats(np.full((2, 3, 40), -1, np.float32))
    step("jh_copy_strided broadcast, reversed rows, strided destination")
    _lib.check(hip._ctx, hip._L.jh_copy_strided(hip._ctx, t.ptr + 3 * 16 * 4, F32, 3, c(2, 3, 16), c(0, -16, 1), out.ptr,
                                                F32, c(120, 40, 1)))
    want = np.full((2, 3, 40), -1, np.float32)
    want[:, :, :16] = a[3:0:-1]
    np.testing.assert_array_equal(hip.Floats(out), want)


@pytest.mark.parametrize("heads,L,D,dims,traditional", [(1, 1, 128, 128, False), (40, 700, 128, 128, False),
                                                        (33, 300, 96, 64, False), (6, 301, 64, 64, True),
                                                        (130, 70, 128, 32, False),
                                                        (39, 700, 128, 128, False), (67, 500, 128, 128, True),
                                                        (8, 512, 128, 128, False)])
@pytest.mark.parametrize("dt", [F32, BF16])
def test_rope_head_groups(hip, oracle, heads, L, D, dims, traditional, dt):
    """Heads that share a position's factors (one, two, four and eight per thread),
    in whole groups and not."""
    rng = np.random.default_rng(heads + L)
    raw, x = _bits(rng.standard_normal((1, heads, L, D)), dt)
    t = hip.FromRaw(dt, raw, *raw.shape)
    step(f"jh_rope heads={heads} L={L} D={D} dims={dims} {dt}")
    got = hip.Floats(hip.RoPE(t, dims, traditional, 1e6, 1.0, 17, out_dtype=F32))
    want = oracle.rope(x, dims, traditional, 1e6, 1.0, 17)
    assert np.abs(got - want).max() <= 1e-6 * np.abs(want).max()  # two products and a sum: 3 * 2^-24, and a rounded angle
    # a call of fewer rows than positions, and one that ends inside a head
    for rows, Lc in ((3, 1000), (L + L // 2, L)):
        if rows <= heads * L:
            out = hip.FromFloats(np.zeros((rows, D), np.float32))
            _lib.check(hip._ctx, hip._L.jh_rope(hip._ctx, t.ptr, dt, rows, Lc, D, dims, int(traditional), 1e6, 1.0, 17, None,
                                                out.ptr, F32))
            np.testing.assert_array_equal(hip.Floats(out), got.reshape(-1, D)[:rows])


@pytest.mark.parametrize("rows,d", [(3, 1), (5, 63), (2, 128), (2, 129), (3, 256), (3, 257), (5, 300), (2, 512), (2, 513),
                                    (9, 1024), (2, 1025), (2, 2048), (2, 2049), (3, 4095), (2, 4097), (2, 6144), (2, 6145),
                                    (2, 8192), (2, 8193), (1, 12288), (1, 12289), (1, 16384), (2, 16385)])
@pytest.mark.parametrize("x_dt,w_dt", [(F32, BF16), (BF16, F16), (BF16, F32)])
def test_rms_norm_lengths(hip, rows, d, x_dt, w_dt):
    """Row lengths at the ends of each kernel's range, odd ones among them. The first
    and the last element of a row hold most of its sum of squares, so that one left
    out or taken twice shows at every length."""
    rng = np.random.default_rng(rows * d)
    x = rng.standard_normal((rows, d))
    x[:, 0], x[:, -1] = np.sqrt(d), -1.5 * np.sqrt(d)
    rx, x = _bits(x, x_dt)
    rw, w = _bits(1 + 0.1 * rng.standard_normal(d), w_dt)
    step(f"jh_rms_norm rows={rows} d={d} x={x_dt} w={w_dt}")
    got = hip.Floats(hip.RMSNorm(hip.FromRaw(x_dt, rx, rows, d), hip.FromRaw(w_dt, rw, d), 1e-6, out_dtype=F32))
    x64 = x.astype(np.float64)
    want = x64 / np.sqrt((x64 ** 2).mean(-1, keepdims=True) + 1e-6) * w
    # a thread adds up to 65 squares one after another and 8 sums follow: 73 * 2^-24
    # of the sum, half that in its root; then a quotient, a root and two products
    assert (np.abs(got - want) <= (37 + 5) * 2.0 ** -24 * np.abs(want)).all()
