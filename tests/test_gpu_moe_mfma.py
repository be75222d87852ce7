"""Expert products of buckets with many pairs on the matrix cores (gather.hip's
moe_mfma_kernel) against the CPU oracle, at the sizes where its tiles end.

Bar 1e-5 of max|oracle| for fp32 results of one product: the products of codes
and bf16 x are exact in fp32 on both sides, 64 .. 2048 of them are summed in
fp32 in another order: sqrt(2048) * 2^-24 = 2.7e-6 of the sum of magnitudes,
which is up to four times the largest result here. Through the SwiGLU block h is
bf16 on the device, so that one takes the parity bar of bf16 results, 1e-2.
"""
import numpy as np
import pytest

from janis_amd import synth
from janis_amd.engine import BF16, F16, F32
from tests.conftest import rel_ok, step, upload_quant

pytestmark = pytest.mark.gpu


def _upload(hip, q, sb):
    if sb == BF16:
        return upload_quant(hip, q), q.s, q.b
    s, b = q.s.astype(np.float16), q.b.astype(np.float16)
    w = upload_quant(hip, q)[0]
    return (w, hip.FromRaw(F16, s, *s.shape), hip.FromRaw(F16, b, *b.shape)), s.astype(np.float32), b.astype(np.float32)


def _buckets(sizes, k_slots, seed):
    """Expert indices [tokens, k_slots] with sizes[e] pairs of expert e, shuffled."""
    idx = np.concatenate([np.full(n, e, np.int32) for e, n in enumerate(sizes)])
    np.random.default_rng(seed).shuffle(idx)
    return idx.reshape(-1, k_slots)


# buckets around the tile's 32 and 64 pairs, an unused expert, several tiles of
# one bucket; rows that are no multiple of a wave's 32 or a block's 128; the
# shortest K and one that is not a power of two; both groups, both scale types.
# (Calls of fewer than 28 K rows of output stay on the dot products: three here,
# and each of them with more rows.)
@pytest.mark.parametrize("sizes,slots,n,k,gs,sb", [
    ((1, 31, 32, 0), 4, 128, 256, 64, BF16), ((33, 63, 64, 4), 4, 33, 768, 64, F16),
    ((65, 0, 130, 1, 4), 8, 100, 512, 128, BF16), ((2, 2, 2, 2, 128), 8, 257, 2048, 64, BF16),
    ((40, 40), 1, 160, 1536, 128, F16), ((33, 63, 64, 4), 4, 161, 768, 64, F16),
    ((2, 2, 2, 2, 128), 8, 433, 2048, 64, BF16), ((40, 40), 1, 545, 1536, 128, F16)])
def test_gather_mfma(hip, oracle, sizes, slots, n, k, gs, sb):
    E, idx = len(sizes), _buckets(sizes, slots, n + k)
    q = synth.quant_linear(810 + n, n, k, gs, lead=(E,))
    (w, s, b), sf, bf = _upload(hip, q, sb)
    for A in {1, slots}:
        xb, x = synth.activations(820 + A, (idx.shape[0], A, 1, k))
        step(f"jh_gather_quant_matmul buckets={sizes} A={A} n={n} k={k} gs={gs} sb={sb}")
        want = oracle.gather_quant_matmul(x, q.w, sf, bf, idx, gs)
        X, it = hip.FromBF16Bits(xb, idx.shape[0], A, 1, k), hip.FromInt32(idx)
        for out_dt, bar in ((F32, 1e-5), (BF16, 2.0 ** -8 + 1e-5)):
            y = hip.Floats(hip.GatherQuantMatmul(X, w, s, b, it, True, gs, 4, out_dtype=out_dt))
            ok, d, sc = rel_ok(y, want, bar)
            assert ok, (A, out_dt, d, sc)


@pytest.mark.parametrize("sizes,H,I,gs,out_dtype", [((1, 31, 0, 64), 256, 512, 64, F32),
                                                    ((65, 7, 96), 1024, 768, 128, BF16)])
def test_moe_swiglu_mfma(hip, oracle, sizes, H, I, gs, out_dtype):
    E, slots = len(sizes), 4
    idx = _buckets(sizes, slots, H)
    qs = [synth.quant_linear(830 + i + H, *(I, H) if i < 2 else (H, I), gs, lead=(E,)) for i in range(3)]
    sc = np.random.default_rng(I).random(idx.shape).astype(np.float32)
    xb, x = synth.activations(831, (idx.shape[0], H))
    st = [upload_quant(hip, q) for q in qs]
    args = (hip.FromBF16Bits(xb, *x.shape), *st, hip.FromInt32(idx), hip.FromFloats(sc), gs, 4)
    step(f"jh_moe_swiglu buckets={sizes} H={H} I={I} gs={gs}")
    first = hip.Floats(hip.MoeSwiGLU(*args, out_dtype=out_dtype))
    ok, d, s = rel_ok(first, oracle.moe_apply(x, *[(q.w, q.s, q.b) for q in qs], idx, sc, gs), 1e-2)
    assert ok, (d, s)
    again = hip.Floats(hip.MoeSwiGLU(*args, out_dtype=out_dtype))
    assert np.array_equal(first.view(np.uint32), again.view(np.uint32))


@pytest.mark.parametrize("n", [64, 232])
def test_gather_mfma_rows_apart(hip, oracle, n):
    """A pair whose x holds a NaN or an infinity, and one with an index outside
    the stack, leave the other pairs of their bucket and tile alone."""
    E, k = 2, 512
    idx = _buckets((40, 24), 4, 3)
    q = synth.quant_linear(840, n, k, lead=(E,))
    w, s, b = upload_quant(hip, q)
    xb, x = synth.activations(841, (16, 4, 1, k))
    xb, x = xb.copy(), x.copy()
    for at, bits in (((3, 1, 0, 5), 0x7FC0), ((9, 2, 0, 300), 0x7F80)):
        xb[at] = bits
        x[at] = synth.bf16_bits_to_f32(np.uint16(bits))
    want = oracle.gather_quant_matmul(x, q.w, q.s, q.b, idx, 64)
    idx = idx.copy()
    idx[12, 0] = E
    step("jh_gather_quant_matmul, rows that are not finite")
    y = hip.Floats(hip.GatherQuantMatmul(hip.FromBF16Bits(xb, 16, 4, 1, k), w, s, b, hip.FromInt32(idx), True, 64, 4,
                                         out_dtype=F32))
    odd = np.zeros((16, 4), bool)
    odd[3, 1] = odd[9, 2] = odd[12, 0] = True
    assert not np.isfinite(y[3, 1]).any() and not np.isfinite(y[9, 2]).any() and np.isnan(y[12, 0]).all()
    ok, d, sc = rel_ok(y[~odd], want[~odd], 1e-5)
    assert ok, (d, sc)


# the register router at the ends of its sizes (64 * 1, 2, 4, 8 experts, and the
# first size past them), ties and rows that are not finite included
@pytest.mark.parametrize("E,k", [(1, 1), (63, 63), (64, 8), (65, 8), (128, 8), (129, 3), (256, 16), (257, 8), (512, 8),
                                 (513, 8)])
def test_moe_route_sizes(hip, oracle, E, k):
    """Bit for bit the CPU path's indices and scores."""
    rng = np.random.default_rng(E)
    logits = np.concatenate([rng.standard_normal((3, E)), rng.integers(0, 3, (3, E)), rng.standard_normal((2, E))])
    logits = logits.astype(np.float32)
    logits[6, E // 2] = np.nan
    logits[7, E // 3] = np.inf
    step(f"jh_moe_route E={E} k={k}")
    it, st = hip.MoeRoute(hip.FromFloats(logits), k, True)
    got_i, got_s = hip.Ints(it), hip.Floats(st)
    for t in range(6):
        p = oracle.softmax_row(logits[t])
        i, v = oracle.topk(p, k)
        total = np.float32(0)
        for x in v:
            total = np.float32(total + x)
        assert np.array_equal(got_i[t], i), t
        assert np.array_equal(got_s[t].view(np.uint32), (v / total).astype(np.float32).view(np.uint32)), t
    # a NaN or an infinity makes every probability NaN: nothing is larger than
    # the first, so the order stays
    assert np.array_equal(got_i[6:], np.tile(np.arange(k, dtype=np.int32), (2, 1))) and np.isnan(got_s[6:]).all()


@pytest.mark.parametrize("n", [64, 232])
@pytest.mark.parametrize("gs", [64, 128])
def test_gather_scales_at_two_bytes(hip, oracle, gs, n):
    """Scales and biases that start at an odd element (2-byte aligned) keep
    their results: such calls stay on the dot products."""
    E, k = 2, 512
    idx = _buckets((40, 24), 4, 5)
    q = synth.quant_linear(850, n, k, gs, lead=(E,))
    w = upload_quant(hip, q)[0]
    shifted = []
    for bits in (q.s_bits, q.b_bits):
        flat = hip.FromBF16Bits(np.concatenate([np.zeros(1, np.uint16), np.asarray(bits, np.uint16).ravel()]),
                                bits.size + 1)
        shifted.append(hip.Wrap(flat.ptr + 2, bits.shape, BF16, keep=flat))
    xb, x = synth.activations(851, (16, 4, 1, k))
    step(f"jh_gather_quant_matmul, scales 2-byte aligned, gs={gs}")
    y = hip.Floats(hip.GatherQuantMatmul(hip.FromBF16Bits(xb, 16, 4, 1, k), w, *shifted, hip.FromInt32(idx), True, gs, 4,
                                         out_dtype=F32))
    ok, d, sc = rel_ok(y, oracle.gather_quant_matmul(x, q.w, q.s, q.b, idx, gs), 1e-5)
    assert ok, (d, sc)


# either side of the lines between the dot products and the matrix cores: 28 K rows
# of output for one stack, 80000 + 10 K for two (pairs times rows)
@pytest.mark.parametrize("n,k", [(335, 768), (336, 768), (223, 512), (224, 512), (895, 2048), (896, 2048)])
def test_gather_at_the_line(hip, oracle, n, k):
    E, idx = 8, _buckets((9, 3, 0, 17, 1, 16, 8, 10), 4, 7)
    q = synth.quant_linear(860 + n, n, k, lead=(E,))
    xb, x = synth.activations(861, (16, 1, 1, k))
    step(f"jh_gather_quant_matmul 64 pairs n={n} k={k}")
    y = hip.Floats(hip.GatherQuantMatmul(hip.FromBF16Bits(xb, 16, 1, 1, k), *upload_quant(hip, q), hip.FromInt32(idx), True,
                                         64, 4, out_dtype=F32))
    ok, d, sc = rel_ok(y, oracle.gather_quant_matmul(x, q.w, q.s, q.b, idx, 64), 1e-5)
    assert ok, (d, sc)


@pytest.mark.parametrize("I", [512, 768])
@pytest.mark.parametrize("slots", [4, 9, 16, 17])
def test_moe_swiglu_slots(hip, oracle, I, slots):
    """More than eight slots per token (the sum over slots takes eight at a time),
    an index outside the stack among them; gate and up on the dot products or on
    the matrix cores, down on the matrix cores."""
    E, H, T = 18, 512, 6
    rng = np.random.default_rng(slots)
    idx = np.stack([rng.permutation(E)[:slots] for _ in range(T)]).astype(np.int32)
    qs = [synth.quant_linear(870 + i, *(I, H) if i < 2 else (H, I), 64, lead=(E,)) for i in range(3)]
    sc = rng.random(idx.shape).astype(np.float32)
    xb, x = synth.activations(871, (T, H))
    want = oracle.moe_apply(x, *[(q.w, q.s, q.b) for q in qs], idx, sc, 64)
    idx[2, slots - 1] = E
    st = [upload_quant(hip, q) for q in qs]
    step(f"jh_moe_swiglu slots={slots} I={I}")
    got = hip.Floats(hip.MoeSwiGLU(hip.FromBF16Bits(xb, T, H), *st, hip.FromInt32(idx), hip.FromFloats(sc), 64, 4,
                                   out_dtype=F32))
    keep = np.arange(T) != 2
    assert np.isnan(got.reshape(T, H)[2]).all()
    ok, d, s = rel_ok(got.reshape(T, H)[keep], want.reshape(T, H)[keep], 1e-2)
    assert ok, (d, s)
