"""Attention in f32 (every head size) and in 16 bits with heads of 32, on the MFMA kernels: against
softmax(q k^T / sqrt(d)) v in f64.

Bars: f32 1e-5 of the largest output (the f32 bar used throughout; sums of up to 1000 terms of one
sign and magnitude carry a few 2^-24); 16 bits one rounding of the output, half a unit in the last
place of the largest output (at most 2^-8 of it in bf16, whose significands have 8 bits, 2^-11 in f16)
and 2e-5 on top: the probabilities are two 16-bit values, within 2^-17 (f16: 2^-22) of themselves, and
their sums f32."""
import numpy as np
import pytest

import kurumi_amd as K
from kurumi_amd import DType, Tensor
from kutest import bf16_bits_to_f32, f32_to_bf16_bits, to_f32

pytestmark = pytest.mark.gpu


def f64_attention(q, k, v, causal, scale=None):
    s = np.einsum("...qd,...kd->...qk", q, k) * (q.shape[-1] ** -0.5 if scale is None else scale)
    if causal:
        s = np.where(np.tril(np.ones(s.shape[-2:], bool)), s, -np.inf)
    e = np.exp(s - s.max(-1, keepdims=True))
    return np.einsum("...qk,...kd->...qd", e / e.sum(-1, keepdims=True), v)


def run(hip, dt, arrays, causal, label):
    g = K.Graph()
    ids = [g.input(a.shape, dt) for a in arrays]
    if dt == DType.F32:
        feeds = {i: Tensor.from_numpy(a) for i, a in zip(ids, arrays)}
    elif dt == DType.BF16:
        feeds = {i: Tensor(dt, a.shape, f32_to_bf16_bits(a).tobytes()) for i, a in zip(ids, arrays)}
    else:
        feeds = {i: Tensor(dt, a.shape, a.astype(np.float16).tobytes()) for i, a in zip(ids, arrays)}
    o = g.sdpa(*ids, causal)
    plan = hip.plan(g, [o], feeds)
    assert plan.steps()[0].startswith(label), plan.steps()
    plan.launch()
    return to_f32(plan.output(0))


# one query; on both sides of the few positions that take the one-query-per-thread kernel (to 4
# with heads of 32, 5 with 64, 3 with 128); a tile less one and plus one; keys for one, some and all of a group's four
# waves; a last partial block in each
SHAPES = [(1, 1, 1), (1, 3, 2), (2, 5, 3), (1, 5, 4), (1, 5, 5), (1, 2, 6), (2, 1, 31), (1, 3, 33), (1, 2, 100), (2, 2, 128), (1, 2, 500), (1, 1, 1000)]


@pytest.mark.parametrize("b,h,s", SHAPES)
@pytest.mark.parametrize("d", [32, 64, 128])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("std", [1.0, 6.0])
def test_f32_attention_matches_f64(hip, b, h, s, d, causal, std):
    print(f"f32 attention {b}x{h}x{s}x{d} causal={causal} std={std}", flush=True)
    rng = np.random.default_rng(s * 10 + d)
    q, k, v = (rng.standard_normal((b, h, s, d)).astype(np.float32) * np.float32(x) for x in (std, 1.0, 1.0))
    got = run(hip, DType.F32, [q, k, v], causal, "attn_rowwise" if s <= {32: 4, 64: 5, 128: 3}[d] else "attn_mfma_f32")
    want = f64_attention(*(x.astype(np.float64) for x in (q, k, v)), causal)
    assert np.abs(got - want).max() <= 1e-5 * np.abs(want).max()


@pytest.mark.parametrize("b,h,s", SHAPES)
@pytest.mark.parametrize("dt", [DType.BF16, DType.F16])
@pytest.mark.parametrize("causal", [False, True])
def test_16_bit_heads_of_32_match_f64(hip, b, h, s, dt, causal):
    print(f"{dt.name} attention {b}x{h}x{s}x32 causal={causal}", flush=True)
    rng = np.random.default_rng(s)
    arrays = [rng.standard_normal((b, h, s, 32)).astype(np.float32) for _ in range(3)]
    arrays = [bf16_bits_to_f32(f32_to_bf16_bits(x)) if dt == DType.BF16 else x.astype(np.float16).astype(np.float32) for x in arrays]
    got = run(hip, dt, arrays, causal, "attn_rowwise" if s <= 4 else "attn_mfma ")
    # the scale is a scalar of the operands' type
    scale = np.float32(32 ** -0.5)
    scale = bf16_bits_to_f32(f32_to_bf16_bits(scale)) if dt == DType.BF16 else np.float16(scale)
    want = f64_attention(*(x.astype(np.float64) for x in arrays), causal, float(scale))
    assert np.abs(got - want).max() <= (2.0 ** (-8 if dt == DType.BF16 else -11) + 2e-5) * np.abs(want).max()


@pytest.mark.parametrize("d", [32, 64, 128])
def test_f32_causal_attention_never_reads_what_a_query_does_not_see(hip, d):
    """Infinities and NaN in later keys and values leave earlier queries' bits alone; the queries
    that see them get what f64 gives."""
    s, p = 150, 40
    rng = np.random.default_rng(d)
    q, k, v = (rng.standard_normal((1, 2, s, d)).astype(np.float32) for _ in range(3))
    clean = run(hip, DType.F32, [q, k, v], True, "attn_mfma_f32")
    v2, k2 = v.copy(), k.copy()
    v2[:, :, p + 1, 3], v2[:, :, p + 20, 5], k2[:, 1, p + 5:, 0] = np.inf, np.nan, np.nan
    got = run(hip, DType.F32, [q, k2, v2], True, "attn_mfma_f32")
    np.testing.assert_array_equal(got[:, :, :p + 1], clean[:, :, :p + 1])
    want = f64_attention(*(x.astype(np.float64) for x in (q, k2, v2)), True)[:, 0, p + 1:]
    np.testing.assert_array_equal(np.isinf(got[:, 0, p + 1:, 3]), True)
    np.testing.assert_array_equal(np.isnan(got[:, 0, p + 20:, 5]), True)
    assert np.isnan(got[:, 1, p + 5:]).all()
    rest = [i for i in range(d) if i not in (3, 5)]
    assert np.abs(got[:, 0, p + 1:][..., rest] - want[..., rest]).max() <= 1e-5 * np.abs(want[..., rest]).max()


@pytest.mark.parametrize("causal", [False, True])
def test_f32_attention_with_minus_infinity_scores(hip, causal):
    """Keys whose score is -inf weigh nothing, also when they fill a whole block; a query with no
    other key gets NaN (0 / 0), as softmax does."""
    s, d = 140, 32
    rng = np.random.default_rng(0)
    q = np.abs(rng.standard_normal((1, 1, s, d))).astype(np.float32)
    k, v = (rng.standard_normal((1, 1, s, d)).astype(np.float32) for _ in range(2))
    k[:, :, :70, 0] = -np.inf
    got = run(hip, DType.F32, [q, k, v], causal, "attn_mfma_f32")[0, 0]
    lo = 70 if causal else 0
    if causal:
        assert np.isnan(got[:70]).all()
    with np.errstate(invalid="ignore"):  # the all -inf rows
        want = f64_attention(*(x.astype(np.float64) for x in (q, k, v)), causal)[0, 0]
    assert np.abs(got[lo:] - want[lo:]).max() <= 1e-5 * np.abs(want[lo:]).max()


# (heads, positions): one tile a work-group; several, whose pipeline runs on into the next tile
@pytest.mark.parametrize("h,s,grid", [(2, 150, None), (3, 300, "8")])
@pytest.mark.parametrize("dt", [DType.BF16, DType.F16])
@pytest.mark.parametrize("causal", [False, True])
def test_16_bit_heads_of_32_with_infinities_and_nan_in_v(hip, monkeypatch, h, s, grid, dt, causal):
    """Queries that see an infinity or NaN get it in its column, and f64's values in the others; other
    heads keep their bits, and queries before it (causal) stay finite: they are within one rounding of
    a run without it. The queries that met it are done again one to a thread: the bits of the kernel
    for a few positions, which NO_MFMA selects."""
    if grid:
        monkeypatch.setenv("KURUMI_HIP_ATTN_GRID", grid)
    p = s // 3
    rng = np.random.default_rng(s)
    arrays = [rng.standard_normal((3, h, s, 32)).astype(np.float32) for _ in range(3)]
    arrays = [bf16_bits_to_f32(f32_to_bf16_bits(x)) if dt == DType.BF16 else x.astype(np.float16).astype(np.float32) for x in arrays]
    q, k, v = arrays
    clean = run(hip, dt, arrays, causal, "attn_mfma ")
    v = v.copy()
    v[1, 1, p + 1, 3], v[1, 1, p + 2, 4], v[1, 1, p + 20, 5] = np.inf, -np.inf, np.nan
    got = run(hip, dt, [q, k, v], causal, "attn_mfma ")
    monkeypatch.setenv("KURUMI_HIP_NO_MFMA", "1")
    rows = run(hip, dt, [q, k, v], causal, "attn_rowwise")[1, 1]
    other = np.ones((3, h), bool)
    other[1, 1] = False
    np.testing.assert_array_equal(got[other], clean[other])
    got, clean = got[1, 1], clean[1, 1]
    first = p + 20 if causal else 0  # the first query that sees all three
    assert (got[first:, 3] == np.inf).all() and (got[first:, 4] == -np.inf).all() and np.isnan(got[first:, 5]).all()
    np.testing.assert_array_equal(got[first:], rows[first:])
    half_unit = 2.0 ** (-8 if dt == DType.BF16 else -11)
    rest = [i for i in range(32) if i not in (3, 4, 5)]
    scale = np.float32(32 ** -0.5)
    scale = bf16_bits_to_f32(f32_to_bf16_bits(scale)) if dt == DType.BF16 else np.float16(scale)
    want = f64_attention(*(x[1, 1].astype(np.float64) for x in arrays), causal, float(np.asarray(scale).item()))
    assert np.abs(got[:, rest] - want[:, rest]).max() <= (half_unit + 2e-5) * np.abs(want).max()
    if causal:
        # both within half a unit in the last place of the largest (the other bar's bound) of f64
        assert np.abs(got[:p + 1] - clean[:p + 1]).max() <= 2 * (half_unit + 2e-5) * np.abs(want).max()


@pytest.mark.parametrize("scale", [-0.375, 0.0])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dt,d,s", [(DType.BF16, 32, 100), (DType.F16, 32, 70), (DType.BF16, 64, 100), (DType.F16, 128, 70), (DType.F32, 32, 100)])
def test_decomposed_attention_with_a_scale_that_is_not_positive(hip, dt, d, s, causal, scale):
    """The chain softmax(q k^T * c) v takes any constant c. Bars as above, whatever the head size: in 16
    bits such a scale takes the one-query-per-thread kernel, whose scores and probabilities are f32."""
    rng = np.random.default_rng(s)
    arrays = [rng.standard_normal((1, 2, s, d)).astype(np.float32) for _ in range(3)]
    if dt == DType.BF16:
        arrays = [bf16_bits_to_f32(f32_to_bf16_bits(x)) for x in arrays]
        mk = lambda x: Tensor(dt, x.shape, f32_to_bf16_bits(x).tobytes())
    elif dt == DType.F16:
        arrays = [x.astype(np.float16).astype(np.float32) for x in arrays]
        mk = lambda x: Tensor(dt, x.shape, x.astype(np.float16).tobytes())
    else:
        mk = Tensor.from_numpy
    g = K.Graph()
    ids = [g.input(x.shape, dt) for x in arrays]
    raw = g.dot_general(ids[0], ids[1], [3], [3], [0, 1], [0, 1])
    sc = g.mul(raw, g.scalar(raw, scale))
    if causal:
        mask = g.expand(g.reshape(g.constant(np.triu(np.full((s, s), -np.inf, np.float32), 1)), [1, 1, s, s]), [1, 2, s, s])
        sc = g.add(sc, mask if dt == DType.F32 else g.cast(mask, dt))
    o = g.dot_general(g.softmax(sc, 3), ids[2], [3], [2], [0, 1], [0, 1])
    plan = hip.plan(g, [o], {i: mk(x) for i, x in zip(ids, arrays)})
    assert len(plan.steps()) == 1 and plan.steps()[0].startswith("attn"), plan.steps()
    plan.launch()
    got = to_f32(plan.output(0))
    want = f64_attention(*(x.astype(np.float64) for x in arrays), causal, scale)
    half_unit = {DType.BF16: 2.0 ** -8, DType.F16: 2.0 ** -11, DType.F32: 0.0}[dt]
    assert np.abs(got - want).max() <= (half_unit + 2e-5) * np.abs(want).max()


# several tiles a work-group: mirrored rounds and a partial last tile; the head-grouped order over two
# rounds; the same over three; one head of many tiles
@pytest.mark.parametrize("b,h,s,grid", [(2, 4, 300, "8"), (2, 8, 256, "16"), (1, 24, 200, "16"), (1, 3, 1500, "8")])
@pytest.mark.parametrize("dt", [DType.BF16, DType.F16])
@pytest.mark.parametrize("causal", [False, True])
def test_16_bit_heads_of_32_over_several_tiles_match_f64(hip, monkeypatch, b, h, s, grid, dt, causal):
    """Queries of standard deviation 6: scores of up to 30, so that the running maximum moves by more than
    the lazy rescale's 2^8. An f32 score of 30 is off by 2^-19, which the exponential makes 2e-6 of a
    probability; 1e-4 covers the sums, the remainders and the fused scale."""
    monkeypatch.setenv("KURUMI_HIP_ATTN_GRID", grid)
    rng = np.random.default_rng(s)
    arrays = [rng.standard_normal((b, h, s, 32)).astype(np.float32) * np.float32(x) for x in (6.0, 1.0, 1.0)]
    arrays = [bf16_bits_to_f32(f32_to_bf16_bits(x)) if dt == DType.BF16 else x.astype(np.float16).astype(np.float32) for x in arrays]
    got = run(hip, dt, arrays, causal, "attn_mfma ")
    scale = np.float32(32 ** -0.5)
    scale = bf16_bits_to_f32(f32_to_bf16_bits(scale)) if dt == DType.BF16 else np.float16(scale)
    want = f64_attention(*(x.astype(np.float64) for x in arrays), causal, float(np.asarray(scale).item()))
    assert np.abs(got - want).max() <= (2.0 ** (-8 if dt == DType.BF16 else -11) + 1e-4) * np.abs(want).max()
