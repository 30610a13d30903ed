"""Reductions along a column and reductions split over slices of their axis, against the oracle.

Sums run over multiples of 1/16 (exact in f32 in any order: at most 2^21 terms of magnitude below
2, in steps of 2^-4, stay below 2^24 steps only for these sizes) and products over +-1, +-2 and
+-1/2 with balanced exponents, so every order of folding gives the oracle's bits; maxima and
indices are exact by nature.
"""
import numpy as np
import pytest

import kurumi_amd as K
from kurumi_amd import DType, Tensor
from kutest import bf16_bits_to_f32, f32_to_bf16_bits, interpret, to_f32

pytestmark = pytest.mark.gpu

OPS = ["sum", "prod", "reduce_max", "argmax", "argmin"]


def values(rng, shape, dt, op):
    if dt in (DType.I32, DType.U8):
        hi = 3 if op == "prod" else 120
        v = rng.integers(0 if dt == DType.U8 else -hi, hi, shape)
        return Tensor(dt, shape, v.astype(dt.storage).tobytes())
    if op == "prod":
        n = int(np.prod(shape))
        v = np.where(rng.random(shape) < 0.5, -1.0, 1.0)
        twos = rng.permutation(n)[: min(n // 2 * 2, 64)]
        flat = v.reshape(-1)
        flat[twos[::2]] *= 2.0   # powers of two: the product is exact wherever it stays in range
        flat[twos[1::2]] *= 0.5
        v = flat.reshape(shape)
    else:
        v = rng.integers(-16, 17, shape) / 16.0
    v = v.astype(np.float32)
    if dt == DType.F64:
        return Tensor(dt, shape, v.astype(np.float64).tobytes())
    if dt == DType.BF16:
        return Tensor(dt, shape, f32_to_bf16_bits(v).tobytes())
    if dt == DType.F16:
        return Tensor(dt, shape, v.astype(np.float16).tobytes())
    return Tensor(dt, shape, v.tobytes())


def check(hip, g, roots, feeds, what):
    print(what, flush=True)
    got = hip.eval_many_with(g, roots, feeds)
    want = interpret(g, roots, feeds)
    for i, (a, b) in enumerate(zip(got, want)):
        np.testing.assert_array_equal(a.numpy(), b.numpy(), err_msg=f"{what} output {i}")


# (shape, axis): slices with a last partial one, vectors of 4/2/1 columns, fewer lines than a wave,
# lines of one element, one thread per short line, a middle axis, and few long contiguous lines
@pytest.mark.parametrize("shape,axis", [((20000, 12), 0), ((4099, 70), 0), ((3000, 257), 0), ((17, 300), 0), ((5, 3), 0),
                                        ((1, 40), 0), ((9, 1100, 6), 1), ((3, 65, 4, 2), 1), ((2, 150001), 1),
                                        ((1, 300000), 1), ((600, 1, 3), 0), ((8191, 2), 0)])
@pytest.mark.parametrize("dt", [DType.F32, DType.BF16, DType.F64, DType.I32, DType.U8])
def test_column_and_split_reductions_match_oracle(hip, shape, axis, dt):
    rng = np.random.default_rng(sum(shape) + axis)
    for op in OPS:
        g = K.Graph()
        x = g.input(shape, dt)
        check(hip, g, [getattr(g, op)(x, axis)], {x: values(rng, shape, dt, op)}, f"{op} {dt.name} {shape} axis {axis}")


@pytest.mark.parametrize("dt", [DType.F32, DType.F16])
def test_column_reductions_of_moved_and_computed_values(hip, dt):
    """Operands read through every kind of view, a per-line and a per-row broadcast, several
    reductions and a full-size output of one region, and values computed from the sums."""
    rng = np.random.default_rng(3)
    g = K.Graph()
    x = g.input((40, 900), dt)
    b = g.input((40,), dt)
    r = g.input((900,), dt)
    feeds = {n: values(rng, s, dt, "sum") for n, s in ((x, (40, 900)), (b, (40,)), (r, (900,)))}
    t = g.transpose(x, 0, 1)                                     # [900, 40], columns strided
    y = g.add(t, g.broadcast_to(b, [900, 40]))                   # b varies with the line
    z = g.add(y, g.broadcast_to(g.reshape(r, [900, 1]), [900, 40]))  # r along the axis
    s, m, a = g.sum(z, 0), g.reduce_max(z, 0), g.argmin(z, 0)
    p = g.sum(g.pad(x, [(300, 5), (1, 2)]), 0)
    f = g.reduce_max(g.flip(g.slice_step(x, [(0, 40, 1), (3, 900, 2)]), [0, 1]), 0)
    after = g.neg(g.mul(s, g.scalar(s, 0.5)))
    check(hip, g, [z, s, m, a, p, f, after], feeds, f"views {dt.name}")
    for root in (s, m, a, after):  # alone: the same bits as together
        check(hip, g, [root], feeds, f"views {dt.name} root {root}")


@pytest.mark.parametrize("shape,axis", [((5000, 6), 0), ((1, 270001), 1)])
def test_split_argmax_keeps_the_nan_and_infinity_rules(hip, shape, axis):
    n = shape[axis]
    rng = np.random.default_rng(7)
    for first, rest in ((np.nan, 0.0), (-np.inf, -np.inf), (0.0, np.nan), (np.inf, np.inf), (1.0, 1.0)):
        v = np.full(shape, rest, np.float32)
        idx = [slice(None)] * 2
        idx[axis] = 0
        v[tuple(idx)] = first
        if rest == 0.0:
            v += (rng.random(shape) < 1e-3).astype(np.float32)
        idx[axis] = n - 1
        if rest == 1.0:
            v[tuple(idx)] = np.nan
        g = K.Graph()
        x = g.input(shape, DType.F32)
        check(hip, g, [g.argmax(x, axis), g.argmin(x, axis), g.reduce_max(x, axis)], {x: Tensor.from_numpy(v)},
              f"first {first} rest {rest}")


def test_column_softmax_and_rmsnorm_match_f64(hip):
    """Two levels of reduction along a column (not split: values are computed from the sums)."""
    rng = np.random.default_rng(5)
    v = rng.standard_normal((700, 33)).astype(np.float32)
    g = K.Graph()
    x = g.input((700, 33), DType.F32)
    y, r = g.softmax(x, 0), g.rmsnorm(x, 0, 1e-6)
    gy, ga, gr = hip.eval_many_with(g, [y, g.argmax(y, 0), r], {x: Tensor.from_numpy(v)})
    e = np.exp(v.astype(np.float64) - v.max(0))
    # f32 sums of 700 terms: a few 2^-24 each, 1e-5 is the f32 bar everywhere else
    np.testing.assert_allclose(gy.numpy(), e / e.sum(0), rtol=1e-5)
    np.testing.assert_array_equal(ga.numpy(), gy.numpy().argmax(0))
    v64 = v.astype(np.float64)
    np.testing.assert_allclose(gr.numpy(), v64 / np.sqrt((v64 * v64).mean(0) + 1e-6), rtol=1e-5)


@pytest.mark.parametrize("shape,axis", [((0, 300000), 1), ((300000, 0), 0), ((0, 100, 5), 1)])
def test_reductions_of_no_lines_are_empty(hip, shape, axis):
    """Long axes of an empty batch: no line, so no result."""
    g = K.Graph()
    x = g.input(shape, DType.F32)
    y = g.softmax(x, axis)
    check(hip, g, [g.sum(x, axis), g.argmax(x, axis), y], {x: Tensor(DType.F32, shape, b"")}, f"no lines {shape} axis {axis}")


# one to eight adjacent lines a thread: short columns with one thread a line and their values in
# registers (from 65536 such threads), long ones with up to 16 threads and 128 KB of LDS (from 16384); a
# middle axis
@pytest.mark.parametrize("shape,axis,dt", [((40, 32768), 0, DType.F32), ((12, 270000), 0, DType.F32), ((100, 65536), 0, DType.F32),
                                           ((3, 30, 22000), 1, DType.F32), ((9, 600000), 0, DType.BF16), ((9, 131072), 0, DType.BF16), ((130, 131072), 0, DType.BF16),
                                           ((130, 131080), 0, DType.BF16)])
def test_column_softmax_rmsnorm_and_argmax_of_many_lines_match_f64(hip, shape, axis, dt):
    """Several levels of reduction over several lines a thread. f32 at the bar of 1e-5; bf16 within one
    rounding of the output (2^-8 of it, as its significands have 8 bits) and 1e-5."""
    print(f"{dt.name} {shape} axis {axis}", flush=True)
    rng = np.random.default_rng(sum(shape))
    v = 2 * rng.standard_normal(shape, dtype=np.float32)
    if dt == DType.BF16:
        bits = f32_to_bf16_bits(v)
        v, t = bf16_bits_to_f32(bits), Tensor(dt, shape, bits.tobytes())
    else:
        t = Tensor.from_numpy(v)
    g = K.Graph()
    x = g.input(shape, dt)
    y = g.softmax(x, axis)
    roots = [y, g.argmax(y, axis), g.rmsnorm(x, axis, 1e-6)]
    plan = hip.plan(g, roots, {x: t})
    plan.launch()
    gy, ga, gr = (to_f32(plan.output(0)), plan.output(1).numpy(), to_f32(plan.output(2)))
    v = v.astype(np.float64)
    e = np.exp(v - v.max(axis, keepdims=True))
    want = e / e.sum(axis, keepdims=True)
    bar = 1e-5 + (2.0 ** -8 if dt == DType.BF16 else 0.0)
    assert (np.abs(gy - want) <= bar * want).all()
    np.testing.assert_array_equal(ga, gy.argmax(axis))
    want = v / np.sqrt((v * v).mean(axis, keepdims=True) + 1e-6)
    assert (np.abs(gr - want) <= bar * np.abs(want)).all()
