"""Line kernels over rows whose length is no multiple of a vector: whole vectors at any alignment,
the elements left over by themselves. Against the oracle, exact where the operation is exact in any
order (sums of multiples of 1/16, maxima, indices), else against f64 at the f32 bar of 1e-5."""
import numpy as np
import pytest

import kurumi_amd as K
from kurumi_amd import DType, Tensor
from kutest import bf16_bits_to_f32, f32_to_bf16_bits, interpret, to_f32

pytestmark = pytest.mark.gpu


def tensor(v, dt):
    v = np.ascontiguousarray(v)
    if dt == DType.BF16:
        return Tensor(dt, v.shape, f32_to_bf16_bits(v.astype(np.float32)).tobytes())
    np_t = {DType.F32: np.float32, DType.F16: np.float16, DType.F64: np.float64, DType.U8: np.uint8, DType.I32: np.int32}[dt]
    return Tensor(dt, v.shape, v.astype(np_t).tobytes())


# every remainder of a 4- and an 8-element vector; one to several chunks per thread; a wave, a
# group and two groups' worth of threads per row; too long to stay in registers
@pytest.mark.parametrize("rows,cols", [(5, 257), (3, 258), (4, 259), (2, 263), (7, 1001), (300, 1003), (3, 16387), (2, 50257), (1, 70001)])
@pytest.mark.parametrize("dt", [DType.F32, DType.BF16, DType.F16, DType.U8, DType.F64])
def test_exact_reductions_of_ragged_rows_match_oracle(hip, rows, cols, dt):
    print(f"{dt.name} {rows}x{cols}", flush=True)
    rng = np.random.default_rng(cols)
    v = rng.integers(0, 100, (rows, cols)) if dt in (DType.U8, DType.I32) else rng.integers(-16, 17, (rows, cols)) / 16.0
    v[0, cols - 1] = 120 if dt == DType.U8 else 5.0   # the maximum among the elements left over
    if rows > 1:
        v[1, :] = v[1, 0]                             # equal values: the first index
    g = K.Graph()
    x = g.input([rows, cols], dt)
    feeds = {x: tensor(v, dt)}
    roots = [g.sum(x, 1), g.reduce_max(x, 1), g.argmax(x, 1), g.argmin(x, 1), g.mul(x, x)]
    for got, want, r in zip(hip.eval_many_with(g, roots, feeds), interpret(g, roots, feeds), roots):
        np.testing.assert_array_equal(got.numpy(), want.numpy(), err_msg=str(r))


@pytest.mark.parametrize("rows,cols", [(5, 257), (4, 1003), (2, 50257), (1, 131071)])
@pytest.mark.parametrize("dt", [DType.F32, DType.BF16, DType.F16])
def test_softmax_argmax_of_ragged_rows(hip, rows, cols, dt):
    print(f"softmax {dt.name} {rows}x{cols}", flush=True)
    rng = np.random.default_rng(cols)
    v = (3 * rng.standard_normal((rows, cols))).astype(np.float32)
    v[0, cols - 1] = 20.0
    g = K.Graph()
    x = g.input([rows, cols], dt)
    t = tensor(v, dt)
    y = g.softmax(x, 1)
    gy, ga = hip.eval_many_with(g, [y, g.argmax(y, 1)], {x: t})
    got = to_f32(gy)
    np.testing.assert_array_equal(ga.numpy(), got.argmax(1))
    x64 = to_f32(t).astype(np.float64)
    e = np.exp(x64 - x64.max(1, keepdims=True))
    want = e / e.sum(1, keepdims=True)
    # one rounding to the type (bf16 2^-9 + 2^-9 of the next value, f16 2^-12; its subnormals end at 2^-25)
    rtol, atol = {DType.F32: (1e-5, 0), DType.BF16: (2.0 ** -8, 0), DType.F16: (2.0 ** -11, 2.0 ** -24)}[dt]
    np.testing.assert_allclose(got, want, rtol=rtol + (1e-5 if dt != DType.F32 else 0), atol=atol)


def test_ragged_rows_of_moved_operands_match_oracle(hip):
    """A slice whose rows start at odd elements, a transposed and a padded operand, a row broadcast
    and a per-row value in one region with odd rows, and the NaN-at-index-0 rule of argmax."""
    rng = np.random.default_rng(9)
    g = K.Graph()
    a, b, c = g.input([6, 400], DType.F32), g.input([301, 6], DType.F32), g.input([6, 299], DType.F32)
    d, r = g.input([301], DType.F32), g.input([6], DType.F32)
    feeds = {n: Tensor.from_numpy((rng.integers(-16, 17, g.shape(n)) / 16).astype(np.float32)) for n in (a, b, c, d, r)}
    z = g.add(g.slice(a, [(0, 6), (3, 304)]), g.transpose(b, 0, 1))
    z = g.add(z, g.pad(c, [(0, 0), (1, 1)]))
    z = g.add(g.mul(z, g.broadcast_to(d, [6, 301])), g.broadcast_to(g.reshape(r, [6, 1]), [6, 301]))
    n = g.input([2, 259], DType.BF16)
    nv = np.ones((2, 259), np.float32)
    nv[0, 0] = nv[1, 258] = np.nan
    feeds[n] = tensor(nv, DType.BF16)
    roots = [z, g.sum(z, 1), g.argmin(z, 1), g.argmax(n, 1)]
    for got, want, i in zip(hip.eval_many_with(g, roots, feeds), interpret(g, roots, feeds), range(4)):
        np.testing.assert_array_equal(got.numpy(), want.numpy(), err_msg=str(i))
