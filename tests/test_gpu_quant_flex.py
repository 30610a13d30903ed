"""QuantMatmul through the GEMM that dequantises as it stages the weight, and the 16-value expansion
before a plain GEMM, against the oracle bit for bit: act values are multiples of 1/16 in [-1, 1],
scales powers of two and mins whole multiples of them that keep every weight exact in bf16, so every
partial sum is a multiple of 2^-10 below 2^14 and exact in f32 in any order."""
import numpy as np
import pytest

import kurumi_amd as K
from kurumi_amd import DType, Tensor
from kutest import f32_to_bf16_bits, interpret

pytestmark = pytest.mark.gpu


def quant_case(rng, m, n, k, bits, group, sym, dt):
    g = K.Graph()
    x = g.input([m, k], dt)
    v = (rng.integers(-16, 17, (m, k)) / 16).astype(np.float32)
    raw = f32_to_bf16_bits(v) if dt == DType.BF16 else v.astype(np.float16) if dt == DType.F16 else v
    feeds = {x: Tensor(dt, (m, k), raw.tobytes())}
    qw = g.constant_bytes(DType.U8, rng.integers(0, 256, (n, k * bits // 8), dtype=np.uint8).tobytes(), [n, k * bits // 8])
    scales = (2.0 ** rng.integers(-6, -3, (n, k // group))).astype(np.float16)
    sc = g.constant_bytes(DType.F16, scales.tobytes(), scales.shape)
    mn = None
    if not sym:
        mn = g.constant_bytes(DType.F16, (scales * -np.float16(2 ** (bits - 1))).tobytes(), scales.shape)
    return g, g.quant_matmul(x, qw, sc, mn, bits, group), feeds


# one and several tiles of each height, cut by M and N; K of one and many stages, ending inside one;
# groups of one unit, of no power of two, longer than a stage; split K
@pytest.mark.parametrize("m,n,k,group", [(9, 64, 256, 16), (33, 70, 336, 48), (65, 130, 160, 32), (70, 33, 1024, 64), (130, 129, 384, 128),
                                         (300, 100, 128, 128), (10, 40, 4096, 256), (1000, 320, 96, 32)])
@pytest.mark.parametrize("bits", [2, 4, 8])
@pytest.mark.parametrize("sym", [True, False])
@pytest.mark.parametrize("dt", [DType.BF16, DType.F16, DType.F32])
def test_dequantising_gemm_matches_oracle(hip, m, n, k, group, bits, sym, dt):
    print(f"{dt.name} int{bits} sym={sym} {m}x{n}x{k} g{group}", flush=True)
    g, y, feeds = quant_case(np.random.default_rng(m + n + k), m, n, k, bits, group, sym, dt)
    mfma = bits == 4 and 9 <= m <= 64 and group % 64 == 0 and dt != DType.F32  # the kernel for few rows of int4
    assert hip.plan(g, [y], feeds).steps()[0].startswith("quant_mfma " if mfma else "quant_dequant+gemm_fused ")
    np.testing.assert_array_equal(hip.eval_with(g, y, feeds).numpy(), interpret(g, [y], feeds)[0].numpy())


@pytest.mark.parametrize("m,n,k,bits,dt", [(163, 11065, 1024, 4, DType.BF16), (163, 3001, 2048, 8, DType.F16), (66, 11065, 4096, 4, DType.F32)])
def test_dequantising_gemm_of_the_largest_tiles_matches_numpy(hip, m, n, k, bits, dt):
    """128 x 128 tiles cut by M and N, unsplit and split (the oracle would take minutes: numpy's f32
    product, whose sums are exact too)."""
    rng = np.random.default_rng(m)
    g, y, feeds = quant_case(rng, m, n, k, bits, 64, True, dt)
    plan = hip.plan(g, [y], feeds)
    assert plan.steps()[0].startswith("quant_dequant+gemm_fused "), plan.steps()
    plan.launch()
    rng = np.random.default_rng(m)  # the same draws again
    v = (rng.integers(-16, 17, (m, k)) / 16).astype(np.float32)
    packed = rng.integers(0, 256, (n, k * bits // 8), dtype=np.uint8)
    scales = (2.0 ** rng.integers(-6, -3, (n, k // 64))).astype(np.float32)
    q = packed.astype(np.int8) if bits == 8 else np.stack([packed << 4, packed], -1).astype(np.int8).reshape(n, k) >> 4
    want = v @ (q.astype(np.float32) * np.repeat(scales, 64, 1)).T
    raw = f32_to_bf16_bits(want) if dt == DType.BF16 else want.astype(np.float16) if dt == DType.F16 else want
    np.testing.assert_array_equal(plan.output(0).numpy(), Tensor(dt, (m, n), raw.tobytes()).numpy())


@pytest.mark.parametrize("m,n,k,group,bits,dt,want", [
    (100, 256, 512, 64, 2, DType.BF16, "quant_dequant+gemm_fused "),   # dequantised in the GEMM
    (4096, 2048, 512, 64, 4, DType.BF16, "quant_dequant+gemm "),       # so many rows that expanding pays
    (20, 64, 240, 24, 8, DType.F16, "quant_dequant+gemm "),            # groups of no whole 16 values
])
def test_quant_path_by_rows_and_group(hip, m, n, k, group, bits, dt, want):
    g, y, feeds = quant_case(np.random.default_rng(1), m, n, k, bits, group, True, dt)
    plan = hip.plan(g, [y], feeds)
    assert plan.steps()[0].startswith(want), plan.steps()
    plan.launch()
    rows = [0, m // 2, m - 1]
    if m > 1000:  # the oracle on a few rows
        sub = K.Graph()
        g2, y2, f2 = quant_case(np.random.default_rng(1), m, n, k, bits, group, True, dt)
        x = next(iter(f2))
        v = f2[x].numpy()[rows]
        rng = np.random.default_rng(1)
        rng.integers(-16, 17, (m, k))
        s = sub.input([3, k], dt)
        qw = sub.constant_bytes(DType.U8, rng.integers(0, 256, (n, k * bits // 8), dtype=np.uint8).tobytes(), [n, k * bits // 8])
        scales = (2.0 ** rng.integers(-6, -3, (n, k // group))).astype(np.float16)
        out = sub.quant_matmul(s, qw, sub.constant_bytes(DType.F16, scales.tobytes(), scales.shape), None, bits, group)
        wanted = interpret(sub, [out], {s: Tensor(dt, (3, k), v.tobytes())})[0].numpy()
        np.testing.assert_array_equal(plan.output(0).numpy()[rows], wanted)
    else:
        np.testing.assert_array_equal(plan.output(0).numpy(), interpret(g, [y], feeds)[0].numpy())
