"""The register-staged MFMA GEMM (f32 operands, 16-bit operands of any alignment, e4m3, split K) against
the oracle, bit for bit: operands are multiples of 1/16 in [-1, 1], so every partial sum of up to
2^16 products is a multiple of 1/256 below 2^16 and exact in f32 in any order."""
import numpy as np
import pytest

import kurumi_amd as K
from kurumi_amd import DType, Tensor
from hipmem import device_memory_free
from kutest import f32_to_bf16_bits, interpret, to_f32

pytestmark = pytest.mark.gpu


def tensor(v, dt):
    v = np.ascontiguousarray(v, np.float32)
    if dt == DType.BF16:
        return Tensor(dt, v.shape, f32_to_bf16_bits(v).tobytes())
    return Tensor(dt, v.shape, (v.astype(np.float16) if dt == DType.F16 else v).tobytes())


def sixteenths(rng, shape):
    return rng.integers(-16, 17, shape) / np.float32(16)


# tiles cut by M, N and K, one element, one column, rows of odd length, whole tiles, long K on few
# tiles (split), many tiles, aligned products of few tiles
SIZES = [(1, 1, 1), (2, 3, 5), (33, 1, 70), (1, 130, 129), (31, 65, 127), (64, 64, 64), (130, 129, 33), (7, 128, 2496),
         (257, 300, 95), (1030, 1400, 256), (5, 7, 9001), (200, 120, 1111), (16, 512, 1024), (300, 264, 2048)]


@pytest.mark.parametrize("m,n,k", SIZES)
@pytest.mark.parametrize("nt", [False, True])
@pytest.mark.parametrize("dt", [DType.F32, DType.BF16, DType.F16])
def test_products_of_any_size_match_oracle(hip, dt, nt, m, n, k):
    print(f"{dt.name} nt={nt} {m}x{n}x{k}", flush=True)
    rng = np.random.default_rng(m * 7 + n * 3 + k)
    g = K.Graph()
    a, b = g.input([m, k], dt), g.input([n, k] if nt else [k, n], dt)
    y = g.dot_general(a, b, [1], [1 if nt else 0])
    feeds = {a: tensor(sixteenths(rng, (m, k)), dt), b: tensor(sixteenths(rng, (n, k) if nt else (k, n)), dt)}
    label = hip.plan(g, [y], feeds).steps()[-1].split()[0]
    direct = dt != DType.F32 and (m, n, k) == (64, 64, 64)  # one stage of K: the direct-to-LDS kernel's
    flex = not direct and k > 16  # K of up to 16: the generic kernel's
    assert ("_flex" in label) == flex and ("_split" in label) == (k in (2496, 9001, 1111, 1024, 2048)), label
    roots = [y, g.cast(y, DType.F16 if dt != DType.F16 else DType.F32)]
    for r in roots:  # each alone: the cast rides in the product's epilogue
        np.testing.assert_array_equal(hip.eval_with(g, r, feeds).numpy(), interpret(g, [r], feeds)[0].numpy())


@pytest.mark.parametrize("dt,m,n,k", [(DType.F32, 3041, 3719, 517), (DType.BF16, 907, 3331, 70), (DType.F16, 907, 3331, 70)])
@pytest.mark.parametrize("nt", [False, True])
def test_the_largest_tiles_match_numpy(hip, dt, m, n, k, nt):
    """128 x 128 tiles, cut by M, N and K (the oracle would take a minute: numpy's f32 product, whose
    sums are exact too)."""
    rng = np.random.default_rng(m)
    g = K.Graph()
    a, b = g.input([m, k], dt), g.input([n, k] if nt else [k, n], dt)
    x, w = sixteenths(rng, (m, k)), sixteenths(rng, (n, k) if nt else (k, n))
    plan = hip.plan(g, [g.dot_general(a, b, [1], [1 if nt else 0])], {a: tensor(x, dt), b: tensor(w, dt)})
    assert "_128x128_flex" in plan.steps()[0], plan.steps()
    plan.launch()
    np.testing.assert_array_equal(to_f32(plan.output(0)), to_f32(tensor(x @ (w.T if nt else w), dt)))


@pytest.mark.parametrize("dt", [DType.F32, DType.BF16])
def test_strided_batched_and_offset_operands_match_oracle(hip, dt):
    """Views the planner hands to the kernel as they are: a sliced operand (its rows start at any
    element), a batch broadcast to a stride of zero, a batch of transposed right operands, and
    reversed rows (a negative row stride)."""
    rng = np.random.default_rng(11)
    g = K.Graph()
    a, b = g.input([3, 50, 83], dt), g.input([3, 83, 45], dt)
    w, bt = g.input([83, 45], dt), g.input([3, 45, 83], dt)
    feeds = {n: tensor(sixteenths(rng, g.shape(n)), dt) for n in (a, b, w, bt)}
    sa = g.slice(a, [(0, 3), (1, 50), (3, 80)])
    sb = g.slice(b, [(0, 3), (3, 80), (2, 44)])
    roots = [g.dot_general(sa, sb, [2], [1], [0], [0]),
             g.dot_general(a, g.broadcast_to(w, [3, 83, 45]), [2], [1], [0], [0]),
             g.dot_general(a, bt, [2], [2], [0], [0]),
             g.dot_general(g.flip(a, [1]), b, [2], [1], [0], [0]),
             g.dot_general(g.slice(a, [(1, 2), (0, 50), (0, 83)]), g.slice(bt, [(2, 3), (0, 45), (0, 83)]), [2], [2], [0], [0])]
    for i, r in enumerate(roots):
        print(f"{dt.name} view {i}", flush=True)
        np.testing.assert_array_equal(hip.eval_with(g, r, feeds).numpy(), interpret(g, [r], feeds)[0].numpy(), err_msg=str(i))


@pytest.mark.parametrize("m,n,k", [(3, 5, 7), (2, 3, 3001)])
def test_f32_products_keep_infinities_nans_and_denormals(hip, m, n, k):
    """Zeros stand in for what lies past K: an infinity or NaN elsewhere must not meet them, and
    f32 denormals are neither flushed on the way in nor out."""
    a, b = np.zeros((m, k), np.float32), np.ones((k, n), np.float32)
    a[0, k - 1] = np.inf
    a[1, 0] = np.float32(1e-41)
    b[:, n - 1] = 2.0
    b[k // 2, 1] = np.nan
    g = K.Graph()
    x, w = g.input([m, k], DType.F32), g.input([k, n], DType.F32)
    got = to_f32(hip.eval_with(g, g.matmul(x, w), {x: tensor(a, DType.F32), w: tensor(b, DType.F32)}))
    want = np.zeros((m, n), np.float32)
    want[0], want[1], want[1, n - 1] = np.inf, np.float32(1e-41), np.float32(1e-41) * 2
    want[:, 1] = np.nan
    np.testing.assert_array_equal(got, want)


# few tiles, cut by M and N, split and unsplit, the last of the rows that take it; one and two stages,
# which the direct-to-LDS kernel keeps
@pytest.mark.parametrize("m,n,k", [(1, 64, 128), (33, 70, 256), (16, 512, 4096), (130, 100, 640), (300, 520, 384), (1024, 65, 384), (1024, 65, 128), (7, 3000, 2048)])
def test_e4m3_products_of_few_tiles_match_oracle(hip, m, n, k):
    """The e4m3 linear's product (operands multiples of 1/16, exact in e4m3, unit scales) in f32."""
    print(f"e4m3 {m}x{n}x{k}", flush=True)
    rng = np.random.default_rng(m + n + k)
    codes = np.array([0x00, 0x18, 0x20, 0x28, 0x30, 0x38, 0x98, 0xa0, 0xa8, 0xb0, 0xb8], np.uint8)  # 0, +-2^-4 .. +-1
    g = K.Graph()
    a, b = g.input([m, k], DType.F8E4M3), g.input([n, k], DType.F8E4M3)
    sx, sw = g.input([1], DType.F32), g.input([n], DType.F32)
    d = g.dot_general(g.cast(a, DType.F32), g.cast(b, DType.F32), [1], [1])
    d = g.mul(d, g.expand(g.reshape(sx, [1, 1]), [m, n]))
    y = g.cast(g.mul(d, g.expand(g.reshape(sw, [1, n]), [m, n])), DType.BF16)
    feeds = {a: Tensor(DType.F8E4M3, (m, k), rng.choice(codes, (m, k)).tobytes()), b: Tensor(DType.F8E4M3, (n, k), rng.choice(codes, (n, k)).tobytes()),
             sx: tensor([0.5], DType.F32), sw: tensor(2.0 ** rng.integers(-2, 3, n), DType.F32)}
    plan = hip.plan(g, [y], feeds)
    label = plan.steps()[-1].split()[0]
    assert label.startswith("gemm_mfma_e4m3") and ("_flex" in label) == (k > 256) and ("_split" in label) == (k >= 2048), label
    plan.launch()
    np.testing.assert_array_equal(plan.output(0).numpy(), interpret(g, [y], feeds)[0].numpy())


def test_steps_of_a_plan_share_their_scratch():
    """Split products, dequantising products and split reductions leave partial sums in one buffer of
    the largest size, not in one each: the device memory that a plan of 33 such steps takes, and its results."""
    count, m, n, k = 16, 32, 4096, 8192
    rng = np.random.default_rng(11)
    a = (rng.integers(-4, 5, (count * m, k)) / 8).astype(np.float32)
    b = (rng.integers(-4, 5, (k, n)) / 8).astype(np.float32)
    q = rng.integers(0, 256, (n, k // 2)).astype(np.uint8)
    scale = np.full((n, k // 64), 0.25, np.float16)
    hip = K.HipBackend()
    g = K.Graph()
    x, w = g.input(a.shape, DType.F32), g.input(b.shape, DType.F32)
    qw = g.constant_bytes(DType.U8, q.tobytes(), list(q.shape))
    sc = g.constant_bytes(DType.F16, scale.tobytes(), list(scale.shape))
    parts = [g.slice(x, [(m * i, m * i + m), (0, k)]) for i in range(count)]
    roots = [g.matmul(p, w) for p in parts] + [g.quant_matmul(p, qw, sc, None, 4, 64) for p in parts] + [g.sum(x, 0)]
    feeds = {x: Tensor.from_numpy(a), w: Tensor.from_numpy(b)}
    free = device_memory_free()
    plan = hip.plan(g, roots, feeds)
    taken = free - device_memory_free()
    labels = plan.steps()
    assert sum("_split" in s for s in labels) == count, labels
    plan.launch()
    got = [plan.output(i).numpy() for i in range(2 * count + 1)]
    for _ in range(3):  # recorded, then replayed
        plan.launch(use_graph=True)
        for i, want in enumerate(got):
            np.testing.assert_array_equal(plan.output(i).numpy(), want)
    np.testing.assert_array_equal(np.concatenate(got[:count]), a @ b)  # sums of few 64ths: exact in any order
    wq = np.stack([(q & 15).astype(np.int8), (q >> 4).astype(np.int8)], -1).reshape(n, k)
    wq = np.where(wq > 7, wq - 16, wq).astype(np.float32) * 0.25
    np.testing.assert_array_equal(np.concatenate(got[count:-1]), a @ wq.T)
    np.testing.assert_array_equal(got[-1], a.sum(0))
    partial = m * n * 4 * int(labels[0].split("_split")[1].split()[0])  # of one product
    outs, ins = (2 * count * m * n + k) * 4, a.nbytes + b.nbytes + q.nbytes + scale.nbytes
    print(f"taken {taken} inputs {ins} outputs {outs} partial sums {partial}", flush=True)
    assert taken <= ins + outs + 8 * partial
