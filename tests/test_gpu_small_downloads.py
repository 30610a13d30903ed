"""Outputs on both sides of the size that goes through pinned memory: alone, from several threads with a
backend each, and from several that share one backend and so its pinned buffer. Whole bytes, so
equality is exact."""
import threading

import numpy as np
import pytest

import kurumi_amd as K
from kurumi_amd import DType, Tensor

pytestmark = pytest.mark.gpu


def make(hip, n):
    g = K.Graph()
    x = g.input([n], DType.U8)
    return g, x, hip.compile(g, g.add(x, x))


def check(plan, g, x, n, seed):
    v = np.random.default_rng(seed).integers(0, 128, n).astype(np.uint8)
    got = plan.run(g, {x: Tensor(DType.U8, (n,), v.tobytes())}).numpy()
    np.testing.assert_array_equal(got, v * 2, err_msg=f"{n} bytes, seed {seed}")


@pytest.mark.parametrize("n", [1, 3, 1280, 16384, 65535, 65536, 65537, 100352])
def test_output_bytes_arrive_whole(hip, n):
    print(f"{n} bytes", flush=True)
    g, x, plan = make(hip, n)
    for seed in range(4):
        check(plan, g, x, n, seed)


@pytest.mark.parametrize("shared", [False, True])
def test_threads_each_get_their_own_bytes(shared):
    sizes = (1000, 4096, 65536, 65537)
    wrong = []
    plans = [None] * len(sizes)
    if shared:  # planned and run once (which records each plan's graph) before the threads start
        be = K.HipBackend()
        for i, n in enumerate(sizes):
            plans[i] = make(be, n)
            check(plans[i][2], *plans[i][:2], n, i)

    def work(i):
        try:
            g, x, plan = plans[i] or make(K.HipBackend(), sizes[i])
            for seed in range(20):
                check(plan, g, x, sizes[i], 100 * i + seed)
        except Exception as e:
            wrong.append(e)

    ts = [threading.Thread(target=work, args=(i,)) for i in range(len(sizes))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not wrong, wrong[0]
