"""Fields through the pinned slabs: what goes in comes out, bit for bit, at sizes
below one slab, of one slab, with a ragged last slab and split over threads, and
from several threads with contexts of their own."""
import threading

import numpy as np
import pytest

import gliomasolver_amd as gh

pytestmark = pytest.mark.gpu


def trip(n, real, seed):
    dtype = np.float32 if real == "f32" else np.float64
    rng = np.random.default_rng(seed)
    v = rng.standard_normal((n, n, n)).astype(dtype)
    ctx = gh.Context(real=real)
    ctx.grid_init_uniform(n // 8)
    ctx.set_field(gh.FIELD_PHI, v)
    assert np.array_equal(ctx.get_field(gh.FIELD_PHI), v)
    b = ctx.get_field_blocks(gh.FIELD_PHI)  # slot order x fastest
    m = n // 8
    want = v.reshape(m, 8, m, 8, m, 8).transpose(0, 2, 4, 1, 3, 5).reshape(-1, 8, 8, 8)
    assert np.array_equal(b, want)
    w = rng.standard_normal(b.shape).astype(dtype)
    ctx.set_field_blocks(gh.FIELD_PHI, w)
    assert np.array_equal(ctx.get_field_blocks(gh.FIELD_PHI), w)
    got = ctx.get_field(gh.FIELD_PHI)
    assert np.array_equal(got, w.reshape(m, m, m, 8, 8, 8).transpose(0, 3, 1, 4, 2, 5).reshape(n, n, n))


@pytest.mark.parametrize("real", ["f32", "f64"])
@pytest.mark.parametrize("n", [8, 16, 32, 64, 128])
def test_round_trip(n, real):
    trip(n, real, n)


def test_round_trip_from_threads():
    bad = []

    def work(t):
        try:
            for k in range(3):
                trip([16, 64, 128][(t + k) % 3], ["f32", "f64"][t & 1], 10 * t + k)
        except BaseException as e:  # reported by the test's own thread
            bad.append(e)

    th = [threading.Thread(target=work, args=(t,)) for t in range(4)]
    for t in th:
        t.start()
    for t in th:
        t.join()
    assert not bad, bad
