"""The likelihood's counted terms against the oracle: states of zeros, of values
lost in u - uc, at, below and above the thresholds, with both labels and with one
label missing where its term is infinite; grids below, at and beyond one pass of
the partition; PET lattices from every point to one."""
import numpy as np
import pytest

import gliomasolver_amd as gh

pytestmark = pytest.mark.gpu
# sums of terms of one sign: their relative error is that of a term (exp, log and
# a difference from 1 that keeps five digits at least) and of 2^21 additions in a tree
REL = 1e-12


def case(n, real, seed, steep):
    rng = np.random.default_rng(seed)
    values = [0.2, 0.25, 0.3, 0.7, 0.71, 1.0] if steep else \
        [0.0, -0.0, 1e-30, 1e-18, 1e-7, 0.1, 0.25, 0.2500001, 0.5, 0.7, 0.70001, 1.0]
    u = np.array(values)[rng.integers(0, len(values), (n, n, n))].astype(np.float32 if real == "f32" else np.float64)
    t1, fl = (rng.random((2, n, n, n)) < 0.4).astype(np.float64)
    if steep:  # every term whose label would make it infinite has the other one
        t1 = (u > 0.7).astype(np.float64)
        fl[u > 0.25] = 1
    else:
        u[: n // 2] *= rng.random((n // 2, n, n)) < 0.05  # a half nearly empty
    pet = np.where(rng.random(u.shape) < 0.5, rng.random(u.shape), 0.0)
    return u, t1, fl, pet


@pytest.mark.parametrize("real", ["f32", "f64"])
@pytest.mark.parametrize("n,step", [(8, 1), (8, 9), (16, 3), (32, 2), (64, 5), (64, 600), (128, 3), (128, 7)])
def test_terms(oracle, real, n, step):
    for slope in (2.0, 1e-3):  # exp(-1 / 1e-3) is 0
        u, t1, fl, pet = case(n, real, 100 * n + step, slope < 1)
        ctx = gh.Context(0, real)
        ctx.grid_init_uniform(n // 8)
        ctx.set_field(gh.FIELD_PHI, u)
        ctx.lik_set_data(t1, fl, pet)
        total, comps, npet = ctx.likelihood((0.0025, 1.0, 0.7, 0.25, slope), stepPET=step)
        want, want_comps, want_npet = oracle.likelihood(u.astype(np.float64), pet, t1, fl, PETsigma2=0.0025,
                                                        PETscale=1.0, slope=slope, stepPET=step)
        assert npet == want_npet
        for a, b in zip((total, *comps), (want, *want_comps)):
            assert np.isfinite(b)
            assert a == pytest.approx(b, rel=REL, abs=1e-9)
        ctx.close()
