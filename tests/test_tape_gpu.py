"""Gradients whose trajectory fits the tape and gradients that recompute it in
segments, because most of the device's memory is taken, are the same bits, and so
are the final states: one solve with still groups, and a batch whose samples end
in different segments."""
import numpy as np
import pytest
import torch

import gliomasolver_amd as gh
from gliomasolver_amd import FIELD_PHI
from test_batch_gpu import LIK, anatomy, observations
from test_still_gpu import N, context

pytestmark = pytest.mark.gpu
LEFT = 8 << 30  # bytes: a tape of 1 GiB


def single(real, state, nsteps):
    ctx, dt = context(real, state)
    rng = np.random.default_rng(1)
    t1, fl = (rng.random((2, N, N, N)) < 0.3).astype(np.float64)
    ctx.lik_set_data(t1, fl, np.where(t1 > 0, 0.5, 0.0))
    loss, grad = ctx.rd_adjoint(nsteps, nsteps * dt, (30.0, 33.0, 29.0), ckpt_every=16)
    phi = ctx.get_field(FIELD_PHI)
    ctx.close()
    return [loss, grad, phi]


def batch(real, steps):
    b = gh.Batch(0, real)
    for bpd, shape, seed in ((8, (70, 60, 64), 3), (4, (32, 35, 30), 4)):
        b.set_observations(b.add_anatomy(bpd, *anatomy(shape, seed)), *observations(8 * bpd, seed))
    smp = [(i % 2, 0.0004, 0.2, 0.01 * n, 14.3 * (2 - i % 2), 16.0, 13.7, n) for i, n in enumerate(steps)]
    b.set_adjoint_samples([s[0] for s in smp], [s[1:7] for s in smp], [s[7] for s in smp], 1.0, 0.1)
    loss, grad, _ = b.adjoint(LIK, ckpt_every=16, stepPET=2)
    out = [loss, grad] + [b.get_phi(i) for i in range(len(smp))]
    b.close()
    return out


def same(run):
    whole = run()
    free = torch.cuda.mem_get_info()[0]
    ballast = torch.empty(free - LEFT, dtype=torch.uint8, device="cuda")
    try:
        cut = run()
    finally:
        del ballast
        torch.cuda.empty_cache()
    for a, b in zip(whole, cut):
        assert np.array_equal(a.view(np.uint8), b.view(np.uint8))


@pytest.mark.parametrize("real,state,nsteps", [("f32", "negative", 2600), ("f32", "moving", 2047), ("f64", "moving", 1500)])
def test_one_solve(real, state, nsteps):
    same(lambda: single(real, state, nsteps))


@pytest.mark.parametrize("real", ["f32", "f64"])
def test_batch(real):
    same(lambda: batch(real, (1800, 1300, 1801, 40, 1, 900)))
