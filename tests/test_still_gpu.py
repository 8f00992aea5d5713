"""Groups of blocks without diffusion that a solve leaves at zero are left out
of the two-step and reverse-step launches (tile 0).  The state, the loss and the
gradients equal, bit for bit, those of the single-step schedule, which runs
every block, for initial states that are zero there, negative there (zero after
the first step), and positive in some of these blocks (which then move), at
the shortest calls that mark the groups and below, over checkpoint intervals
with and without a short last segment."""
from __future__ import annotations

import numpy as np
import pytest

import gliomasolver_amd as gh
from gliomasolver_amd import FIELD_PG, FIELD_PHI, FIELD_PW

pytestmark = pytest.mark.gpu
N = 64


def context(real, state):
    dt = np.float32 if real == "f32" else np.float64
    rng = np.random.default_rng(5)
    z, y, x = np.meshgrid(*(np.arange(N),) * 3, indexing="ij")
    head = (x - 30) ** 2 + (y - 33) ** 2 + (z - 29) ** 2 < 17 ** 2
    pw = np.where(head, rng.uniform(0.1, 0.9, head.shape), 0.0).astype(dt)
    pg = np.where(head, 1.0 - pw, 0.0).astype(dt)
    phi = np.where(head, rng.uniform(0.0, 0.6, head.shape), 0.0)
    if state == "negative":
        phi[:8, :16] = -0.25
        phi[56:, 56:, 56:] = -0.0
    elif state == "moving":
        phi[0:8, 0:8, 16:24] = rng.uniform(0.0, 0.3, (8, 8, 8))  # a group of eight with one moving block
        phi[60, 60, 60] = 1e-30
    ctx = gh.Context(0, real)
    ctx.grid_init_uniform(N // 8)
    for f, a in ((FIELD_PW, pw), (FIELD_PG, pg), (FIELD_PHI, phi)):
        ctx.set_field(f, a)
    ctx.rd_prepare(0.0021, 0.00021, 0.31)
    ctx.checkpoint_save(0)
    return ctx, 0.9 / (6 * N * N * 0.0021)


@pytest.mark.parametrize("real", ["f32", "f64"])
@pytest.mark.parametrize("state", ["zero", "negative", "moving"])
def test_gpu_still_groups_are_bit_identical(real, state):
    ctx, dt = context(real, state)
    assert ctx.rd_zero_flux_blocks() > 256
    for steps in (8, 9, 10, 31):
        out = {}
        for tile in (1, 0, 0):
            ctx.rd_set_tile(tile)
            ctx.checkpoint_load(0)
            ctx.rd_steps(steps, dt)
            u = ctx.get_field(FIELD_PHI)
            if tile in out:
                assert np.array_equal(u.view(np.uint8), out[tile].view(np.uint8))
            out[tile] = u
        assert np.array_equal(out[0].view(np.uint8), out[1].view(np.uint8)), (state, steps)
    rng = np.random.default_rng(6)
    t1 = (rng.uniform(size=(N, N, N)) < 0.1).astype(np.float64)
    ctx.lik_set_data(t1, 1 - t1, np.where(t1 > 0, rng.uniform(0, 0.5, t1.shape), 0.0))
    for steps, every in ((1, 4), (2, 1), (11, 4), (12, 6), (21, 64)):
        res = []
        for tile in (2, 0):
            ctx.rd_set_tile(tile)
            ctx.checkpoint_load(0)
            loss, grad = ctx.rd_adjoint(steps, steps * dt, (30.0, 33.0, 29.0), 1.5, every)
            res.append((loss, grad, ctx.get_field(FIELD_PHI)))
        for a, b in zip(*res):
            assert np.array_equal(a, b), (state, steps, every)
    ctx.close()


def test_gpu_still_groups_in_a_batch_match_single_solves():
    """Samples of several lengths on grids with tissue-free blocks, one of them
    ending in every segment position: each equals its own single solve."""
    z, y, x = np.meshgrid(*(np.arange(40),) * 3, indexing="ij")
    head = (x - 20) ** 2 + (y - 20) ** 2 + (z - 20) ** 2 < 11 ** 2
    wm = np.where(head, 0.7, 0.0)
    gm = np.where(head, 0.3, 0.0)
    rng = np.random.default_rng(8)
    t1 = (rng.uniform(size=head.shape) < 0.1).astype(np.float64)
    pet = np.where(t1 > 0, rng.uniform(0, 0.5, t1.shape), 0.0)
    b = gh.Batch(0, "f32")
    a = b.add_anatomy(5, gm, wm, 0 * wm)
    b.set_observations(a, t1, 1 - t1, pet)
    steps = np.array([13, 12, 9, 8, 1, 2])
    rows = np.array([(0.0021, 0.2 + 0.01 * i, n * 0.04, 20.0, 19.0, 21.0) for i, n in enumerate(steps)])
    b.set_adjoint_samples([a] * len(steps), rows, steps)
    loss, grad, _ = b.adjoint(gh.Context.LIK_DEFAULT, ckpt_every=4)
    phi = [b.get_phi(i) for i in range(len(steps))]
    for i in range(len(steps)):
        b.set_adjoint_samples([a], rows[i:i + 1], steps[i:i + 1])
        l1, g1, _ = b.adjoint(gh.Context.LIK_DEFAULT, ckpt_every=64)
        assert np.array_equal(l1[0], loss[i]) and np.array_equal(g1[0], grad[i]) and np.array_equal(b.get_phi(0), phi[i])
    b.close()


@pytest.mark.parametrize("real", ["f32", "f64"])
@pytest.mark.parametrize("cancel", [False, True])
@pytest.mark.parametrize("n", [8, 24, 32])
def test_gpu_clamped_steps_match_oracle_with_cancelling_cells(oracle, real, cancel, n):
    """Pairs and the single odd step on clamped states against the oracle, with
    and without cells of p_w = -p_g != 0 -- out of the domain, but with nonzero
    face coefficients -- and, as a batch sample, on a grid of 3 blocks per side
    (1 / h^2 is no power of two)."""
    t = np.float32 if real == "f32" else np.float64
    rng = np.random.default_rng(n)
    wm = rng.uniform(0.1, 0.9, (n, n, n))
    gm = rng.uniform(0, 1, (n, n, n)) * (1 - wm)
    hole = rng.uniform(size=wm.shape) < 0.3
    wm[hole] = 0
    gm[hole] = 0
    Dw, rho = 0.0021, 0.31
    dt = 0.9 / (6 * n * n * Dw)
    if n == 24:  # through the batch: its anatomies have no negative fractions
        b = gh.Batch(0, real)
        a = b.add_anatomy(3, gm, wm, 0 * wm)
        pw, pg = b.get_anatomy(a)
        for steps in (2, 3, 4, 9):
            b.set_adjoint_samples([a], [(Dw, rho, steps * dt, 11.0, 12.0, 13.0)], [steps], 2.0, 0.7)
            u0 = b.get_phi(0)
            b.run()
            ref = oracle.rd_steps(u0, pw, pg, t(Dw), t(Dw / 10), t(rho), t(1.0 / n), steps * dt / steps, steps)
            assert np.array_equal(b.get_phi(0).view(np.uint8), ref.view(np.uint8)), steps
        b.close()
        return
    pw, pg = wm.astype(t), gm.astype(t)
    if cancel:
        c = rng.uniform(size=pw.shape) < 0.1
        pg[c] = -pw[c]
    phi = rng.uniform(0, 0.4, pw.shape).astype(t)
    phi[rng.uniform(size=pw.shape) < 0.4] = 0
    ctx = gh.Context(0, real)
    ctx.grid_init_uniform(n // 8)
    for f, v in ((FIELD_PW, pw), (FIELD_PG, pg)):
        ctx.set_field(f, v)
    ctx.rd_prepare(Dw, Dw / 10, rho)
    assert ctx.rd_schedule_info() == (0, True)
    for steps in (3, 4, 10):
        ctx.set_field(FIELD_PHI, phi)
        ctx.rd_steps(steps, dt)
        ref = oracle.rd_steps(phi, pw, pg, t(Dw), t(Dw / 10), t(rho), t(1.0 / n), dt, steps)
        assert np.array_equal(ctx.get_field(FIELD_PHI).view(np.uint8), ref.view(np.uint8)), steps
    ctx.close()
