"""dphidt and single steps of grids whose blocks are partly without diffusion
(their records are not read), for states that are negative, -0, beyond 1, infinite
or not a number in and next to these blocks: the bits of the oracle, for every
number of blocks per workgroup and for the two-pass form, over one block to 512,
with no such block, some and only such."""
import numpy as np
import pytest

import gliomasolver_amd as gh
from gliomasolver_amd import FIELD_PG, FIELD_PHI, FIELD_PW

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("real", ["f32", "f64"])
@pytest.mark.parametrize("tissue", ["all", "part", "none"])
@pytest.mark.parametrize("n", [8, 16, 64])
def test_single_steps(oracle, real, tissue, n):
    dt_ = np.float32 if real == "f32" else np.float64
    rng = np.random.default_rng(n)
    head = np.zeros((n, n, n), bool) if tissue == "none" else np.ones((n, n, n), bool)
    if tissue == "part":
        head[: n // 2 + 3] = False
        head[:, :, : n // 4] = False
    pw = np.where(head, rng.uniform(0.0, 1.0, head.shape), 0.0).astype(dt_)
    pg = np.where(head, 1.0 - pw, 0.0).astype(dt_)
    odd = np.array([0.0, -0.0, -0.3, 0.4, 1.0, 2.5, np.inf, -np.inf, np.nan, 1e-30, -1e-30])
    phi = np.where(rng.random(head.shape) < 0.2, odd[rng.integers(0, len(odd), head.shape)],
                   rng.uniform(-0.1, 0.9, head.shape)).astype(dt_)
    Dw, rho, h = float(dt_(0.0021)), float(dt_(0.31)), 1.0 / n
    Dg = float(dt_(0.1 * Dw))
    dt = 0.4 / (6 * n * n * Dw)
    want = oracle.rd_steps(phi, pw, pg, Dw, Dg, rho, h, dt, 1)
    ctx = gh.Context(0, real)
    ctx.grid_init_uniform(n // 8)
    for f, a in ((FIELD_PW, pw), (FIELD_PG, pg)):
        ctx.set_field(f, a)
    ctx.rd_prepare(Dw, Dg, rho)
    for way in (0, 1, 2, 4, "two passes"):
        ctx.set_field(FIELD_PHI, phi)
        if way == "two passes":
            ctx.rd_rhs()
            ctx.rd_update(dt)
        else:
            ctx.rd_set_tile(way)
            ctx.rd_steps(1, dt)
        got = ctx.get_field(FIELD_PHI)
        assert np.array_equal(got.view(np.uint8), want.view(np.uint8)), way
    ctx.close()
