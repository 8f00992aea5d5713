"""A new wavelet order on a live multi-level grid: the face ghosts, the per-solve
constants made from them and the steps follow it, without another prepare."""
from __future__ import annotations

import numpy as np
import pytest

from gliomasolver_amd import FIELD_PG, FIELD_PHI, FIELD_PW
from amr_util import balanced_random_grid
from test_amr_gpu import bits_equal, make_ctx, random_fields
from test_face_patches_gpu import two_level_jump

pytestmark = pytest.mark.gpu

GRIDS = {
    "patches": lambda: balanced_random_grid(np.random.default_rng(9), base_level=2, max_level=4, nrefine=6),
    "packets": lambda: two_level_jump(3),
}


@pytest.mark.parametrize("prepare_again", [False, True])
@pytest.mark.parametrize("real", ["f32", "f64"])
@pytest.mark.parametrize("orders", [(2, 4), (4, 2), (4, 2, 4)])
@pytest.mark.parametrize("grid", sorted(GRIDS))
def test_gpu_steps_follow_a_new_order(oracle, real, orders, grid, prepare_again):
    rows = GRIDS[grid]()
    t = np.float32 if real == "f32" else np.float64
    fields = random_fields(rows, t, 17)
    Dw, Dg, rho, dt, k = 2e-5, 2e-6, 0.08, 0.02, 2
    print("[gpu] order change", grid, real, orders, len(rows), "blocks", flush=True)
    ctx = make_ctx(real, rows, orders[0], fields, max_level=6)
    ctx.rd_prepare(Dw, Dg, rho)
    ref = fields[FIELD_PHI]
    for i, order in enumerate(orders):
        if i:
            ctx.grid_configure(order, 6, 0)
            if prepare_again:
                ctx.rd_prepare(Dw, Dg, rho)
        ctx.rd_steps(k, dt)
        out = ctx.get_field_blocks(FIELD_PHI).reshape(len(rows), 512)
        ref = oracle.amr_rd_steps(rows, order, ref, fields[FIELD_PW], fields[FIELD_PG], t(Dw), t(Dg), t(rho), dt, k)
        assert bits_equal(out, ref), "order %d: max |diff| %g" % (order, np.abs(out.astype(float) - ref).max())
    ctx.close()
