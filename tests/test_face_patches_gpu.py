"""Face ghosts of the multi-level RD step where one synthesis level is not
enough for some of them: the grid takes term packets instead of patches --
summed in the step kernel on small grids, by their own kernel before it on
large ones -- and stays bit-exact to the oracle; balanced grids next to them
take the patches, with 512 or 256 lanes a block."""
from __future__ import annotations

import numpy as np
import pytest

from gliomasolver_amd import FIELD_PG, FIELD_PHI, FIELD_PW
from amr_util import apply_refine, balanced_random_grid, canonical
from test_amr_gpu import bits_equal, make_ctx, random_fields

pytestmark = pytest.mark.gpu


def two_level_jump(base):
    n = 1 << base
    rows = canonical([[base, x, y, z] for z in range(n) for y in range(n) for x in range(n)])
    for corner in ((base, 3, 2, 1), (base + 1, 6, 4, 2)):
        rows = apply_refine(rows, [k for k in range(len(rows)) if tuple(rows[k]) == corner])
    return rows


GRIDS = {
    "jump-526": lambda: two_level_jump(3),
    "jump-4110": lambda: two_level_jump(4),
    "balanced-small": lambda: balanced_random_grid(np.random.default_rng(9), base_level=2, max_level=4, nrefine=6),
    "balanced-large": lambda: balanced_random_grid(np.random.default_rng(9), base_level=4, max_level=5, nrefine=4),
}


@pytest.mark.parametrize("real", ["f32", "f64"])
@pytest.mark.parametrize("order", [4, 2])
@pytest.mark.parametrize("grid", sorted(GRIDS))
def test_gpu_face_ghosts_match_oracle(oracle, real, order, grid):
    rows = GRIDS[grid]()
    t = np.float32 if real == "f32" else np.float64
    fields = random_fields(rows, t, 11)
    print("[gpu] face ghosts", grid, real, order, len(rows), "blocks", flush=True)
    ctx = make_ctx(real, rows, order, fields, max_level=6)
    Dw, Dg, rho, dt, k = 2e-5, 2e-6, 0.08, 0.02, 2
    ctx.rd_prepare(Dw, Dg, rho)
    ctx.rd_steps(k, dt)
    out = ctx.get_field_blocks(FIELD_PHI).reshape(len(rows), 512)
    counts = ctx.adapt_counters()
    ctx.close()
    ref = oracle.amr_rd_steps(rows, order, fields[FIELD_PHI], fields[FIELD_PW], fields[FIELD_PG], t(Dw), t(Dg),
                              t(rho), dt, k)
    assert bits_equal(out, ref), "max |diff| %g" % np.abs(out.astype(float) - ref).max()
    assert counts["faces_device"] >= 1 and counts["faces_host"] == 0, counts


@pytest.mark.parametrize("real", ["f32", "f64"])
@pytest.mark.parametrize("order", [4, 2])
@pytest.mark.parametrize("grid", ["jump-526", "balanced-small"])
def test_gpu_lab_details_match_oracle(oracle, real, order, grid):
    """Details whose labs hold coarse points that need a further synthesis
    (two-level jump) and labs of single cells only: equal to the oracle's."""
    rows = GRIDS[grid]()
    fields = random_fields(rows, np.float32 if real == "f32" else np.float64, 13)
    ctx = make_ctx(real, rows, order, fields, max_level=6)
    det = ctx.fwt_details()
    counts = ctx.adapt_counters()
    ctx.close()
    ref = oracle.amr_details(rows, order, fields[FIELD_PHI], list(range(len(rows))))
    assert np.array_equal(det, ref), "max |diff| %g" % np.abs(det - ref).max()
    assert counts["labs_device"] >= 1 and counts["labs_host"] == 0, counts
