"""Which code the grids of the face-ghost and lab tests reach: patches on 2:1
grids and packets where a ghost needs a further synthesis, and labs of either
kind, so that a comparison with the oracle is one of the path it is meant for."""
from __future__ import annotations

import numpy as np
import pytest

from test_amr_gpu import make_ctx, random_fields
from test_face_patches_gpu import GRIDS

TAPS = {4: (2, 9), 2: (1, 6)}  # coarse points of a lab per axis: from 4 * index - first on, so many


def jump_faces(rows):
    """Faces whose neighbour is no leaf of the same level."""
    have = {tuple(r) for r in rows.tolist()}
    n = 0
    for L, x, y, z in rows.tolist():
        for a in range(3):
            for d in (-1, 1):
                i = [x, y, z]
                i[a] = (i[a] + d) % (1 << L)
                n += (L, *i) not in have
    return n


def lab_kinds(rows, order):
    """(labs with a jump whose coarse points all are single cells, labs with one
    that lies in a leaf two levels coarser than the block)."""
    top = int(rows[:, 0].max())
    N = 8 << top
    level = np.full((1 << top,) * 3, -1)
    for L, x, y, z in rows.tolist():
        w = 1 << (top - L)
        level[z * w:(z + 1) * w, y * w:(y + 1) * w, x * w:(x + 1) * w] = L
    first, count = TAPS[order]
    single = multi = 0
    for L, x, y, z in rows.tolist():
        near = [level[np.ix_(*[(np.array([i - 1, i, i + 1]) % (1 << L) << (top - L)) + k for i in (z, y, x)])]
                for k in range(1 << (top - L))]
        if L == 0 or all((v == L).all() for v in near):
            continue
        pts = [((4 * i - first + np.arange(count)) << (top - L + 1)) % N >> 3 for i in (z, y, x)]
        if (level[np.ix_(*pts)] < L - 1).any():
            multi += 1
        else:
            single += 1
    return single, multi


@pytest.mark.parametrize("order", [4, 2])
@pytest.mark.parametrize("grid", sorted(GRIDS))
def test_labs_of_both_kinds(grid, order):
    single, multi = lab_kinds(GRIDS[grid](), order)
    assert single > 0
    assert (multi > 0) == grid.startswith("jump"), (single, multi)


@pytest.mark.gpu
@pytest.mark.parametrize("real", ["f32", "f64"])
@pytest.mark.parametrize("order", [4, 2])
@pytest.mark.parametrize("grid", sorted(GRIDS))
def test_gpu_face_path(real, order, grid):
    rows = GRIDS[grid]()
    fields = random_fields(rows, np.float32 if real == "f32" else np.float64, 11)
    print("[gpu] face path", grid, real, order, flush=True)
    ctx = make_ctx(real, rows, order, fields, max_level=6)
    assert set(ctx.face_ghost_info().values()) == {0}
    ctx.rd_prepare(2e-5, 2e-6, 0.08)
    ctx.rd_steps(1, 0.02)
    info = ctx.face_ghost_info()
    ctx.close()
    n = jump_faces(rows)
    jump = grid.startswith("jump")
    assert info == {"patches": 0 if jump else n, "packets": n if jump else 0, "entries": 0}
