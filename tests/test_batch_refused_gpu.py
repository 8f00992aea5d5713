"""Samples that gh_batch cannot lay out leave the batch without samples: the calls
that would use their buffers refuse, and good samples work afterwards."""
from __future__ import annotations

import numpy as np
import pytest

import gliomasolver_amd as gh
from test_batch_gpu import LIK, anatomy, observations

pytestmark = pytest.mark.gpu
ROW = (0.02, 0.2, 4.0, 0.5, 0.5, 0.5)
ADJ = (0.0004, 0.2, 1.0, 64.0, 64.0, 64.0)
TOO_MANY = 65536  # of 4,096 blocks: 2^31 / 8 in all


@pytest.mark.parametrize("adjoint", [False, True])
@pytest.mark.parametrize("before", [False, True])
def test_refused_samples(adjoint, before):
    b = gh.Batch(0, "f32")
    b.set_observations(b.add_anatomy(16, *anatomy((24, 24, 24), 3)), *observations(128, 3))

    def set_samples(n):
        if adjoint:
            b.set_adjoint_samples([0] * n, [ADJ] * n, [20] * n, 1.0, 0.1)
        else:
            b.set_samples([0] * n, [ROW] * n)

    def use():
        if adjoint:
            return b.adjoint(LIK, ckpt_every=8)[1]
        b.run()
        return b.likelihood(LIK)

    want = None
    if before:
        set_samples(2)
        want = use()
    with pytest.raises(gh.GHError, match="too many blocks"):
        set_samples(TOO_MANY)
    for call in (b.run, lambda: b.likelihood(LIK), lambda: b.adjoint(LIK), lambda: b.get_phi(0), lambda: b.sample_info(0)):
        with pytest.raises((gh.GHError, IndexError)):  # (IndexError: the wrapper knows of no samples)
            call()
    set_samples(2)
    got = use()
    assert np.isfinite(got).all() and (want is None or np.array_equal(want, got))
    b.close()
