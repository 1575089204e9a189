"""Evaluations of few cells on wide grids: up to 1,024 columns every Newton pass of a task is made
by one work-group, beyond them by passes; the same bits by either route at any number of points."""
import numpy as np
import pytest

from radiolensfit2_amd import _native as N
from radiolensfit2_amd import pipeline as P
from radiolensfit2_amd import synth

pytestmark = pytest.mark.gpu

LEN = 900e3


@pytest.mark.parametrize("facet", [15, 16, 17, 127, 1008, 1009, 1023, 1024, 1025])
@pytest.mark.parametrize("nrow", [40, 3900])
def test_one_launch_matches_the_passes(gpu, facet, nrow):
    rng = np.random.default_rng([facet, nrow])
    n = 2 * nrow
    u, v = rng.uniform(-0.2 * LEN, 0.2 * LEN, (2, nrow))
    obs = synth.Observation(None, u, v, np.zeros(nrow), 2 * np.pi / np.array([0.25, 0.24]), np.ones(2),
                            np.ones(n, np.float32), np.zeros(n, bool), LEN,
                            20 * (rng.standard_normal(n) + 1j * rng.standard_normal(n)))
    dev = P.DeviceObservation(obs)
    H = N.hip()
    try:
        cells = dev.extract_only(2e-7, -1e-7, 80., 1.0, facet)
        assert 0 < cells <= min(n, facet * facet)
        dev.set_prior(P.rprior_for(80., P.r_grid()))
        e = rng.uniform(-0.5, 0.5, (33, 2))
        for points in (1, 8, 9, 33):
            got = dev.loglik(*e[:points].T, detail=True)
            N.check(H.rl2_tune_set(N.RL2_TUNE_TILE_PASSES, 3), "rl2_tune_set")
            try:
                passes = dev.loglik(*e[:points].T, detail=True)
            finally:
                N.check(H.rl2_tune_set(N.RL2_TUNE_TILE_PASSES, 0), "rl2_tune_set")
            for a, b in zip(got, passes):
                np.testing.assert_array_equal(a[..., 1:] if a.ndim == 2 else a,
                                              b[..., 1:] if b.ndim == 2 else b)
    finally:
        dev.close()
