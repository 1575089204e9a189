"""The buffers of an observation's evaluations, made by its first one and made anew when one has
more points than they hold: every evaluation gives what the first gave, point by point."""
import numpy as np
import pytest

from radiolensfit2_amd import _native as N
from radiolensfit2_amd import pipeline as P
from radiolensfit2_amd import synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [0.5, 3.2])  # one launch per evaluation, and passes
def test_evaluations_before_and_after_the_buffers_grow(gpu, scale):
    rng = np.random.default_rng(5)
    nrow, length = 60000, 150000.0
    u, v = rng.uniform(-0.2 * length, 0.2 * length, (2, nrow))
    vis = rng.standard_normal(nrow) + 1j * rng.standard_normal(nrow)
    obs = synth.Observation(None, u, v, np.zeros(nrow), np.array([2 * np.pi / 0.25]), np.ones(1),
                            np.ones(nrow, np.float32), np.zeros(nrow, bool), length, vis)
    dev = P.DeviceObservation(obs)
    try:
        cells = dev.extract_only(0., 0., 80., scale, N.hip().facet_size(scale, length))
        assert (cells <= 8192) == (scale < 1)
        dev.set_prior(P.rprior_for(80., P.r_grid()))
        e = rng.uniform(-0.5, 0.5, (600, 2))
        first = [np.concatenate(x) for x in zip(*(dev.loglik(*e[k:k + 8].T) for k in range(0, 600, 8)))]
        for n in (1, 8, 9, 256, 257, 8, 600, 1, 8):
            for got, want in zip(dev.loglik(*e[:n].T), first):
                np.testing.assert_array_equal(got, want[:n])
    finally:
        dev.close()
