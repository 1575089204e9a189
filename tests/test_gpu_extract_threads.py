"""Two host threads that extract into different slots of one observation, or evaluate on one each,
get their own results (an extraction's cells on facets whose cells the compaction writes for the
caller, and on wider ones)."""
import threading

import numpy as np
import pytest

from radiolensfit2_amd import _native as N
from radiolensfit2_amd import pipeline as P
from radiolensfit2_amd import synth

pytestmark = pytest.mark.gpu

LEN = 93000.0
GALAXIES = [(2e-4, -1e-4, 80.0, 1.0), (-3e-4, 5e-4, 50.0, 0.7)]


@pytest.mark.parametrize("facets", [(24, 24), (64, 40), (256, 12), (257, 90)])
def test_threads_extract_into_their_own_slots(gpu, facets):
    rng = np.random.default_rng(facets[0])
    nrow, nch = 4000, 2
    n = nrow * nch
    u, v = rng.uniform(-0.2 * LEN, 0.2 * LEN, (2, nrow))
    obs = synth.Observation(None, u, v, rng.uniform(-50, 50, nrow),
                            2 * np.pi / np.array([0.25, 0.23]), np.ones(nch),
                            rng.uniform(0.5, 2.0, n).astype(np.float32), rng.random(n) < 0.1,
                            3 * LEN, rng.standard_normal(n) + 1j * rng.standard_normal(n))
    dev = P.DeviceObservation(obs)
    try:
        alone = [dev.extract(*g, f, slot=k) for k, (g, f) in enumerate(zip(GALAXIES, facets))]
        wrong = []

        def loop(k):
            for i in range(100):
                got = dev.extract(*GALAXIES[k], facets[k], slot=k)
                if not all(np.array_equal(a, b) for a, b in zip(got, alone[k])):
                    wrong.append((k, i))

        threads = [threading.Thread(target=loop, args=(k,)) for k in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not wrong
    finally:
        dev.close()


def test_threads_evaluate_and_fit_on_their_own_observations(gpu):
    """Each thread's evaluations return on its own observation's results."""
    rng = np.random.default_rng(3)
    devs, points, alone = [], rng.uniform(-0.4, 0.4, (6, 2)), []
    try:
        for k, (g, scale) in enumerate(zip(GALAXIES, (0.6, 3.2))):  # one launch, and passes
            n = 20000
            u, v = rng.uniform(-0.2 * LEN, 0.2 * LEN, (2, n))
            obs = synth.Observation(None, u, v, np.zeros(n), np.array([2 * np.pi / 0.25]),
                                    np.ones(1), np.ones(n, np.float32), np.zeros(n, bool), 3 * LEN,
                                    rng.standard_normal(n) + 1j * rng.standard_normal(n))
            dev = P.DeviceObservation(obs)
            devs.append(dev)
            dev.extract_only(*g[:3], scale, N.hip().facet_size(scale, 3 * LEN))
            dev.set_prior(P.rprior_for(g[2], P.r_grid()))
            res = dev.fit()
            alone.append((dev.loglik(*points.T, detail=True), (res.e1, res.e2, res.error)))
        wrong = []

        def loop(k):
            for i in range(60):
                got = devs[k].loglik(*points.T, detail=True)
                if not all(np.array_equal(a[..., 1:] if a.ndim > 1 else a,
                                          b[..., 1:] if b.ndim > 1 else b, equal_nan=True)
                           for a, b in zip(got, alone[k][0])):
                    wrong.append((k, i))
                if i % 20 == 0:
                    res = devs[k].fit()
                    if (res.e1, res.e2, res.error) != alone[k][1]:
                        wrong.append((k, i, "fit"))

        threads = [threading.Thread(target=loop, args=(k,)) for k in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not wrong
    finally:
        for dev in devs:
            dev.close()
