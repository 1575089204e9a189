"""Two host threads that extract into different slots of one observation each get their own
facet's cells, on facets whose cells the compaction writes for the caller and on wider ones."""
import threading

import numpy as np
import pytest

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
