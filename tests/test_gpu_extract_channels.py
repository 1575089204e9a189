"""The extraction of observations with few rows and many channels, whose work-groups share out the
channels: the same bits as the run-merging variants, plain and with the fused subtraction, and
no slower than they are."""
import time

import numpy as np
import pytest

from oracle import oracle as O
from radiolensfit2_amd import _native as N
from radiolensfit2_amd import pipeline as P
from radiolensfit2_amd import synth

pytestmark = pytest.mark.gpu

LEN = 93000.0
FIELDS = ("e1", "e2", "var_e1", "var_e2", "oneDimvar", "maxL", "error", "ncoords")


def _observation(nrow, nch):
    rng = np.random.default_rng([nrow, nch])
    wn = 2 * np.pi / np.linspace(0.25, 0.2, nch)
    r = np.exp(rng.uniform(np.log(100.0), np.log(0.18 * LEN), nrow))  # baselines of all lengths
    a = rng.uniform(0, 2 * np.pi, nrow)
    n = nrow * nch
    vis = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    return synth.Observation(None, r * np.cos(a), r * np.sin(a), rng.uniform(-50, 50, nrow), wn,
                             np.linspace(1.0, 0.8, nch), rng.uniform(0.5, 2.0, n).astype(np.float32),
                             rng.random(n) < 0.05, LEN, vis)


class _Variant:
    def __init__(self, v):
        self.v = v

    def __enter__(self):
        N.check(N.hip().rl2_tune_set(N.RL2_TUNE_GRID_VARIANT, self.v), "rl2_tune_set")

    def __exit__(self, *_):
        N.check(N.hip().rl2_tune_set(N.RL2_TUNE_GRID_VARIANT, 5), "rl2_tune_set")


@pytest.mark.parametrize("precision", [N.RL2_PREC_FP64, N.RL2_PREC_MIXED])
@pytest.mark.parametrize("nch", [1, 3, 4, 5, 8, 9, 33, 64])
@pytest.mark.parametrize("nrow", [1, 2, 511, 512, 513, 2761])
def test_every_channel_is_gridded_once(gpu, nrow, nch, precision):
    obs = _observation(nrow, nch)
    facet = N.hip().facet_size(1.0, LEN)
    cat = synth.Catalog(np.array([80., 60., 40.]), np.array([1.0, .7, .5]), np.zeros(3), np.zeros(3),
                        np.array([2e-4, -1e-4, 3e-4]), np.array([-1e-4, 2e-4, 1e-4]), np.zeros(3))
    dev = P.DeviceObservation(obs, precision=precision)
    try:
        dev.checkpoint()

        def both():  # an extraction, then a loop whose second and third have the subtraction
            dev.restore()
            facets = dev.extract(2e-4, -1e-4, 80., 1.0, facet)
            res, _ = dev.process(cat, do_refit=0)
            got = P.results_array(res)
            return [*facets, *(got[k] for k in FIELDS), dev.residual()]
        got = both()
        with _Variant(3):
            want = both()
    finally:
        dev.close()
    for a, b in zip(got, want):
        np.testing.assert_array_equal(a, b)


def _tracks(dishes, times, nch):
    """Dishes at log-spaced distances up to 150 km over eight hours."""
    rng = np.random.default_rng([dishes, 31])
    r = np.exp(rng.uniform(np.log(300.0), np.log(150e3), dishes))
    th = rng.uniform(0, 2 * np.pi, dishes)
    i, j = np.triu_indices(dishes, 1)
    bx, by = (r * np.cos(th))[j] - (r * np.cos(th))[i], (r * np.sin(th))[j] - (r * np.sin(th))[i]
    h = np.radians(np.linspace(-60, 60, times))[:, None]
    u = (np.cos(h) * bx - np.sin(h) * by).reshape(-1)
    v = 0.7 * (np.sin(h) * bx + np.cos(h) * by).reshape(-1)
    wn = 2 * np.pi * (950e6 + 240e6 / nch * (np.arange(nch) + 0.5)) / 299792458.0
    length = np.ceil(np.abs([u, v]).max()) * wn[-1] / (2 * np.pi)
    n = len(u) * nch
    vis = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    return synth.Observation(None, u, v, 0.1 * u, wn, np.ones(nch), np.ones(n, np.float32),
                             np.zeros(n, bool), length, vis)


@pytest.mark.parametrize("dishes,times,nch,scale", [(24, 10, 64, 0.35), (24, 10, 64, 1.0),
                                                    (24, 4, 256, 1.0), (64, 10, 256, 0.35)])
def test_many_channels_are_not_slower_than_merging_runs(gpu, dishes, times, nch, scale):
    """The shortest of twenty calls of each, in turn.  With one work-group for all channels of
    512 rows these took 1.1 to 1.4 times as long as by merging runs; shared out, a tenth to a
    quarter."""
    obs = _tracks(dishes, times, nch)
    dev = P.DeviceObservation(obs)
    try:
        facet = N.hip().facet_size(scale, obs.len)
        best = {1: np.inf, 5: np.inf}  # 1: runs of 2 rows, 1024 slots
        for _ in range(20):
            for v in best:
                with _Variant(v):
                    t = time.perf_counter()
                    dev.extract_only(1e-3, -5e-4, 80., scale, facet)
                    best[v] = min(best[v], time.perf_counter() - t)
    finally:
        dev.close()
    assert best[5] <= best[1], best


@pytest.mark.parametrize("precision", [N.RL2_PREC_FP64, N.RL2_PREC_MIXED])
@pytest.mark.parametrize("what", ["visibility", "sigma2", "flux"])
def test_without_a_finite_bound_every_visibility_is_counted(gpu, what, precision):
    """An infinite value leaves the integer sums without a scale: the run-merging kernel takes the
    call, whichever variant is chosen.  Cells and weights are those of the data all the same."""
    obs = _observation(1025, 5)
    gal = (2e-4, -1e-4, 80.0, 1.0)
    facet = N.hip().facet_size(1.0, LEN)
    obs.flag[777] = False
    dev = P.DeviceObservation(obs, precision=precision)
    want = dev.extract(*gal, facet)
    dev.close()
    if what == "visibility":
        obs.vis[777] = complex(-np.inf, 1.0)
    elif what == "sigma2":
        obs.sigma2[777] = np.inf
    else:
        gal = (2e-4, -1e-4, np.inf, 1.0)
    dev = P.DeviceObservation(obs, precision=precision)
    got = dev.extract(*gal, facet)
    dev.close()
    for k in (2, 3, 4):
        np.testing.assert_array_equal(got[k], want[k])


def test_more_channels_than_a_launch_has_shares_of_sixteen(gpu):
    """1,048,577 channels are one more than 65,535 work-groups of sixteen; against the oracle."""
    nch, nrow = 65535 * 16 + 17, 2
    obs = _observation(nrow, nch)
    facet = N.hip().facet_size(1.0, LEN)
    gal = (2e-4, -1e-4, 80.0, 1.0)
    zero = np.zeros(obs.nvis, np.complex128)
    dev = P.DeviceObservation(obs, vis_sky=zero)
    got = dev.extract(*gal, facet)
    dev.close()
    want = O.extract(obs, *gal, facet, obs.vis, zero)
    for k in (2, 3, 4):
        np.testing.assert_array_equal(got[k], want[k])
    # a term is rounded to 2^-31 of the bound (1,024 rows of so many channels fit 62 bits), and
    # a facet's visibility is sum(x) w / sum(sigma^2) over w terms, sigma^2 at least 0.5
    w = want[4][want[4] != 0]
    bound = 80.0 + 2 * np.abs(obs.vis).max()
    assert (np.abs(got[0] - want[0]) / w).max() <= 2.0 ** -29 * bound
