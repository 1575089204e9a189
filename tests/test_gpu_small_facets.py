"""Likelihood evaluations on small facets, which run every Newton pass of a task in one
work-group: facets of exactly n cells at the edges of its rows of 256 and chunks of 2048
cells, against the launch-per-pass route (bit for bit) and the FP64 oracle."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O
from radiolensfit2_amd import _native as N
from radiolensfit2_amd import pipeline as P
from radiolensfit2_amd import synth
from tests import _common as T

pytestmark = pytest.mark.gpu

LEN, LAMBDA, FLUX, SCALE = 93000.0, 0.25, 80.0, 1.0


def _facet_of(n, flux=FLUX):
    """An observation whose visibilities sit on n distinct cell centres of the widest facet."""
    rng = np.random.default_rng(n)
    facet = N.hip().facet_size(3.5, LEN)
    inc = 2 * LEN / facet
    cells = np.sort(rng.choice(facet * facet, n, replace=False))
    u = ((cells % facet) + 0.5) * inc - LEN
    v = ((cells // facet) + 0.5) * inc - LEN
    s2 = np.float32((flux * np.sqrt(n) / 40.0) ** 2)
    shape = (1 + (2 * np.pi * SCALE * np.pi / 648000) ** 2 * (u * u + v * v)) ** -1.5
    vis = flux * shape * np.exp(2j * np.pi * (2e-7 * u - 1e-7 * v))
    vis = vis + np.sqrt(s2) * (rng.standard_normal(n) + 1j * rng.standard_normal(n))
    wn = np.array([2 * np.pi / LAMBDA])
    obs = synth.Observation(None, u * LAMBDA, v * LAMBDA, np.zeros(n), wn, np.ones(1),
                            np.full(n, s2, np.float32), np.zeros(n, bool), LEN, vis)
    round_model = (flux * shape).astype(np.complex128)
    dev = P.DeviceObservation(obs, vis_sky=round_model)
    fv, fs, uu, vv, sw = dev.extract(0.0, 0.0, flux, SCALE, facet)
    assert len(uu) == n
    dev.set_prior(P.rprior_for(flux, P.r_grid()))
    return dev, fv, fs, uu, vv


@pytest.mark.parametrize("n", [1, 63, 64, 255, 256, 257, 1793, 2047, 2048, 2049, 4096, 4097,
                               6145, 8191, 8192, 8193])
@pytest.mark.parametrize("points", [1, 9])
def test_small_facets_match_the_passes_and_the_oracle(gpu, n, points):
    dev, fv, fs, uu, vv = _facet_of(n)
    H = N.hip()
    try:
        rng = np.random.default_rng(7)
        e = rng.uniform(-0.5, 0.5, (points, 2))
        got = dev.loglik(e[:, 0], e[:, 1], detail=True)
        N.check(H.rl2_tune_set(N.RL2_TUNE_TILE_PASSES, 3), "rl2_tune_set")  # keeps the passes
        try:
            passes = dev.loglik(e[:, 0], e[:, 1], detail=True)
        finally:
            N.check(H.rl2_tune_set(N.RL2_TUNE_TILE_PASSES, 0), "rl2_tune_set")
        for a, b in zip(got, passes):
            np.testing.assert_array_equal(a[..., 1:] if a.ndim == 2 else a,
                                          b[..., 1:] if b.ndim == 2 else b)
        params, keep = T.oracle_params(fv, fs, uu, vv, FLUX)
        for k in range(min(points, 2)):
            lr, nit, err = np.zeros(40), np.zeros(40, np.int32), C.c_int()
            le = O.lib().orl2_loglikelihood_detail(C.byref(params), e[k, 0], e[k, 1],
                                                   C.byref(err), O.ptr(lr),
                                                   nit.ctypes.data_as(O.c_int_p))
            if n < 255:
                continue  # a handful of cells: the sign of the determinant is rounding
            assert got[1][k] == err.value
            np.testing.assert_array_equal(got[3][k, 1:24], nit[1:24])
            np.testing.assert_allclose(got[2][k, 1:24], lr[1:24], rtol=0, atol=1e-8)
            assert abs(got[0][k] - le) <= 1e-8
    finally:
        dev.close()


@pytest.mark.parametrize("n", [200, 9000])
@pytest.mark.parametrize("points", [1, 8, 9, 40])
def test_results_polled_for_are_those_of_a_synchronised_evaluation(gpu, n, points):
    """Evaluations that return on their results (L_e alone, L_r of up to 8 points) in turns on one
    set of buffers, and one that synchronises (with statistics): the same bits every time."""
    dev = _facet_of(n)[0]
    try:
        e = np.random.default_rng(points).uniform(-0.5, 0.5, (2, points, 2))
        P.stats_enable(True)
        want = [dev.loglik(x[:, 0], x[:, 1], detail=True) for x in e]
        P.stats_enable(False)
        for _ in range(3):
            for x, w in zip(e, want):
                for detail in (False, True):
                    got = dev.loglik(x[:, 0], x[:, 1], detail=detail)
                    for a, b in zip(got, w):
                        np.testing.assert_array_equal(a[..., 1:] if a.ndim == 2 else a,
                                                      b[..., 1:] if b.ndim == 2 else b)
    finally:
        P.stats_enable(False)
        dev.close()
