"""The sky model's kernel (rl2_obs_add_sources): what a catalog may hold at its limits, and its
accuracy, against the model's own expression in plain FP64 and in 80 bits."""
import numpy as np
import pytest

from radiolensfit2_amd import _native as N
from radiolensfit2_amd import pipeline as P
from radiolensfit2_amd import synth

pytestmark = pytest.mark.gpu

ARCSEC = np.pi / 648000.0


def _empty_observation(u, v, w, nch):
    """Zero visibilities at the given baselines (metres)."""
    wn = 2 * np.pi / np.linspace(0.25, 0.22, nch)
    n = len(u) * nch
    return synth.Observation(None, u, v, w, wn, np.linspace(1.0, 0.9, nch), np.ones(n, np.float32),
                             np.zeros(n, bool), 2.0 * np.abs([u, v]).max() * wn[-1] / (2 * np.pi),
                             np.zeros(n, np.complex128))


def _catalog(rows):
    """rows: (flux, scale, e1, e2, l, m)"""
    c = np.array(rows, np.float64).T.copy()
    return synth.Catalog(*(np.ascontiguousarray(x) for x in c), np.zeros(len(rows)))


def _sum_of_models(obs, cat, real=np.float64):
    """sum of flux spec shape exp(i k (u l + v m + w n)), shape = 1 / (den sqrt(den))."""
    u, v, w = (x.astype(real) for x in (obs.u, obs.v, obs.w))
    out = np.zeros((obs.nch, len(u)), np.result_type(real, np.complex64))
    with np.errstate(divide="ignore", over="ignore", invalid="ignore"):
        for g in range(len(cat)):
            f, s, e1, e2, l, m = (real(x[g]) for x in (cat.flux, cat.scale, cat.e1, cat.e2, cat.l,
                                                       cat.m))
            det = 1 - e1 * e1 - e2 * e2
            sf = (s * real(ARCSEC)) ** 2 / (det * det)
            kk = ((1 + e1) * u + e2 * v) ** 2 + (e2 * u + (1 - e1) * v) ** 2
            n = real(np.sqrt(1 - cat.l[g] ** 2 - cat.m[g] ** 2) - 1)  # the host forms it, in FP64
            p = u * l + v * m + w * n
            for c in range(obs.nch):
                k = real(obs.wn[c])
                den = 1 + sf * k * k * kk
                shape = real(obs.spec[c]) * f / (den * np.sqrt(den))
                out[c] += shape * (np.cos(k * p) + 1j * np.sin(k * p))
    return out.reshape(-1)


LIMITS = {
    "unit_e1": (50., .9, 1., 0., 1e-3, -5e-4), "unit_e2": (50., .9, 0., -1., 1e-3, -5e-4),
    "beyond_unit": (50., .9, 1.5, 0., 1e-3, -5e-4), "point": (50., 0., .1, -.2, 1e-3, -5e-4),
    "wide": (50., 1e5, .1, -.2, 1e-3, -5e-4), "square_overflows": (50., 1e200, .1, -.2, 1e-3, -5e-4),
    "infinite_scale": (50., np.inf, .1, -.2, 1e-3, -5e-4), "no_flux": (0., .9, .1, -.2, 1e-3, -5e-4),
    "below_horizon": (50., .9, .1, -.2, 2., 0.), "nan_scale": (50., np.nan, .1, -.2, 1e-3, -5e-4),
}


@pytest.mark.parametrize("precision", [N.RL2_PREC_FP64, N.RL2_PREC_MIXED])
@pytest.mark.parametrize("nch", [1, 3, 4, 9])
def test_sources_at_the_limits_of_a_catalog(gpu, nch, precision):
    """A source whose model vanishes (an ellipticity on the unit circle, a scalelength without a
    finite square) adds nothing and leaves the others; one that is not a number makes NaN."""
    rng = np.random.default_rng(nch)
    obs = _empty_observation(*rng.uniform(-3000, 3000, (2, 300)), rng.uniform(-50, 50, 300), nch)
    dev = P.DeviceObservation(obs, precision=precision)
    try:
        dev.checkpoint()
        for name, row in LIMITS.items():
            cat = _catalog([row, (30., .6, .05, .02, 1e-4, 2e-4)])
            dev.restore()
            dev.add_sources(cat)
            got, want = dev.residual(), _sum_of_models(obs, cat)
            np.testing.assert_array_equal(np.isfinite(got), np.isfinite(want), err_msg=name)
            # phases below 200 revolutions: their rounding is 200 2 pi 2^-52 of the model
            tol = 1e-12 if precision == N.RL2_PREC_FP64 else 2.0 ** -23
            ok = np.isfinite(want)
            assert np.all(np.abs(got[ok] - want[ok]) <= tol * 80.), name
    finally:
        dev.close()


def _rms(x):
    return float(np.sqrt(np.mean(np.abs(x.astype(np.clongdouble)) ** 2)))


@pytest.mark.parametrize("reach", [3e-4, 1e-2, 0.3])
@pytest.mark.parametrize("metres", [5e3, 150e3])
def test_sources_are_as_accurate_as_the_plain_expression(gpu, metres, reach):
    """The error against 80 bits is no larger than that of the model's expression in FP64
    (k p, cos, sin, 1 / (den sqrt(den))), in the whole value and in its modulus."""
    rng = np.random.default_rng(int(metres))
    obs = _empty_observation(*rng.uniform(-metres, metres, (2, 5000)),
                             rng.uniform(-0.1, 0.1, 5000) * metres, 6)
    dev = P.DeviceObservation(obs)
    err, mod = [], []
    try:
        dev.checkpoint()
        for g in range(8):
            cat = _catalog([(50., rng.uniform(.3, 3.), *rng.uniform(-.4, .4, 2),
                             *rng.uniform(-reach, reach, 2))])
            dev.restore()
            dev.add_sources(cat)
            plain = _sum_of_models(obs, cat)
            true = _sum_of_models(obs, cat, np.longdouble)
            size = np.abs(true)
            err.append([(x - true) / size for x in (dev.residual(), plain)])
            mod.append([np.abs(x.astype(np.clongdouble)) / size - 1 for x in (dev.residual(), plain)])
    finally:
        dev.close()
    for kind in (err, mod):
        got, plain = (np.concatenate([x[k] for x in kind]) for k in (0, 1))
        assert _rms(got) <= _rms(plain), (_rms(got), _rms(plain))
