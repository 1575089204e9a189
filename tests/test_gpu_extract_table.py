"""The extraction's default gridding (one table of cells per 512 rows, several copies of each
sum): observations at the edges of its row blocks, in few cells and in more than its table holds,
against the run-merging variant (bit for bit: integer sums of the same terms) and the oracle."""
import numpy as np
import pytest

from oracle import oracle as O
from radiolensfit2_amd import _native as N
from radiolensfit2_amd import pipeline as P
from radiolensfit2_amd import synth

pytestmark = pytest.mark.gpu

LEN, NCH, FLUX, SCALE = 93000.0, 5, 80.0, 1.0


def _observation(nrow, spread, special, length=LEN):
    rng = np.random.default_rng(nrow)
    wn = 2 * np.pi / np.linspace(0.25, 0.22, NCH)
    r = {"one": 2.0, "wide": 0.2 * length}[spread]  # metres: a cell or two, or a cell per row
    u, v = rng.uniform(-r, r, (2, nrow)) + 300.0
    n = nrow * NCH
    vis = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    s2 = rng.uniform(0.5, 2.0, n).astype(np.float32)
    flag = rng.random(n) < 0.1
    flag[0] = False
    if special and nrow > 2:
        vis[1] = complex(np.nan, 1.0)
        s2[nrow + 2] = np.nan
    spec = np.linspace(1.0, 0.9, NCH)
    return synth.Observation(None, u, v, rng.uniform(-50, 50, nrow), wn, spec, s2, flag, length, vis)


@pytest.mark.parametrize("precision", [N.RL2_PREC_FP64, N.RL2_PREC_MIXED])
@pytest.mark.parametrize("spread", ["one", "wide"])
@pytest.mark.parametrize("nrow", [1, 2, 3, 511, 512, 513, 1023, 1024, 1025, 2049, 5001])
def test_extraction_table_matches_the_runs_and_the_oracle(gpu, nrow, spread, precision):
    H = N.hip()
    facet = H.facet_size(SCALE, LEN)
    gal = (2e-4, -1e-4, FLUX, SCALE)
    for special in (False, True):
        obs = _observation(nrow, spread, special)
        zero = np.zeros(obs.nvis, np.complex128)
        dev = P.DeviceObservation(obs, precision=precision, vis_sky=zero)
        try:
            got = dev.extract(*gal, facet)
            N.check(H.rl2_tune_set(N.RL2_TUNE_GRID_VARIANT, 3), "rl2_tune_set")
            try:
                runs = dev.extract(*gal, facet)
            finally:
                N.check(H.rl2_tune_set(N.RL2_TUNE_GRID_VARIANT, 5), "rl2_tune_set")
        finally:
            dev.close()
        for a, b in zip(got, runs):
            np.testing.assert_array_equal(a, b)
        if special:
            continue
        want = O.extract(obs, *gal, facet, obs.vis, zero)
        # complex64 residual: 2^-24 of the largest visibility; otherwise a few ulp of a term
        # and the fixed point's 2^-48 of the bound
        tol = 1e-12 if precision == N.RL2_PREC_FP64 else 2.0 ** -23
        top = FLUX + np.abs(obs.vis).max()
        assert len(got[0]) == len(want[0])
        # a facet's visibility is sum(x) w / sum(sigma^2) over w terms, with sigma^2 of 0.5 to 2:
        # at most 2 w times a term
        w = want[4][want[4] != 0]
        assert (np.abs(got[0] - want[0]) / w).max() <= tol * top * 2
        np.testing.assert_allclose(got[1], want[1], rtol=1e-12)
        np.testing.assert_array_equal(got[2], want[2])
        np.testing.assert_array_equal(got[3], want[3])
        np.testing.assert_array_equal(got[4], want[4])


@pytest.mark.parametrize("spread", ["one", "wide"])
@pytest.mark.parametrize("facet", [1, 2, 31, 32, 33, 64, 97, 255, 256, 257, 300])
def test_compaction_at_the_edges_of_its_tiles(gpu, facet, spread):
    """Facets of less than, exactly and more than whole tiles of 1,024 cells, and either side of
    the 65,536 cells whose copies the compaction writes for the caller, against the oracle."""
    obs = _observation(3000, spread, False, 3 * LEN)  # facets of up to 360 columns
    zero = np.zeros(obs.nvis, np.complex128)
    gal = (2e-4, -1e-4, FLUX, SCALE)
    dev = P.DeviceObservation(obs, vis_sky=zero)
    try:
        dev.extract(*gal, facet)
        got = dev.extract(*gal, facet)  # on accumulators that a compaction has cleared
        n = dev.extract_only(*gal, facet)
    finally:
        dev.close()
    want = O.extract(obs, *gal, facet, obs.vis, zero)
    assert n == len(got[0]) == len(want[0])
    w = want[4][want[4] != 0]
    top = FLUX + np.abs(obs.vis).max()
    # as above; sums of up to 15,000 FP64 terms in the reference's order: 15,000 / 2 ulp at worst
    assert (np.abs(got[0] - want[0]) / w).max() <= 1e-12 * top * 2
    np.testing.assert_allclose(got[1], want[1], rtol=1e-12)
    for k in (2, 3, 4):
        np.testing.assert_array_equal(got[k], want[k])
