"""rl2_marg_position_eval on many arguments, which are taken one per lane: the same bits as one
per wave, on either side of the change and for more arguments than a launch has waves."""
import numpy as np
import pytest

from radiolensfit2_amd import _native as N

pytestmark = pytest.mark.gpu


def _eval(x):
    out = np.zeros_like(x)
    assert N.hip().rl2_marg_position_eval(len(x), N.dptr(x), N.dptr(out)) == 0, \
        N.hip().rl2_last_error()
    return out


@pytest.mark.parametrize("n", [10239, 10240, 10241, 40001])
def test_lanes_and_waves_give_the_same_bits(gpu, n):
    rng = np.random.default_rng(n)
    x = np.exp(rng.uniform(np.log(2.9), np.log(130.0), n))
    x[:12] = [np.nan, np.inf, -np.inf, 0., -1., 2.9955, 2.99550001, 40., 42.9955, 100., 100.0001, 1e300]
    waves = np.concatenate([_eval(np.ascontiguousarray(p)) for p in np.array_split(x, 8)])
    np.testing.assert_array_equal(_eval(x), waves)


def test_more_arguments_than_a_launch_has_waves(gpu):
    x = np.full(2 ** 26, 7.0)
    x[-1] = 50.0
    few = _eval(np.array([7.0, 50.0]))
    out = _eval(x)
    assert out[-1] == few[1] and np.all(out[:-1] == few[0])
