"""Gradients of the proposal network at batches on either side of the blocks that its products are
made in: 16 rows (a tile), 256 (a block of the bias gradients), 512 (a block of the weight
gradients' sums), and sums that are no multiple of 4 or 16 long."""
import ctypes as C

import numpy as np
import pytest

from oracle import mlp_oracle as M
from radiolensfit2_amd import _native as N

pytestmark = pytest.mark.gpu


def _fp(a):
    return a.ctypes.data_as(C.POINTER(C.c_float))


@pytest.mark.parametrize("rows", [1, 3, 15, 16, 17, 255, 256, 257, 511, 512, 513, 770])
def test_gradients_match_the_oracle(gpu, rows):
    """Operands are rounded to 8 bits in both; a value whose FP32 and FP64 sums round apart (1e-6
    over 2^-8, one in some 4,000) moves by 2^-8, so norms agree to about 2^-8 / 60 = 7e-5, and the
    FP32 sums of up to 770 terms to 5e-5."""
    rng = np.random.default_rng(rows)
    x = rng.standard_normal((rows, M.N_IN)).astype(np.float32)
    y = np.concatenate([rng.uniform(-0.3, 0.3, (rows, 2)), rng.normal(-0.1, 0.4, (rows, 1))],
                       1).astype(np.float32)
    p = M.init_params(rows).astype(np.float32)
    H = N.hip()
    h = C.c_void_p()
    N.check(H.rl2_proposal_create(C.byref(h), 7), "rl2_proposal_create")
    try:
        H.rl2_proposal_set_params(h, _fp(p))
        loss = C.c_float()
        assert H.rl2_proposal_gradients(h, rows, _fp(x), _fp(y), C.byref(loss)) == 0
        g = np.zeros(M.n_params(), np.float32)
        H.rl2_proposal_get_grads(h, _fp(g))
    finally:
        H.rl2_proposal_destroy(h)
    want_loss, want = M.gradients(p.astype(np.float64), x.astype(np.float64), y.astype(np.float64),
                                  bf16_ops=True)
    assert abs(loss.value - want_loss) <= 2e-3 * max(1.0, abs(want_loss))
    k = 0
    for layer, (i, o) in enumerate(M.DIMS):
        for kind, n in (("weights", i * o), ("biases", o)):
            a, b = g[k:k + n], want[k:k + n]
            assert np.linalg.norm(a - b) <= 2e-3 * np.linalg.norm(b), (layer, kind)
            k += n
