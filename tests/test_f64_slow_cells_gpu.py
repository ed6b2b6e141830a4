"""The FP64 D3Q27 WENO5 step's slow cells (one workgroup per cell) against the oracle, bit for bit:
density jumps whose cells iterate on past the hand-over, many of them to the cap, in every form of the
interpolator, on lines, with wide windows and with data that is not finite."""
import numpy as np
import pytest

import pyoracle as po
from helpers import smooth_random_state
from lbmpond_amd import Pond

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("interp", ["weno5c", "weno5", "weno5g"])
@pytest.mark.parametrize("shape,T0,bad", [((17, 6, 3), 0.1, False), ((9, 4, 3), 0.2, True), ((9, 4, 3), 0.9, False),
                                          ((40, 1, 1), 0.1, False), ((3, 1, 2), 0.2, False)])
def test_slow_cells(gpu, shape, T0, bad, interp):
    f = list(smooth_random_state(shape, seed=3, T0=T0))
    x = np.arange(f[0].size) % shape[0]
    f[0] = np.where(x < shape[0] // 2, 4.0 * f[0], f[0])
    if bad:
        f[0][20], f[4][50] = np.nan, np.inf
    o = po.Oracle("D3Q27", shape, interp)
    o.set_state(*f)
    o.step(1)
    with Pond("D3Q27", shape, interp, "fp64") as p:
        p.set_state(*f)
        p.step(1)
        got, pop = p.fields(), p.populations()
    ref = o.fields()
    if shape == (17, 6, 3):
        assert (ref["niter"] == 100).any()
    for k in ("rho", "ux", "uy", "uz", "T", "niter"):
        assert np.array_equal(got[k], ref[k], equal_nan=True), k
    assert np.array_equal(pop, o.populations(), equal_nan=True)
