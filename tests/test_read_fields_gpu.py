"""Large reads (several threads, pinned chunks) against the same planes read one at a time, which stay
below the size that takes them: every element of every plane, with a ragged last chunk, twice."""
import ctypes

import numpy as np
import pytest

from helpers import smooth_random_state
from lbmpond_amd import Pond
from lbmpond_amd.pond import _I32, _dptr, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["split", "fp64"])
def test_all_planes_match_single_planes(gpu, precision):
    shape = (101, 99, 97)
    f = smooth_random_state(shape, seed=2, T0=0.02)
    with Pond("D3Q27", shape, "weno5c", precision) as p:
        p.set_state(*f)
        for _ in range(2):
            p.step(1)
            got = p.fields()
            for i, k in enumerate(("rho", "ux", "uy", "uz", "T")):
                one = np.full(p.n, np.nan)
                ptrs = [None] * 5
                ptrs[i] = _dptr(one)
                assert lib().pond_get_fields(p._h, *ptrs, ctypes.cast(None, _I32)) == 0
                assert np.array_equal(one, got[k]), k
            assert np.array_equal(p.niter(), got["niter"]) and (got["niter"] > 0).all()
