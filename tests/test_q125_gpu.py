"""The D3Q125 split step (two cells per wave, lane = stencil node) at the sizes where its cell
chunks and halves run out, with and without mirror walls, against the FP64 step; the FP64 step
(shared basis, scalar node loads, mirrored nodes through LDS) against the oracle; and
pond_copy_state between contexts of one precision (whole buffers) against the source."""
import numpy as np
import pytest

import pyoracle as po
from helpers import STATE_ERRORS, smooth_random_state, state_errors
from lbmpond_amd import Pond

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mirror", [0, 7])
@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 1, 1), (5, 3, 1), (2, 7, 3), (17, 4, 3)])
def test_split_q125_small_grids(gpu, shape, mirror):
    # one step from the same state: the split path's stated accuracy (1e-5 of FP64, every cell)
    f = smooth_random_state(shape, seed=sum(shape), T0=0.05, u_amp=0.0 if mirror else 0.05)
    with Pond("D3Q125", shape, "weno5", "fp64", mirror=mirror) as a, \
            Pond("D3Q125", shape, "weno5", "split", mirror=mirror) as b:
        a.set_state(*f)
        a.step(2)
        b.copy_state_from(a)
        a.step(1)
        b.step(1)
        ref, got = a.fields(), b.fields()
    assert (ref["niter"] < 100).all() and (got["niter"] < 100).all() and (got["niter"] > 0).all()
    # (velocities against the thermal speed where the flow is at rest)
    du = max(np.abs(got[k] - ref[k]).max() for k in ("ux", "uy", "uz"))
    assert du <= 1e-5 * np.sqrt(ref["T"]).max()
    errs = state_errors(got, ref)
    for k in STATE_ERRORS:
        if k != "u":
            assert errs[k] <= 1e-5, (k, errs[k])


@pytest.mark.parametrize("bad", [False, True])
@pytest.mark.parametrize("mirror", [0, 1, 2, 4, 7])
@pytest.mark.parametrize("shape", [(1, 1, 1), (3, 2, 1), (5, 3, 2)])
def test_fp64_q125_matches_oracle(gpu, shape, mirror, bad):
    n = int(np.prod(shape))
    rho, ux, uy, uz, T = smooth_random_state(shape, seed=n, T0=0.05, u_amp=0.0 if mirror else 0.05)
    if bad:  # a non-finite term is dropped from its sum
        rho[0], T[n // 2] = np.inf, np.nan
    steps = 1 if bad else 2
    o = po.Oracle("D3Q125", shape, "weno5", **({"mirror": mirror} if mirror else {}))
    o.set_state(rho, ux, uy, uz, T)
    o.step(steps)
    with Pond("D3Q125", shape, "weno5", "fp64", mirror=mirror) as p:
        p.set_state(rho, ux, uy, uz, T)
        p.step(steps)
        got, f = p.fields(), p.populations()
    ref = o.fields()
    for k in ("rho", "ux", "uy", "uz", "T", "niter"):
        assert np.array_equal(got[k], ref[k], equal_nan=True), k
    assert np.array_equal(f, o.populations(), equal_nan=True)


@pytest.mark.parametrize("lattice,precision", [("D1Q5", "fp64"), ("D3Q27", "fp64"), ("D3Q27", "split"),
                                               ("D3Q125", "fp64"), ("D3Q125", "split")])
def test_copy_state_same_precision(gpu, lattice, precision):
    shape = (67, 1, 1) if lattice == "D1Q5" else (9, 5, 3)
    f = smooth_random_state(shape, seed=8, T0=0.03, dims=1 if lattice == "D1Q5" else 3)
    with Pond(lattice, shape, "lagr4", precision) as a, Pond(lattice, shape, "lagr4", precision) as b:
        a.set_state(*f)
        a.step(3)
        b.copy_state_from(a)
        for _ in range(2):
            ga, gb = a.fields(), b.fields()
            assert np.array_equal(a.populations(), b.populations())
            for k in ga:
                assert np.array_equal(ga[k], gb[k]), k
            assert a.diagnostics() == b.diagnostics()
            a.step(2)
            b.step(2)
