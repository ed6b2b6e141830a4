"""The FP64 D3Q27 step (nine lanes per cell, seven cells per wave) against the oracle, bit for bit:
grids of fewer cells than a wave holds, around its chunks and with odd rows, every interpolator, the
mirror axes, cells hot enough for the one-target path beside cold ones, and a chunk longer than the
grid."""
import numpy as np
import pytest

import pyoracle as po
from helpers import smooth_random_state
from lbmpond_amd import Pond

pytestmark = pytest.mark.gpu

FIELDS = ("rho", "ux", "uy", "uz", "T")


def check_bits(shape, interp, fields, steps, mirror=0, **kw):
    print(f"[groups] {shape} {interp} mirror={mirror} {kw}", flush=True)
    o = po.Oracle("D3Q27", shape, interp, **({"mirror": mirror} if mirror else {}))
    o.set_state(*fields)
    o.step(steps)
    with Pond("D3Q27", shape, interp, "fp64", mirror=mirror, **kw) as p:
        p.set_state(*fields)
        p.step(steps)
        got, f = p.fields(), p.populations()
    ref = o.fields()
    for k in FIELDS:
        assert np.array_equal(got[k], ref[k], equal_nan=True), k
    assert np.array_equal(got["niter"], ref["niter"])
    assert np.array_equal(f, o.populations(), equal_nan=True)


@pytest.mark.parametrize("interp", ["weno5c", "lagr4", "weno5", "weno5g"])
@pytest.mark.parametrize("shape", [(1, 1, 2), (2, 3, 1), (7, 2, 1), (5, 3, 3), (64, 2, 1), (65, 1, 2)])
def test_small_and_odd_grids(gpu, shape, interp):
    check_bits(shape, interp, smooth_random_state(shape, seed=sum(shape), T0=0.02), 2)


@pytest.mark.parametrize("mirror", [1, 2, 4, 7])
def test_mirror_axes(gpu, mirror):
    shape = (9, 5, 4)
    check_bits(shape, "lagr4", smooth_random_state(shape, seed=3, T0=0.02, u_amp=0.0), 2, mirror=mirror)


@pytest.mark.parametrize("interp,mirror", [("weno5c", 0), ("lagr4", 0), ("lagr4", 6), ("weno5", 0)])
def test_hot_and_nonfinite_cells_beside_cold_ones(gpu, interp, mirror):
    shape = (13, 6, 3)
    rho, ux, uy, uz, T = smooth_random_state(shape, seed=5, T0=0.05, u_amp=0.0 if mirror else 0.05)
    T[::7] = 0.9      # s = sqrt(3 T) > 1.5: one target at a time
    T[3::11] = 0.3    # windows several cells apart
    rho[20], T[50] = np.nan, np.inf
    check_bits(shape, interp, (rho, ux, uy, uz, T), 1, mirror=mirror)


@pytest.mark.parametrize("chunk", [0, 1, 2, 1 << 30])
def test_chunks(gpu, chunk):
    shape = (50, 5, 3)
    check_bits(shape, "weno5c", smooth_random_state(shape, seed=6, T0=0.02), 2, refill_chunk=chunk)
