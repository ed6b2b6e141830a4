"""The split D3Q27 step (three lanes per cell, 21 cells per wave): grids of fewer cells than a wave
holds and around its runs, odd rows and mirror walls against the FP64 step, and every run length,
from one tile to longer than the grid, bit for bit against the default, with the plain and the
learned start."""
import numpy as np
import pytest

from helpers import smooth_random_state
from lbmpond_amd import Pond

pytestmark = pytest.mark.gpu

FIELDS = ("rho", "ux", "uy", "uz", "T", "niter")


@pytest.mark.parametrize("interp,mirror", [("weno5c", 0), ("lagr4", 0), ("lagr4", 2), ("lagr4", 7)])
@pytest.mark.parametrize("shape", [(1, 2, 1), (4, 5, 1), (7, 3, 1), (11, 2, 2), (64, 1, 2), (65, 3, 1)])
def test_one_step_within_1e5_of_fp64(gpu, shape, interp, mirror):
    f = smooth_random_state(shape, seed=sum(shape), T0=0.02, u_amp=0.0 if mirror else 0.05)
    with Pond("D3Q27", shape, interp, "fp64", mirror=mirror) as a, \
            Pond("D3Q27", shape, interp, "split", mirror=mirror) as b:
        a.set_state(*f)
        a.step(1)
        b.copy_state_from(a)
        a.step(1)
        b.step(1)
        ref, got = a.fields(), b.fields()
    conv = (ref["niter"] < 100) & (got["niter"] < 100)
    assert conv.mean() > 0.9 and (got["niter"] > 0).all()
    # the split path's stated accuracy; velocities against the thermal speed
    for k in ("rho", "T"):
        assert (np.abs(got[k] - ref[k])[conv] <= 1e-5 * np.abs(ref[k])[conv].max()).all(), k
    for k in ("ux", "uy", "uz"):
        assert (np.abs(got[k] - ref[k])[conv] <= 1e-5 * np.sqrt(ref["T"]).max()).all(), k


@pytest.mark.parametrize("learned", [False, True])
@pytest.mark.parametrize("shape,interp", [((64, 8, 8), "weno5c"), ((37, 6, 5), "weno5c"), ((37, 6, 5), "lagr4")])
def test_run_lengths_are_bitwise_neutral(gpu, shape, interp, learned):
    f = smooth_random_state(shape, seed=7, T0=0.01)
    outs = []
    for kw in ({}, {"refill_chunk": 0}, {"refill_chunk": 3}, {"refill_chunk": 1 << 30}, {"tile_patch": 0}):
        with Pond("D3Q27", shape, interp, "split", use_mlp=learned, **kw) as p:
            if learned:
                p.mlp_init(seed=5)
                params, scales = p.mlp_params()
                p.mlp_set_params(0.2 * params, scales)
            p.set_state(*f)
            p.step(4)
            outs.append((p.fields(), p.populations()))
    for o, pop in outs[1:]:
        for k in FIELDS:
            assert np.array_equal(o[k], outs[0][0][k]), k
        assert np.array_equal(pop, outs[0][1])
