"""The one-launch D1Q5 line step (32 lanes per cell) against the oracle, bit for bit: lengths
around its two-cells-per-wave tiles and its length limit, every interpolator and mirror, a
velocity across the line (the full tensor weights) and non-finite cells."""
import numpy as np
import pytest

import pyoracle as po
from helpers import smooth_random_state
from lbmpond_amd import Pond

pytestmark = pytest.mark.gpu

FIELDS = ("rho", "ux", "uy", "uz", "T")


def run_both(n, interp, fields, steps, **kw):
    print(f"[line] {interp} n={n} steps={steps} {kw}", flush=True)
    o = po.Oracle("D1Q5", (n, 1, 1), interp, **kw)
    o.set_state(*fields)
    o.step(steps)
    with Pond("D1Q5", (n, 1, 1), interp, "fp64", **kw) as p:
        p.set_state(*fields)
        p.step(steps)
        got, f, t = p.fields(), p.populations(), p.timing()
    ref = o.fields()
    for k in FIELDS:
        assert np.array_equal(got[k], ref[k], equal_nan=True), k
    assert np.array_equal(got["niter"], ref["niter"])
    assert np.array_equal(f, o.populations(), equal_nan=True)
    assert t["steps"] == steps and t["total_ms"] > 0


@pytest.mark.parametrize("interp,mirror", [("weno5", 0), ("weno5g", 0), ("lagr4", 0), ("lagr4", 1), ("lagr4", 7)])
@pytest.mark.parametrize("n", [1, 2, 3, 5, 64, 129])
def test_line_lengths(gpu, n, interp, mirror):
    # (a state at rest fits the walls of the mirrored axis)
    f = smooth_random_state((n, 1, 1), seed=n, T0=0.03, u_amp=0.0 if mirror else 0.05, dims=1)
    run_both(n, interp, f, 4, **({"mirror": mirror} if mirror else {}))


@pytest.mark.parametrize("n", [(1 << 16) - 1, (1 << 16) + 1])
def test_lagr4_on_both_sides_of_the_length_limit(gpu, n):
    run_both(n, "lagr4", smooth_random_state((n, 1, 1), seed=4, T0=0.03, dims=1), 2)


@pytest.mark.parametrize("interp", ["weno5", "weno5g", "lagr4"])
def test_velocity_across_the_line_and_nonfinite_cells(gpu, interp):
    n = 70
    rho, ux, uy, uz, T = smooth_random_state((n, 1, 1), seed=9, T0=0.03, dims=1)
    uy[10:20] = 0.3
    uz[15:25] = -0.7
    run_both(n, interp, (rho, ux, uy, uz, T), 3)
    rho[3], T[40], ux[60] = np.nan, np.inf, 1e30
    for v in (rho, ux, uy, uz, T):
        v[30] = 0.0
    run_both(n, interp, (rho, ux, uy, uz, T), 2)
