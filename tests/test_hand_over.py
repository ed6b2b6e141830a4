"""The iteration after which the D3Q27 steps leave a cell to their second kernel (pass1_iters): that it
reaches the kernels, and that the results do not depend on it, bit for bit, for states whose cells
mostly go on past the hand-over, many of them to the cap, with stencil windows of several widths and
too far apart for the shared pass, data that is not finite, and starts predicted and abandoned."""
import numpy as np
import pytest

import hip_stub
from helpers import smooth_random_state
from lbmpond_amd import Pond

FIELDS = ("rho", "ux", "uy", "uz", "T", "niter")


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    return hip_stub.build(str(tmp_path_factory.mktemp("stub")))


@pytest.mark.parametrize("precision,interp,kernel,arg", [
    ("split", "weno5c", "k_step_split27_cells", 12), ("fp64", "weno5c", "k_step_f64_27ILi", 7),
    ("fp64", "weno5", "k_step_f64_27ILi", 7), ("fp64", "weno5g", "k_step_f64_27ILi", 7)])
def test_parameter_reaches_the_kernel(stub, precision, interp, kernel, arg):
    out = hip_stub.run(stub, f"""
stub.stub_watch({kernel!r}.encode(), {arg})
for k in (1, 3, 50):
    with Pond("D3Q27", (16, 8, 4), {interp!r}, {precision!r}, pass1_iters=k) as p:
        p.set_state(*[np.ones(p.n)] * 5)
        p.step(1)
    args, blocks = last({kernel!r})
    print(*args)
""")
    assert out.split() == ["1", "3", "50"]


@pytest.mark.parametrize("precision,kernel,arg", [("split", "k_step_split27_cells", 13), ("fp64", "k_step_f64_27ILi", 8)])
def test_given_hand_over_keeps_the_bound_on_the_list(stub, precision, kernel, arg):
    """the number of cells that go at once, whatever their wave does, with pass1_iters given and not"""
    out = hip_stub.run(stub, f"""
stub.stub_watch({kernel!r}.encode(), {arg})
for k in (3, None):
    with Pond("D3Q27", (64, 64, 32), "weno5c", {precision!r}, pass1_iters=k) as p:
        p.set_state(*[np.ones(p.n)] * 5)
        p.step(1)
    print(*last({kernel!r})[0])
""").split()
    assert out[0] == out[1] and 0 < int(out[0]) < 64 * 64 * 32


def jump_state(shape, T0, bad=False):
    f = list(smooth_random_state(shape, seed=3, T0=T0))
    x = np.arange(f[0].size) % shape[0]
    f[0] = np.where(x < shape[0] // 2, 4.0 * f[0], f[0])
    if bad:
        f[0][20], f[4][50] = np.nan, np.inf
    return f


def same_for_every_hand_over(shape, interp, precision, f, steps, values, learned=False, **kw):
    outs = []
    for k in values:
        print(f"[hand-over] {precision} {interp} {shape} {k}", flush=True)
        with Pond("D3Q27", shape, interp, precision, pass1_iters=k, use_mlp=learned, **kw) as p:
            if learned:
                p.mlp_init(seed=5)
                params, scales = p.mlp_params()
                p.mlp_set_params(0.2 * params, scales)
            p.set_state(*f)
            p.step(steps)
            outs.append((p.fields(), p.populations()))
    for o, pop in outs[1:]:
        for k in FIELDS:
            assert np.array_equal(o[k], outs[0][0][k], equal_nan=True), k
        assert np.array_equal(pop, outs[0][1], equal_nan=True)
    return outs[0][0]["niter"]


@pytest.mark.gpu
@pytest.mark.parametrize("learned", [False, True])
@pytest.mark.parametrize("shape,T0,bad", [((17, 9, 8), 0.05, False), ((17, 9, 8), 0.2, False), ((9, 4, 3), 0.2, True),
                                          ((24, 5, 3), 0.6, False), ((9, 4, 3), 2.5, False), ((40, 1, 1), 0.1, False),
                                          ((64, 8, 8), 0.2, False)])
def test_split(gpu, shape, T0, bad, learned):
    niter = same_for_every_hand_over(shape, "weno5c", "split", jump_state(shape, T0, bad), 3 if learned else 1,
                                     (100000, 1, 3, 8, None), learned)
    if shape == (17, 9, 8) and T0 == 0.2 and not learned:
        assert (niter > 16).sum() > 50


@pytest.mark.gpu
def test_split_to_the_cap(gpu):
    niter = same_for_every_hand_over((17, 9, 8), "weno5c", "split", jump_state((17, 9, 8), 0.2), 1,
                                     (100000, 1, 8, None), split_tol_rel=0.0, split_tol_abs=0.0)
    assert (niter >= 100).mean() > 0.9


@pytest.mark.gpu
@pytest.mark.parametrize("interp", ["weno5c", "weno5", "weno5g"])
@pytest.mark.parametrize("shape,T0,bad", [((17, 6, 3), 0.1, False), ((9, 4, 3), 0.2, True), ((9, 4, 3), 0.9, False)])
def test_fp64(gpu, shape, T0, bad, interp):
    niter = same_for_every_hand_over(shape, interp, "fp64", jump_state(shape, T0, bad), 1, (100000, 1, 3, 8, None))
    if shape == (17, 6, 3):
        assert (niter >= 100).any()


@pytest.mark.gpu
@pytest.mark.parametrize("interp", ["weno5", "weno5g"])
@pytest.mark.parametrize("learned", [False, True])
def test_split_as_written(gpu, interp, learned):
    """the second kernel of the WENO5 as written, which takes cells only where pass1_iters asks for it"""
    niter = same_for_every_hand_over((17, 6, 3), interp, "split", jump_state((17, 6, 3), 0.05), 2 if learned else 1,
                                     (None, 1, 3, 8), learned)
    assert (niter > 8).any()


def many_slow(shape, T0):
    """density jumps 16 cells apart: a quarter of the cells go past 8 iterations"""
    f = list(smooth_random_state(shape, seed=3, T0=T0))
    x = np.arange(f[0].size) % shape[0]
    f[0] = np.where(x % 16 < 8, 3.0 * f[0], f[0])
    return f


@pytest.mark.gpu
@pytest.mark.parametrize("shape,tol,least", [((64, 48, 48), None, 8192), ((40, 40, 30), 0.0, 32768)])
def test_split_more_cells_than_go_at_once(gpu, shape, tol, least):
    """late cells beyond those that go at once, in waves with and without cells left to start"""
    niter = same_for_every_hand_over(shape, "weno5c", "split", many_slow(shape, 0.2), 1, (100000, 8, None),
                                     split_tol_rel=tol, split_tol_abs=tol)
    assert (niter > 8).sum() > least


def step_ms(shape, precision, f, pass1_iters, **kw):
    with Pond("D3Q27", shape, "weno5c", precision, pass1_iters=pass1_iters, **kw) as p:
        ms = []
        for _ in range(3):
            p.set_state(*f)
            p.step(1)
            p.sync()
            ms.append(p.timing()["last_ms"])
        print(f"[cap] {precision} {shape} first {pass1_iters}: {min(ms):.2f} ms", flush=True)
        return min(ms)


@pytest.mark.gpu
def test_split_cells_that_all_go_to_the_cap_keep_their_waves(gpu):
    """the workgroup kernel takes several times as long for a cell's iteration as full waves"""
    shape = (80, 80, 80)
    f = smooth_random_state(shape, seed=3, T0=0.02)
    tol0 = dict(split_tol_rel=0.0, split_tol_abs=0.0)
    assert step_ms(shape, "split", f, None, **tol0) < 2 * step_ms(shape, "split", f, 100000, **tol0)


@pytest.mark.gpu
@pytest.mark.parametrize("shape,tol,least", [((32, 24, 20), None, 3000), ((12, 20, 14), 0.0, 3000)])
def test_fp64_more_cells_than_go_at_once(gpu, shape, tol, least):
    niter = same_for_every_hand_over(shape, "weno5c", "fp64", many_slow(shape, 0.2), 1, (100000, 8, None),
                                     tol_rel=tol, tol_abs=tol)
    assert (niter > 8).sum() > least


@pytest.mark.gpu
def test_fp64_cells_that_all_go_to_the_cap_keep_their_waves(gpu):
    shape = (40, 40, 40)
    f = smooth_random_state(shape, seed=3, T0=0.02)
    tol0 = dict(tol_rel=0.0, tol_abs=0.0)
    assert step_ms(shape, "fp64", f, None, **tol0) < 2 * step_ms(shape, "fp64", f, 100000, **tol0)


@pytest.mark.gpu
def test_split_as_written_after_hundreds_of_iterations(gpu):
    """the second kernel of the WENO5 as written takes a cell's count over whatever the first pass's length"""
    niter = same_for_every_hand_over((6, 4, 3), "weno5", "split", jump_state((6, 4, 3), 0.05), 1, (None, 200, 255, 300),
                                     max_iter=400, split_tol_rel=0.0, split_tol_abs=0.0)
    assert (niter == 400).any()
