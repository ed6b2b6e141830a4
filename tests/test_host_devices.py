"""Reads from a thread whose current device is not the context's (the HIP runtime replaced by
tests/hip_stub.py): small ones, and large ones, which go through several threads."""
import pytest

import hip_stub


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    return hip_stub.build(str(tmp_path_factory.mktemp("stub")))


@pytest.mark.parametrize("precision", ["fp64", "split"])
@pytest.mark.parametrize("shape", [(8, 6, 4), (101, 99, 37)])
def test_read_with_another_device_current(stub, shape, precision):
    out = hip_stub.run(stub, f"""
shape = {shape!r}
f = [np.random.default_rng(k).uniform(0.5, 1, shape[0] * shape[1] * shape[2]).astype(np.float32) for k in range(5)]
stub.hipSetDevice(1)
p = Pond("D3Q27", shape, "weno5c", {precision!r})
p.set_state(*f)
stub.hipSetDevice(0)
got = p.fields()
d = ctypes.c_int(-1)
stub.hipGetDevice(ctypes.byref(d))
print(d.value, "niter" in got and all(v.size == p.n for v in got.values()))
""")
    assert out.split() == ["0", "True"]


@pytest.mark.parametrize("lattice,shape,interp,precision,per_cell", [
    # two states (populations and moments), the node records, the iteration counts and what the second
    # kernel's list takes: 4 bytes per cell for a list of cells, 48 for a two-pass step's entries
    ("D3Q27", (64, 64, 16), "weno5c", "fp64", 2 * (28 * 8 + 5 * 8) + 32 + 4 + 4),
    ("D3Q27", (64, 64, 16), "weno5g", "fp64", 2 * (28 * 8 + 5 * 8) + 32 + 4 + 4),
    ("D3Q27", (64, 64, 16), "lagr4", "fp64", 2 * (28 * 8 + 5 * 8) + 32 + 4),
    ("D3Q27", (64, 64, 16), "weno5c", "split", 2 * (28 * 4 + 4 * 4 + 8) + 16 + 4 + 4),
    ("D3Q27", (64, 64, 16), "weno5", "split", 2 * (28 * 4 + 4 * 4 + 8) + 16 + 4 + 48),
    ("D3Q27", (64, 64, 16), "lagr4", "split", 2 * (28 * 4 + 4 * 4 + 8) + 16 + 4),
    ("D3Q125", (16, 16, 16), "weno5", "fp64", 2 * (128 * 8 + 5 * 8) + 4),
    ("D3Q125", (16, 16, 16), "weno5", "split", 2 * (128 * 4 + 4 * 4 + 8) + 4),
    ("D1Q5", (65536, 1, 1), "lagr4", "fp64", 2 * (5 * 8 + 5 * 8) + 4 + 8),
    ("D1Q5", (65600, 1, 1), "lagr4", "fp64", 2 * (5 * 8 + 5 * 8) + 8 + 4 + 8 + 48),
    ("D1Q5", (256, 256, 1), "weno5", "fp64", 2 * (5 * 8 + 5 * 8) + 8 + 4 + 8 + 48),
])
def test_device_memory_per_cell(stub, lattice, shape, interp, precision, per_cell):
    """a context holds what its step uses"""
    out = hip_stub.run(stub, f"""
with Pond({lattice!r}, {shape!r}, {interp!r}, {precision!r}) as p:
    print(p.device_bytes() - {per_cell} * p.n)
""")
    assert 0 < int(out) < 300000  # the header of the list and the reductions' buffer
