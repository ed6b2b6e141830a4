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
