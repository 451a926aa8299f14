"""Multi-RHS products whose X and Y overlap on the device: the bits of separate
vectors, at an order with more row groups than the device runs at once."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hm(H):
    return H.generate(40009, leaf=16, geometry="cube")


@pytest.mark.parametrize("storage", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("nrhs", [16, 64])
@pytest.mark.parametrize("shift", [0, 1, -34])  # doubles from X to Y; -34: 17 16-byte words below
@pytest.mark.parametrize("accumulate", [0, 1])
def test_overlapping_vectors(gpu, H, hm, storage, nrhs, shift, accumulate):
    n = hm.nd * nrhs
    x0, y0 = max(0, -shift), max(0, shift)
    v = np.random.default_rng(6).uniform(-1, 1, n + abs(shift))
    p = H.Plan(hm, storage=storage)
    assert H.lib.hmvm_plan_reserve_multi(p._p, nrhs) == 0
    buf, ref, out = H.DeviceBuffer(8 * len(v)), H.DeviceBuffer(8 * n), np.empty(n)
    buf.upload(v)
    ref.upload(v[y0:y0 + n].copy())
    assert H.lib.hmvm_plan_apply_multi(p._p, buf.value + 8 * x0, ref.value, nrhs, accumulate, None) == 0
    assert H.lib.hmvm_device_synchronize() == 0
    ref.download(out)
    assert H.lib.hmvm_plan_apply_multi(p._p, buf.value + 8 * x0, buf.value + 8 * y0, nrhs, accumulate, None) == 0
    assert H.lib.hmvm_device_synchronize() == 0
    got = buf.download(np.empty(len(v)))
    p.close()
    assert np.array_equal(got[y0:y0 + n], out)
    rest = np.ones(len(v), bool)
    rest[y0:y0 + n] = False
    assert np.array_equal(got[rest], v[rest])
