"""Calls on host vectors at odd and even orders, and above the order up to
which they go through pinned memory (131,072): the device product's bits,
also added to y, and with other vectors in between."""
import numpy as np
import pytest

from test_krylov_sizes import block_matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nd", [1, 2, 255, 513, 4097, 131072, 131073])
def test_host_equals_device(gpu, H, tmp_path, nd):
    h = block_matrix(H, str(tmp_path / "m.bin"), nd)
    rng = np.random.default_rng(nd)
    x, x2, y = rng.uniform(-1, 1, (3, nd))
    p = H.Plan(h)
    dx, dy = H.DeviceBuffer(8 * nd), H.DeviceBuffer(8 * nd)
    dx.upload(x)
    p.apply(dx.value, dy.value)
    ref = np.empty(nd)
    dy.download(ref)
    for mode in (0, 1, 2):
        p.set_mode(mode)
        assert np.array_equal(p.apply_host(x), ref)
        other = p.apply_host(x2)
        acc = y.copy()
        p.apply_host(x, acc, accumulate=True)
        assert np.array_equal(acc, y + ref) and np.array_equal(p.apply_host(x2), other)
        both = x.copy()
        p.apply_host(both, both)  # x and y the same array
        assert np.array_equal(both, ref)
    p.close()
