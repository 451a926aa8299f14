"""Default plans of small matrices (stage-1 bands): sums of a band above FLT_MAX
before the leaf's factor scales give finite t and y, in all modes."""
import numpy as np
import pytest

from test_multi_wide import ND, TOL, WIDE, positive_matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", ["f64", "f32", "bf16"])
def test_band_sums_above_the_fp32_range(gpu, H, O, tmp_path, storage):
    """BF16 factors are stored in (-1, 1): with factors around 1e-6 and x around
    1e36 a band's sum of the stored values exceeds FLT_MAX (2,049 to 5,003
    columns of about 0.5e36), that of a lane's 80 columns does not."""
    h = positive_matrix(H, str(tmp_path / "w.bin"), WIDE, factor=1e-6)
    x = 1e36 * np.random.default_rng(3).uniform(0.5, 1, ND)
    ref = O.seq_2(h, x) * 1e-30
    p = H.Plan(h, storage=storage)
    assert p.info()["n_tslots"] == p.info()["n_t"]  # bands
    y = p.apply_host(x)
    assert np.isfinite(y).all()
    assert np.linalg.norm(y * 1e-30 - ref) <= TOL[storage] * np.linalg.norm(ref)
    for mode in (1, 2):
        p.set_mode(mode)
        assert np.array_equal(p.apply_host(x), y) and p.fault() == 0
    p.close()
