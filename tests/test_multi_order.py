"""BF16 products with several right-hand sides: t is rounded to BF16, so its
sums keep one order whatever the layout of the one-vector launches: the same
bits from plans of other t_modes and tile sizes of the other launches, and at
chunks of less than a step, ranks above a group, and stacks of several
groups of columns."""
import numpy as np
import pytest

from test_multi_groups import odd_matrix
from test_schedule_replay import big_rank_matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["odd", "big", "cube"])
@pytest.mark.parametrize("nrhs", [16, 32, 64])
def test_same_bits(gpu, H, O, tmp_path, kind, nrhs):
    if kind == "odd":
        h = odd_matrix(H, str(tmp_path / "odd.bin"), 2100)
    elif kind == "big":
        h = big_rank_matrix(H, str(tmp_path / "big.bin"))
    else:
        h = H.generate(6007, geometry="cube", eps=1e-6)
    X = np.random.default_rng(nrhs).uniform(-1, 1, (h.nd, nrhs))
    for base in ({}, {"w1": 64}, {"w1": 3000, "max_rows": 20}):
        ref = None
        for kw in ({}, {"t_mode": 1}, {"t_mode": 0}, {"w2": 500, "w3": 700, "max_rows_b": 40}):
            p = H.Plan(h, storage="bf16", **base, **kw)
            Y = p.apply_multi_host(X)
            p.close()
            if ref is None:
                ref = Y
                for c in (0, nrhs - 1):  # the bar of test_multi_rhs.py
                    y = O.seq_2(h, np.ascontiguousarray(X[:, c]))
                    assert np.linalg.norm(Y[:, c] - y) <= 2e-2 * np.linalg.norm(y)
            assert np.array_equal(Y, ref), (base, kw)
