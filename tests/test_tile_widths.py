"""The default tile sizes around the lines of their rule: products of the same
matrix under the tile sizes that the rule gives to other matrix sizes, against
the oracle, and plans of the default at each size checked."""
import numpy as np
import pytest

TOL = {"f64": 1e-13, "f32": 2e-6, "bf16": 2e-2}  # the bars of test_multi_rhs.py
STEPS = [(64, 64, 64), (1024, 1024, 96), (8192, 1365, 64), (8192, 5461, 64), (20480, 13653, 192), (32768, 24576, 160)]


@pytest.mark.parametrize("storage", ["f64", "f32", "bf16"])
def test_default_widths_check(H, storage):
    for n, kw in ((90, {"leaf": 100}), (1000, {}), (2600, {"leaf": 64, "eps": 1e-6}), (9001, {"geometry": "cube"})):
        H.plan_check(H.generate(n, **kw), storage=storage)


@pytest.mark.gpu
@pytest.mark.parametrize("storage", ["f64", "f32", "bf16"])
def test_products_across_the_rule(gpu, H, O, storage):
    h = H.generate(4003, geometry="cube", leaf=48, eps=1e-6)
    x = np.random.default_rng(7).standard_normal(h.nd)
    ref = O.seq_2(h, x)
    for w, w3, rows in STEPS:
        p = H.Plan(h, storage=storage, w1=w, w2=w, w3=w3, max_rows_b=rows)
        y = p.apply_host(x)
        p.close()
        assert np.linalg.norm(y - ref) <= TOL[storage] * np.linalg.norm(ref), (w, w3, rows)
