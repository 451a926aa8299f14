"""Default plans of small matrices: stage-1 tiles are bands of one slot per t
entry, written to t by the launches and to the slots by the persistent launch,
which sums them.  All modes give one another's bits; against the oracle at
matrices without low-rank leaves, of ranks above a tile's rows, and with leaves
that straddle bands."""
import numpy as np
import pytest

from test_multi_groups import odd_matrix, rel
from test_schedule_replay import big_rank_matrix, replay

TOL = {"f64": 1e-13, "f32": 2e-6, "bf16": 2e-2}  # the bars of test_multi_rhs.py


def matrix(H, tmp_path, kind):
    if kind == "dense":
        return H.generate(90, leaf=100)
    if kind == "big":
        return big_rank_matrix(H, str(tmp_path / "big.bin"))
    if kind == "odd":
        return odd_matrix(H, str(tmp_path / "odd.bin"), 400)
    return H.generate(2500, geometry="cube", eps=1e-6)


@pytest.mark.parametrize("kind", ["dense", "big", "odd", "cube"])
@pytest.mark.parametrize("kw", [{}, {"w1": 64, "max_rows": 17}, {"w1": 1 << 20}])
def test_bands_replay(H, O, tmp_path, kind, kw):
    h = matrix(H, tmp_path, kind)
    for storage in ("f64", "f32", "bf16"):
        H.plan_check(h, storage=storage, **kw)
    x = np.random.default_rng(3).uniform(-1, 1, h.nd)
    for multi in (False, True):  # through the slots, and straight to t
        y, s = replay(H, h, x, multi=multi, **kw)
        assert s["n_tslots"] == s["n_t"] == len(s["tmap"]) == s["tsum"]["n"]
        assert rel(y, O.seq_2(h, x)) <= 1e-13


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["dense", "big", "odd", "cube"])
@pytest.mark.parametrize("storage", ["f64", "f32", "bf16"])
def test_bands_modes(gpu, H, O, tmp_path, kind, storage):
    h = matrix(H, tmp_path, kind)
    rng = np.random.default_rng(5)
    x, x2 = rng.uniform(-1, 1, (2, h.nd))
    p = H.Plan(h, storage=storage)
    assert p.info()["n_tslots"] == p.info()["n_t"]
    y0, y2 = p.apply_host(x), p.apply_host(x2)
    assert rel(y0, O.seq_2(h, x)) <= TOL[storage]
    for mode in (1, 2, 0):
        p.set_mode(mode)
        assert np.array_equal(p.apply_host(x2), y2) and np.array_equal(p.apply_host(x), y0) and p.fault() == 0
    n = p.info()["ntiles_a"]
    perm = np.arange(n, dtype=np.int32)[::-1].copy()
    p.set_tile_order(0, perm)  # tiles uploaded again
    assert np.array_equal(p.apply_host(x2), y2) and np.array_equal(p.apply_host(x), y0)
    if p.info()["ntiles_b"]:  # the timed launch B reads the t that launch A wrote
        p.profile_tiles(1, 1)
        assert np.array_equal(p.apply_host(x), y0)
    dx, dy = H.DeviceBuffer(8 * h.nd), H.DeviceBuffer(8 * h.nd)
    g = p.graph(dx.value, dy.value)
    for v, ref in ((x, y0), (x2, y2), (x, y0)):
        dx.upload(v)
        g.launch()
        out = np.empty(h.nd)
        dy.download(out)
        assert np.array_equal(out, ref)
    g.close()
    p.close()
