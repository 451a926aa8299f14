"""Multi-RHS products of stacks wider than one stage-1 group (2,048 columns),
whose groups leave slots that a t sum adds, and sums beyond the FP32 range."""
import numpy as np
import pytest

from test_schedule_replay import write_format1

TOL = {"f64": 1e-13, "f32": 2e-6, "bf16": 2e-2}  # the bars of test_multi_rhs.py
ND = 5100


def positive_matrix(H, path, leaves, factor=1.0):
    """Leaves of values 0.5 .. 1 times `factor`."""
    write_format1(path, ND, leaves, np.random.default_rng(1))
    h = H.loadHmatrix(path)
    a = h.arrays()
    for v in (a["rowmat"], a["rowmat_t"]):
        v[:] = (0.75 + 0.25 * v) * factor
    return h


# (ltmtx, ndl, ndt, nstrtl, nstrtt, kt): columns one above one group's, one
# above two groups', and of a ragged third group; ranks around the 16-row tiles
# and above a group; two leaves each of the same columns
WIDE = [(1, 40, 2049, 1, 3, 17), (1, 65, 4097, 50, 900, 33), (1, 7, 4097, 200, 900, 1),
        (1, 129, 5003, 300, 60, 70), (1, 16, 5003, 700, 60, 300)]


def product(H, h, storage, X):
    p = H.Plan(h, storage=storage)
    Y = p.apply_multi_host(X)
    p.close()
    return Y


@pytest.mark.gpu
@pytest.mark.parametrize("storage", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("nrhs", [16, 32, 64])
def test_infinite_entries_stay_infinite(gpu, H, tmp_path, storage, nrhs):
    """All factors are positive: an infinite entry of X makes the rows of its
    leaves infinite, of its sign, not NaN; other entries of Y keep their bits."""
    h = positive_matrix(H, str(tmp_path / "w.bin"), WIDE)
    X = np.random.default_rng(2).uniform(0.5, 1, (ND, nrhs))
    Y = product(H, h, storage, X)
    Xb, want = X.copy(), Y.copy()
    for col, row, bad in ((0, 100, np.inf), (3, 2500, -np.inf), (nrhs - 1, 5050, np.inf)):
        Xb[row, col] = bad
        for _, m, n, r, c, _ in WIDE:
            if c - 1 <= row < c - 1 + n:
                want[r - 1:r - 1 + m, col] = bad
    assert np.isinf(want).any()
    assert np.array_equal(product(H, h, storage, Xb), want)


@pytest.mark.gpu
@pytest.mark.parametrize("nrhs", [16, 32, 64])
def test_bf16_t_above_the_fp32_range_before_its_scales(gpu, H, O, tmp_path, nrhs):
    """BF16 factors are stored in (-1, 1): with factors around 1e-6 and X
    around 1e36 the sum of the stored values of a row exceeds FLT_MAX (5,003
    columns of about 0.75 times 1e36), t and y do not, nor does a chunk of 64
    columns."""
    h = positive_matrix(H, str(tmp_path / "w.bin"), WIDE, factor=1e-6)
    X = 1e36 * np.random.default_rng(3).uniform(0.5, 1, (ND, nrhs))
    Y = product(H, h, "bf16", X)
    assert np.isfinite(Y).all()
    for c in (0, nrhs - 1):
        ref = O.seq_2(h, np.ascontiguousarray(X[:, c]))
        assert np.linalg.norm(Y[:, c] * 1e-30 - ref * 1e-30) <= TOL["bf16"] * np.linalg.norm(ref * 1e-30)


@pytest.mark.gpu
@pytest.mark.parametrize("storage,nrhs", [("f32", 16), ("f32", 32), ("f32", 64), ("bf16", 16), ("bf16", 32), ("bf16", 64)])
def test_rows_of_y_above_the_fp32_range(gpu, H, O, tmp_path, storage, nrhs):
    """12 dense leaves of 400 columns side by side, X around 1e36: the sum of a
    leaf is below FLT_MAX, that of a wave's share of the columns (1,200) and y
    (FP64) above.  Rows 1 to 64 are taller than a group, rows 101 to 120 part
    of one."""
    h = positive_matrix(H, str(tmp_path / "d.bin"),
                        [(2, m, 400, r, 1 + 400 * q, 0) for m, r in ((64, 1), (20, 101)) for q in range(12)])
    X = 1e36 * np.random.default_rng(4).uniform(0.5, 1, (ND, nrhs))
    Y = product(H, h, storage, X)
    assert np.isfinite(Y).all() and Y.max() > 3.5e38
    for c in (0, nrhs - 1):
        ref = O.seq_2(h, np.ascontiguousarray(X[:, c]))
        assert np.linalg.norm(Y[:, c] * 1e-30 - ref * 1e-30) <= TOL[storage] * np.linalg.norm(ref * 1e-30)


def long_sums(H, path, big, nrhs, stage1):
    """64 leaves of 64 columns side by side, all ones, X one but for `big` in
    the first row.  Dense leaves (64 rows taller than a group and 20 rows that
    are part of one), or one stack of rank 32 of which y is the first row."""
    leaves = [(2, m, 64, r, 1 + 64 * q, 0) for m, r in ((64, 1), (20, 101)) for q in range(64)]
    if stage1:
        leaves = [(1, 64, 4096, 1, 1, 32), (1, 20, 4096, 101, 1, 32)]
    write_format1(path, ND, leaves, np.random.default_rng(1))
    h = H.loadHmatrix(path)
    a = h.arrays()
    for v in (a["rowmat"], a["rowmat_t"]):
        v[:] = 1.0
    if stage1:
        for i, (_, m, _, _, _, k) in enumerate(leaves):
            a["rowmat"][a["a2"][i] + m:a["a2"][i] + m * k] = 0.0
    X = np.ones((ND, nrhs))
    X[0] = big
    return h, X


@pytest.mark.gpu
@pytest.mark.parametrize("nrhs", [16, 32, 64])
@pytest.mark.parametrize("storage,big,stage1", [("f64", 2.0**53, False), ("f64", 2.0**53, True),
                                                ("bf16", 2.0**30, False), ("f32", 2.0**28, False),
                                                ("f32", 2.0**28, True)])
def test_chains_of_roundings_stay_short(gpu, H, tmp_path, storage, big, stage1, nrhs):
    """Ones added to a number of which one is half the last bit or less are lost, and
    kept in sums of their own: of 4,096 columns no more than the 64 of a leaf
    may be added in the same chain as the first."""
    h, X = long_sums(H, str(tmp_path / "l.bin"), big, nrhs, stage1)
    Y = product(H, h, storage, X)
    for r, m in ((0, 64), (100, 20)):
        assert np.abs(Y[r:r + m] - big - 4095).max() <= 64, np.unique(Y[r:r + m] - big)


@pytest.mark.gpu
@pytest.mark.parametrize("nrhs", [16, 32, 64])
@pytest.mark.parametrize("storage", ["f64", "f32", "bf16"])
def test_wide_stacks_match_oracle(gpu, H, O, tmp_path, storage, nrhs, monkeypatch):
    """Random factors, at once and in windows; BF16 (whose t is rounded to BF16)
    keeps its bits under other layouts of the one-vector launches."""
    write_format1(str(tmp_path / "r.bin"), ND, WIDE + [(2, 33, 65, 900, 1, 0), (2, 17, 9, 950, 20, 0)],
                  np.random.default_rng(5))
    h = H.loadHmatrix(str(tmp_path / "r.bin"))
    X = np.random.default_rng(nrhs).uniform(-1, 1, (ND, nrhs))
    ref = {c: O.seq_2(h, np.ascontiguousarray(X[:, c])) for c in (0, 5, nrhs - 1)}

    def check(**kw):
        p = H.Plan(h, storage=storage, **kw)
        one = p.info()["device_bytes"]
        Y = p.apply_multi_host(X)
        held.append(p.info()["device_bytes"] - one)
        p.close()
        for c, r in ref.items():
            assert np.linalg.norm(Y[:, c] - r) <= TOL[storage] * np.linalg.norm(r), c
        return Y

    held = []
    Y = check()
    for kw in ({"t_mode": 1}, {"t_mode": 0}, {"t_mode": 2}, {"w2": 500, "w3": 700, "max_rows_b": 40}):
        Z = check(**kw)
        assert storage != "bf16" or np.array_equal(Z, Y), kw
    # in windows: a quarter of the values' bytes less than all takes
    monkeypatch.setenv("HMVM_MULTI_LIMIT", str(held[0] - h.mat2.len * {"f64": 8, "f32": 4, "bf16": 2}[storage] // 4))
    Z = check()
    assert held[-1] < held[0]
    assert storage != "bf16" or np.array_equal(Z, Y)
