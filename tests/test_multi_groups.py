"""The multi-RHS schedule at the sizes where it can go wrong: rows around the
16-row tiles and the 16/32/64-row groups, columns around the slices of 4 and 8
and the batches of 16 and 32, ranks above a group, leaves that cover part of a
group, packed values in windows, and non-finite entries of X."""
import numpy as np
import pytest

from test_schedule_replay import big_rank_matrix, write_format1

TOL = {"f64": 1e-13, "f32": 2e-6, "bf16": 2e-2}  # the bars of test_multi_rhs.py


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def odd_matrix(H, path, nd):
    """Overlapping and ragged leaves: rows and columns one below, at and one
    above the tile, slice and group sizes, ranks 1 to 70, rows no leaf covers."""
    rng = np.random.default_rng(nd)
    leaves = []
    for m in (1, 15, 16, 17, 31, 33, 63, 64, 65, 129):
        for n in (1, 3, 4, 5, 8, 9, 17, 33, 127):
            r, c = int(rng.integers(0, nd - m)) + 1, int(rng.integers(0, nd - n)) + 1
            k = int(rng.choice([0, 1, 2, 7, 16, 17, 70]))
            leaves.append((1, m, n, r, c, k) if rng.random() < 0.6 else (2, m, n, r, c, 0))
    write_format1(path, nd, leaves, rng)
    return H.loadHmatrix(path)


@pytest.mark.parametrize("storage", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("t_mode", [0, 1, 2, 3])
def test_schedule_check(H, tmp_path, storage, t_mode):
    """plan_check builds the multi-RHS schedule too and checks that it packs
    every element once, writes every row once and stays inside its buffers."""
    for nd in (400, 2100, 17000):
        H.plan_check(odd_matrix(H, str(tmp_path / "odd.bin"), nd), storage=storage, t_mode=t_mode)
    for h in (H.generate(5000, geometry="cube", eps=1e-6), H.dummymatrix(40, 40, 6), H.generate(90, leaf=100),
              big_rank_matrix(H, str(tmp_path / "big.bin"))):
        H.plan_check(h, storage=storage, t_mode=t_mode)


def check(H, O, h, storage, nrhs, seed=3):
    X = np.random.default_rng(seed).uniform(-1, 1, (h.nd, nrhs))
    p = H.Plan(h, storage=storage)
    Y = p.apply_multi_host(X)
    p.close()
    for c in (0, 1, nrhs // 2 + 1, nrhs - 1):
        assert rel(Y[:, c], O.seq_2(h, np.ascontiguousarray(X[:, c]))) <= TOL[storage], c
    return X, Y


@pytest.mark.gpu
@pytest.mark.parametrize("storage", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("nrhs", [16, 32, 64])
def test_groups_match_oracle(gpu, H, O, tmp_path, storage, nrhs):
    # around each line of the rule on the matrix order (2,048, 8,192, 16,384 rows)
    for nd in (400, 2047, 2048, 17000):
        check(H, O, odd_matrix(H, str(tmp_path / "odd.bin"), nd), storage, nrhs)
    for h in (H.generate(1000), H.generate(9001, geometry="cube", leaf=48), H.generate(16385, leaf=17),
              H.dummymatrix(40, 40, 6), H.generate(90, leaf=100)):
        check(H, O, h, storage, nrhs)


@pytest.mark.gpu
@pytest.mark.parametrize("storage", ["f64", "f32", "bf16"])
def test_two_waves_a_group(gpu, H, O, storage):
    """From 81,920 rows on a group has two waves (a band of dense blocks on the
    diagonal and one low-rank leaf)."""
    nd, b = 82000, 41
    h = H.dummymatrix(b, b, 4)  # values of one small matrix, repeated by a batch
    p = H.Plan([h] * (nd // h.nd + 1), storage=storage)
    assert p.nd >= 81920
    X = np.random.default_rng(5).uniform(-1, 1, (p.nd, 16))
    Y = p.apply_multi_host(X)
    n = h.nd
    for q in (0, 1, p.nd // n // 2, p.nd // n - 1):
        for c in (0, 15):
            ref = O.seq_2(h, np.ascontiguousarray(X[q * n:(q + 1) * n, c]))
            assert rel(Y[q * n:(q + 1) * n, c], ref) <= TOL[storage]
    p.close()


@pytest.mark.gpu
@pytest.mark.parametrize("storage", ["f64", "bf16"])
def test_packed_in_windows(gpu, H, O, tmp_path, storage, monkeypatch):
    """Where the device lacks the memory for all packed values, every apply
    packs and uses them window by window: same product, also accumulated and
    after another width."""
    h = H.generate(5000, geometry="cube", eps=1e-6)
    for window in (70000, 1000000):
        monkeypatch.setenv("HMVM_MULTI_WINDOW", str(window))
        check(H, O, h, storage, 16)
        X = np.random.default_rng(8).uniform(-1, 1, (h.nd, 32))
        p = H.Plan(h, storage=storage)
        Y = p.apply_multi_host(X)
        assert np.array_equal(p.apply_multi_host(X), Y)
        acc = Y.copy()
        p.apply_multi_host(X, acc, accumulate=True)
        assert rel(acc, 2 * Y) <= 1e-14
        p.close()
    monkeypatch.setenv("HMVM_MULTI_WINDOW", "8")  # below one group's values
    p = H.Plan(h, storage=storage)
    with pytest.raises(H.HMVMError):
        p.apply_multi_host(X)
    p.close()


@pytest.mark.gpu
@pytest.mark.parametrize("storage", ["f64", "f32", "bf16"])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_nonfinite_entries_stay_with_their_leaves(gpu, H, storage, bad):
    """A non-finite entry of X reaches the rows of its own matrix of a batch
    only, although groups, slices and zero columns lie side by side."""
    mats = [H.generate(333, leaf=20), H.generate(517, geometry="cube"), H.generate(101, leaf=7)]
    p = H.Plan(mats, storage=storage)
    o = p.row_offsets
    X = np.random.default_rng(9).uniform(-1, 1, (p.nd, 16))
    Y = p.apply_multi_host(X)
    assert np.isfinite(Y).all()
    Xb = X.copy()
    Xb[o[1] + 5, 3] = Xb[o[2] - 1, 7] = bad
    Yb = p.apply_multi_host(Xb)
    p.close()
    ok = np.ones(Y.shape, bool)
    ok[o[1]:o[2], 3] = ok[o[1]:o[2], 7] = False
    assert np.array_equal(Yb[ok], Y[ok])
    assert not np.isfinite(Yb[~ok]).any()

