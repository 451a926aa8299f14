"""Device memory of the multi-RHS schedule: what a plan reports, and what it
does where memory is short."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BYTES = {"f64": 8, "f32": 4, "bf16": 2}
TOL = {"f64": 1e-13, "f32": 2e-6, "bf16": 2e-2}  # the bars of test_multi_rhs.py


def reserve(H, p, nrhs):
    return H.lib.hmvm_plan_reserve_multi(p._p, nrhs)


@pytest.mark.parametrize("storage", ["f64", "f32", "bf16"])
def test_device_bytes_count_the_packed_copy(gpu, H, storage, monkeypatch):
    h = H.generate(5000, geometry="cube", eps=1e-6)
    p = H.Plan(h, storage=storage)
    values = BYTES[storage] * h.mat2.len
    one = p.info()["device_bytes"]
    held = []
    for nrhs in (16, 32, 16, 64):
        assert reserve(H, p, nrhs) == 0
        held.append(p.info()["device_bytes"] - one)
    work = held[1] - held[0]  # 16 right-hand sides
    assert work >= 16 * h.nd * 16 and held[2] == held[1] and held[3] - held[1] == 2 * work
    assert values <= held[0] - work <= 3 * values
    p.close()
    monkeypatch.setenv("HMVM_MULTI_WINDOW", "70000")
    p = H.Plan(h, storage=storage)
    assert reserve(H, p, 16) == 0
    assert p.info()["device_bytes"] - one < held[0] - values + BYTES[storage] * 70000 + values // 4  # pack records stay
    p.close()


@pytest.mark.parametrize("storage", ["f64", "f32", "bf16"])
def test_window_shrinks_until_the_work_buffers_fit(gpu, H, O, storage, monkeypatch):
    """Where memory is short (a limit), reserving takes a window that leaves room
    for the work buffers: below half of the values, after growth to more
    columns, and again on a plan that already has a window."""
    h = H.generate(5000, geometry="cube", eps=1e-6)
    X = np.random.default_rng(8).uniform(-1, 1, (h.nd, 64))
    refs = {c: O.seq_2(h, np.ascontiguousarray(X[:, c])) for c in (0, 15)}

    def check(p, nrhs):
        Y = p.apply_multi_host(np.ascontiguousarray(X[:, :nrhs]))
        for c, ref in refs.items():
            assert np.linalg.norm(Y[:, c] - ref) <= TOL[storage] * np.linalg.norm(ref)

    p = H.Plan(h, storage=storage)
    one = p.info()["device_bytes"]
    held = {}
    for nrhs in (16, 64):
        assert reserve(H, p, nrhs) == 0
        held[nrhs] = p.info()["device_bytes"] - one
    p.close()
    work = (held[64] - held[16]) // 3  # 16 right-hand sides
    packed = held[16] - work
    for limit, steps in ((packed // 3 + work, (16,)), (packed + 2 * work, (16, 64)), (packed // 2 + work, (16, 32, 64))):
        monkeypatch.setenv("HMVM_MULTI_LIMIT", str(limit + packed // 4))  # the schedule's lists and pack records
        p = H.Plan(h, storage=storage)
        for nrhs in steps:
            assert reserve(H, p, nrhs) == 0, (limit, nrhs, H.lib.hmvm_hip_last_error_message())
            assert p.info()["device_bytes"] - one <= limit + packed // 4
            check(p, nrhs)
        p.close()
    monkeypatch.setenv("HMVM_MULTI_LIMIT", str(work))  # not even one group's values
    p = H.Plan(h, storage=storage)
    with pytest.raises(H.HMVMError, match="HMVM_MULTI_LIMIT"):
        check(p, 16)
    monkeypatch.delenv("HMVM_MULTI_LIMIT")
    check(p, 64)
    p.close()
