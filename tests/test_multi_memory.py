"""Device memory of the multi-RHS schedule: what a plan reports."""
import pytest

pytestmark = pytest.mark.gpu

BYTES = {"f64": 8, "f32": 4, "bf16": 2}


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
