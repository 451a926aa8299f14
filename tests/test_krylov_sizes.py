"""BiCGSTAB at orders around its kernels' blocks (256 rows) and above what its
largest grid covers in one pass (512 blocks), against the CPU iteration; and a
start that is already converged, which runs no iteration."""
import numpy as np
import pytest

from test_krylov import cpu_bicgstab
from test_schedule_replay import write_format1

pytestmark = pytest.mark.gpu


def block_matrix(H, path, nd):
    """Dense blocks of up to 64 rows on the diagonal, shifted: well conditioned."""
    rng = np.random.default_rng(nd)
    leaves = [(2, min(64, nd - r), min(64, nd - r), r + 1, r + 1, 0) for r in range(0, nd, 64)]
    write_format1(path, nd, leaves, rng)
    h = H.loadHmatrix(path)
    a = h.arrays()
    for i, (_, m, _, _, _, _) in enumerate(leaves):
        for v in (a["rowmat"], a["rowmat_t"]):
            v[a["a1"][i]:a["a1"][i] + m * m:m + 1] += 20.0
    return h


@pytest.mark.parametrize("nd", [2, 255, 256, 257, 4097, 131072, 140001])
def test_matches_cpu(gpu, H, O, tmp_path, nd):
    h = block_matrix(H, str(tmp_path / "m.bin"), nd)
    iters = 1 if nd < 255 else 3  # (two rows: solved by two)
    b = np.random.default_rng(7).uniform(0.5, 1, nd)
    u_c, rel_c = cpu_bicgstab(O, h, b, np.zeros(nd), iters)
    p = H.Plan(h)
    runs = [p.bicgstab(b, max_iter=iters, tol=0.0, use_graph=g, check_every=c) for g, c in ((False, 0), (True, 1), (True, 2))]
    p.close()
    for u, r in runs:
        assert np.array_equal(u, runs[0][0]) and r["iters"] == iters and r["relres"] == runs[0][1]["relres"]
        # rounding differences of 1e-16 per operation, amplified by three iterations
        assert np.linalg.norm(u - u_c) <= 1e-8 * np.linalg.norm(u_c) and abs(r["relres"] - rel_c) <= 1e-8


@pytest.mark.parametrize("graph", [False, True])
def test_converged_start(gpu, H, graph):
    h = H.generate(1000)
    p = H.Plan(h)
    u = np.random.default_rng(3).uniform(-1, 1, h.nd)
    b = p.apply_host(u)
    u2, r = p.bicgstab(b, u0=u, max_iter=5, tol=1e-10, use_graph=graph)
    assert np.array_equal(u2, u) and r["iters"] == 0 and r["relres"] < 1e-10 and not r["graph_used"]
    p.close()
