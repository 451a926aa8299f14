"""The work that programs hand to this framework, as cases that can be timed.

A case is one product with an H-matrix (or one solve made of such products)
through a public entry point.  Every matrix comes from the package's own
generator (the 1/(4 pi r) point kernel on a sphere or a cube surface, ACA
compressed), as the tests and the benchmark use it, so leaf shapes, ranks and
factor values are those of real H-matrices; the vectors are drawn from the
seed.  A program uploads a matrix once and multiplies many vectors, so the
plan belongs to what it has in hand.
"""
import ctypes
import functools
import math

import numpy as np
import torch  # before the package: both then share one HIP runtime

import hacapk_hmvm_amd as H

ELEM_BYTES = {"f64": 8, "f32": 4, "bf16": 2}


# ---- the matrices ------------------------------------------------------------
# Generating one takes up to seconds on the host and gives the same matrix each
# time; a few are kept per process.
@functools.lru_cache(maxsize=5)
def _matrix(n, geometry, leaf, eps):
    return H.generate(n, geometry=geometry, leaf=leaf, eps=eps)


def _sizes(case):
    """Orders of the matrices of a batch, spread evenly over log N, none round."""
    c, lo, hi = case["count"], math.log(case["n_min"]), math.log(case["n_max"])
    return [int(math.exp(lo + (hi - lo) * (i + 0.5) / c)) + i % 7 for i in range(c)]


@functools.lru_cache(maxsize=1)
def _batch(count, n_min, n_max, leaf):
    case = {"count": count, "n_min": n_min, "n_max": n_max}
    return [H.generate(n, geometry=("sphere", "cube")[i % 2], leaf=leaf, eps=(1e-4, 1e-6)[i // 2 % 2], seed=3000 + i)
            for i, n in enumerate(_sizes(case))]


def _matrices(case):
    if case["kind"] == "batch":
        return _batch(case["count"], case["n_min"], case["n_max"], case["leaf"])
    return [_matrix(case["n"], case["geometry"], case["leaf"], case["eps"])]


# ---- the cases ---------------------------------------------------------------
def listed():
    def one(name, kind, n, geometry, storage, leaf=32, eps=1e-4, **more):
        return {"name": name, "kind": kind, "n": n, "geometry": geometry, "leaf": leaf, "eps": eps,
                "storage": storage, **more}

    return [
        # The smallest product: a coarse mesh, every launch nearly empty.
        one("apply-f64-1000", "apply", 1000, "sphere", "f64"),
        # The reference benchmark's size that a CPU still runs easily: one
        # product of an outer solver's loop on a small mesh.
        one("apply-f64-4096", "apply", 4096, "sphere", "f64"),
        # The drop-in call of a program written for the reference (v += A b on
        # host vectors, copies in and out included), odd order.
        one("dropin-f64-10007", "dropin", 10007, "cube", "f64"),
        # The headline workload in double precision.
        one("apply-f64-101250", "apply", 101250, "cube", "f64"),
        # The same with FP32 storage for a single-precision program.
        one("apply-f32-101250", "apply", 101250, "cube", "f32"),
        # BF16 storage, as a preconditioner would use it: larger leaves, odd order.
        one("apply-bf16-60013", "apply", 60013, "sphere", "bf16", leaf=64),
        # Several excitations at once on a small mesh.
        one("multi16-f64-4096", "multi", 4096, "sphere", "f64", nrhs=16),
        # Block products of a block Krylov method: 32 vectors, double precision.
        one("multi32-f64-101250", "multi", 101250, "cube", "f64", nrhs=32),
        # 16 vectors, single precision, tight tolerance, odd order.
        one("multi16-f32-30011", "multi", 30011, "sphere", "f32", leaf=64, eps=1e-6, nrhs=16),
        # 64 vectors of a randomised sketch, lowest precision.
        one("multi64-bf16-50021", "multi", 50021, "cube", "bf16", nrhs=64),
        # Independent matrices of many sizes in one batched plan, replayed as a
        # captured graph, single precision.
        {"name": "batch24-f32-graph", "kind": "batch", "count": 24, "n_min": 2000, "n_max": 20000, "leaf": 32,
         "storage": "f32"},
        # A Krylov solve for the charge density under the potential of outer
        # point charges: the few BiCGSTAB iterations (two products each) that
        # take it below 1e-3, host right-hand side and solution.
        one("bicgstab-f64-20000", "bicgstab", 20000, "sphere", "f64", iters=4),
    ]


def draw(rng):
    kind = rng.choice(["apply", "apply", "apply", "multi", "multi", "multi", "dropin", "batch", "bicgstab"])
    if kind == "batch":
        n_min = rng.randint(1000, 3000)
        return {"kind": kind, "count": rng.randint(4, 24), "n_min": n_min, "n_max": rng.randint(2 * n_min, 20000),
                "leaf": rng.choice([16, 32, 64]), "storage": rng.choice(["f64", "f32", "bf16"])}
    top = {"apply": 70000, "multi": 60000, "dropin": 40000, "bicgstab": 20000}[kind]
    case = {"kind": kind, "n": int(math.exp(rng.uniform(math.log(1000), math.log(top)))),
            "geometry": rng.choice(["sphere", "cube"]), "leaf": rng.choice([16, 32, 48, 64]),
            "eps": rng.choice([1e-4, 1e-4, 1e-6]),
            "storage": "f64" if kind in ("dropin", "bicgstab") else rng.choice(["f64", "f32", "bf16"])}
    if kind == "multi":
        case["nrhs"] = rng.choice([16, 32, 64])
    if kind == "bicgstab":
        case["iters"] = rng.randint(2, 4)
    return case


# ---- inputs ------------------------------------------------------------------
def _vectors(case, seed):
    """The input vectors on the host: U[-1, 1], as the benchmark draws them; for
    a solve the potential of 8 point charges outside the surface."""
    nd = sum(h.nd for h in _matrices(case))
    if case["kind"] == "bicgstab":
        rng = np.random.default_rng(seed)
        at, q = rng.standard_normal((8, 3)), rng.uniform(-1.0, 1.0, 8)
        at *= 3.0 / np.linalg.norm(at, axis=1, keepdims=True)
        h = _matrices(case)[0]
        xyz = np.empty((nd, 3))
        H.lib.hgen_points(ctypes.byref(h.params), xyz.ctypes.data_as(H.c_double_p), None)
        return sum(c / (4 * np.pi * np.linalg.norm(xyz - s, axis=1)) for c, s in zip(q, at))
    shape = (nd, case["nrhs"]) if case["kind"] == "multi" else (nd,)
    return np.random.default_rng(seed).uniform(-1.0, 1.0, shape)


def prepare(case, seed):
    kind, mats, x = case["kind"], _matrices(case), _vectors(case, seed)
    if kind == "dropin":
        # the first call on a matrix uploads it: done before a program's loop
        H.hmvm_hip_2(np.zeros(mats[0].nd), mats[0], np.zeros(mats[0].nd))
        return {"kind": kind, "h": mats[0], "x": x}
    plan = H.Plan(mats if kind == "batch" else mats[0], storage=case["storage"])
    if kind == "bicgstab":
        return {"kind": kind, "plan": plan, "b": x, "iters": case["iters"]}
    s = {"kind": kind, "plan": plan, "storage": case["storage"], "x": torch.from_numpy(x).cuda(),
         "y": torch.zeros(x.shape, dtype=torch.float64, device="cuda"), "stream": torch.cuda.Stream()}
    torch.cuda.synchronize()
    if kind == "multi":
        s["nrhs"] = case["nrhs"]
        if H.lib.hmvm_plan_reserve_multi(plan._p, case["nrhs"]):
            raise H.HMVMError(H.lib.hmvm_hip_last_error_message().decode())
    if kind == "batch":
        s["graph"] = plan.graph(s["x"].data_ptr(), s["y"].data_ptr())
    return s


def _single(s):
    """y as the program goes on with it: a program that stores its matrix in
    FP32 or BF16 works on single-precision vectors."""
    if s["storage"] == "f64":
        return s["y"]
    with torch.cuda.stream(s["stream"]):
        return s["y"].to(torch.float32)


def run(s):
    kind = s["kind"]
    if kind == "dropin":
        v = np.zeros(s["h"].nd)
        return H.hmvm_hip_2(v, s["h"], s["x"])
    if kind == "bicgstab":
        return s["plan"].bicgstab(s["b"], max_iter=s["iters"], tol=0.0, use_graph=True, check_every=0)[0]
    stream = s["stream"].cuda_stream
    if kind == "apply":
        s["plan"].apply(s["x"].data_ptr(), s["y"].data_ptr(), stream=stream)
    elif kind == "batch":
        s["graph"].launch(stream)
    elif H.lib.hmvm_plan_apply_multi(s["plan"]._p, s["x"].data_ptr(), s["y"].data_ptr(), s["nrhs"], 0, stream):
        raise H.HMVMError(H.lib.hmvm_hip_last_error_message().decode())
    return _single(s)


def work(case):
    """Every stored element once, every vector once; two operations per element and vector."""
    mats = _matrices(case)
    length, nd = sum(h.mat2.len for h in mats), sum(h.nd for h in mats)
    s, r = ELEM_BYTES[case["storage"]], case.get("nrhs", 1)
    products = 2 * case["iters"] + 1 if case["kind"] == "bicgstab" else 1
    return {"bytes": products * (s * length + 16 * nd * r), "flops": products * 2 * length * r}


# ---- the same in 64 bits, from the leaves alone --------------------------------
def _product(h, x):
    a = h.arrays()
    kt, ndl, ndt = a["kt"].tolist(), a["ndl"].tolist(), a["ndt"].tolist()
    r0, c0 = (a["nstrtl"] - 1).tolist(), (a["nstrtt"] - 1).tolist()
    o1, o2, lowrank, vals = a["a1"].tolist(), a["a2"].tolist(), (a["ltmtx"] == 1).tolist(), a["rowmat"]
    y = np.zeros(x.shape)
    for i in range(len(kt)):
        m, n, k = ndl[i], ndt[i], kt[i]
        xi, yi = x[c0[i]:c0[i] + n], y[r0[i]:r0[i] + m]
        if lowrank[i]:
            t = vals[o1[i]:o1[i] + k * n].reshape(k, n) @ xi
            yi += vals[o2[i]:o2[i] + k * m].reshape(k, m).T @ t
        else:
            yi += vals[o1[i]:o1[i] + m * n].reshape(m, n) @ xi
    return y


def _bicgstab(h, b, iters):
    u, r = np.zeros(b.shape), b.copy()
    shadow, p, ap = r.copy(), np.zeros(b.shape), np.zeros(b.shape)
    beta = zeta = 0.0
    for _ in range(iters):
        p = r + beta * (p - zeta * ap)
        ap = _product(h, p)
        rho = shadow @ r
        alpha = rho / (shadow @ ap)
        t = r - alpha * ap
        at = _product(h, t)
        zeta = (at @ t) / (at @ at)
        u += alpha * p + zeta * t
        r = t - zeta * at
        beta = alpha / zeta * (shadow @ r) / rho
    return u


def exact(case, seed):
    mats, x = _matrices(case), _vectors(case, seed)
    if case["kind"] == "bicgstab":
        return _bicgstab(mats[0], x, case["iters"])
    cuts = np.cumsum([0] + [h.nd for h in mats])
    return np.concatenate([_product(h, x[cuts[q]:cuts[q + 1]]) for q, h in enumerate(mats)])
