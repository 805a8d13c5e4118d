"""Timed workloads of the solver through its public Python entry points.

Each case is one call that a user's program makes: a whole solve from host
data (``pdhcg_amd.solve``), a whole batch (``solve_batch``), a sequence of
cone projections, or the training of the warm-start network.  The instance
families are those of ``pdhcg_amd.workloads``; the conic family below is the
conic mix without exponential blocks (with them its inner solve runs to the
iteration limit and its path depends on the last bit of every step).

Sizes of the single solves run from the smallest instances of the tests (60
variables) to the large low-rank QP (10^6 variables, 10^7 nonzeros).  Solves
stop at a relative KKT tolerance, or at an iteration limit where the whole
solve would take seconds.
"""
from __future__ import annotations

import math
from dataclasses import replace

import numpy as np
import scipy.sparse as sp

import pdhcg_amd
from pdhcg_amd import PRECISION_FP64, PRECISION_MIXED, capi, workloads
from pdhcg_amd.warmstart import MLP

_PRECISION = {"fp64": PRECISION_FP64, "mixed": PRECISION_MIXED}


def listed():
    return [
        # the smallest calls: an instance of the test suite's size, where
        # launches, allocations and host work are everything
        dict(name="qp_tiny", kind="tiny", objective="lowrank_diag", n=60, m=30, precision="fp64", eps=1e-6,
             iterations=100000),
        # the small random convex QP with a general sparse Q (inner solve)
        dict(name="qp_sparse_q", kind="sparse_q", n=2000, m=1000, precision="fp64", eps=1e-4, iterations=100000),
        # an ordinary LP: power-law rows, box bounds
        dict(name="lp_medium", kind="family", objective="lp", n=20000, m=10000, nnz=200000, rank=0, precision="fp64",
             eps=1e-4, iterations=100000),
        # the parametric family's stated size: sparse rows and a dense low-rank term
        dict(name="lowrank_medium", kind="family", objective="lowrank", n=100000, m=50000, nnz=1000000, rank=50,
             precision="fp64", eps=1e-4, iterations=100000),
        # the large low-rank QP from host data, stopped after 400 iterations
        dict(name="lowrank_large", kind="family", objective="lowrank", n=1000000, m=500000, nnz=10000000, rank=50,
             precision="fp64", eps=1e-6, iterations=400),
        # half of it in mixed precision (FP32 iterates and matrices, FP64 evaluation)
        dict(name="lowrank_large_mixed", kind="family", objective="lowrank", n=500000, m=250000, nnz=5000000, rank=50,
             precision="mixed", eps=1e-6, iterations=300),
        # many small portfolio problems of uneven size in one call
        dict(name="portfolio_batch", kind="portfolio", count=256, n_low=50, n_high=2000, k_low=10, k_high=50,
             precision="fp64", eps=1e-6),
        # the same in mixed precision
        dict(name="portfolio_batch_mixed", kind="portfolio", count=256, n_low=50, n_high=2000, k_low=10, k_high=50,
             precision="mixed", eps=1e-6),
        # instances of one parametric family, solved together at the tolerance
        # at which warm-start training data are made
        dict(name="parametric_batch", kind="parametric", count=256, n=2000, m=1000, nnz=20000, rank=50,
             precision="fp64", eps=1e-4),
        # a conic QP: SOC, RSOC, power and PSD blocks, a sparse Q, affine SOC rows
        dict(name="conic_qp", kind="conic", soc=300, rsoc=200, power=1000, psd=12, psd_low=8, psd_high=64,
             precision="fp64", eps=1e-6, iterations=60),
        # PSD projections alone: matrices that move a little from point to
        # point, as a solver's iterates do
        dict(name="psd_sequence", kind="psd", blocks=67, order_low=16, order_high=128, points=8),
        # training the warm-start network on solved instances
        dict(name="warm_start_train", kind="train", z=16, hidden=1024, out=3000, samples=4096, batch=256, epochs=4),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["tiny", "sparse_q", "family", "family", "family", "portfolio", "parametric", "conic", "psd",
                       "train"])
    precision = rng.choice(["fp64", "mixed"])
    if kind == "tiny":
        n = _log(rng, 20, 500)
        return dict(kind=kind, objective=rng.choice(["lp", "diag", "sparse", "lowrank", "lowrank_diag",
                                                     "lowrank_dense_d", "lowrank_sparse_r"]),
                    n=n, m=max(5, n // rng.choice([2, 3, 5])), precision=precision, eps=1e-6, iterations=5000)
    if kind == "sparse_q":
        n = _log(rng, 300, 6000)
        return dict(kind=kind, n=n, m=max(10, n // rng.choice([1, 2, 4])), precision=precision, eps=1e-4,
                    iterations=2000)
    if kind == "family":
        objective = rng.choice(["lp", "diag", "lowrank", "lowrank"])
        n = _log(rng, 1000, 400000)
        m = max(10, int(n * rng.uniform(0.2, 1.2)))
        return dict(kind=kind, objective=objective, n=n, m=m, nnz=int(m * rng.uniform(8, 24)),
                    rank=rng.randint(3, 70) if objective == "lowrank" else 0, precision=precision, eps=1e-4,
                    iterations=400)
    if kind == "portfolio":
        low = _log(rng, 20, 400)
        return dict(kind=kind, count=_log(rng, 8, 256), n_low=low, n_high=low + _log(rng, 50, 1600), k_low=3,
                    k_high=rng.randint(8, 60), precision=precision, eps=1e-6)
    if kind == "parametric":
        n = _log(rng, 200, 3000)
        m = max(20, int(n * rng.uniform(0.3, 0.8)))
        return dict(kind=kind, count=_log(rng, 8, 200), n=n, m=m, nnz=10 * n, rank=rng.randint(5, 60),
                    precision=precision, eps=1e-4)
    if kind == "conic":
        high = rng.randint(9, 64)
        return dict(kind=kind, soc=_log(rng, 10, 300), rsoc=_log(rng, 10, 200), power=_log(rng, 20, 1000),
                    psd=rng.randint(1, 12), psd_low=rng.randint(2, 8), psd_high=high, precision="fp64", eps=1e-6,
                    iterations=40)
    if kind == "psd":
        high = rng.randint(17, 140)
        return dict(kind=kind, blocks=_log(rng, 1, 100), order_low=rng.randint(2, 16), order_high=high, points=6)
    return dict(kind=kind, z=rng.randint(3, 40), hidden=16 * rng.randint(4, 64), out=_log(rng, 200, 4000),
                samples=_log(rng, 512, 4096), batch=16 * rng.choice([4, 8, 13, 16, 32]), epochs=4)


# ---------------------------------------------------------------------------
# instances
# ---------------------------------------------------------------------------

def _family(case, seed):
    """The large sparse QP's family at any size: power-law rows in A, box
    [0, 5], diagonal Q, dense R and diagonal D (or a part of the objective)."""
    rng = np.random.default_rng(seed)
    n, m, k = case["n"], case["m"], case["rank"]
    lens = workloads.zipf_lengths(rng, m, max(m, case["nnz"]), 1.5, min(5000, n))
    ptr = np.zeros(m + 1, dtype=np.int64)
    np.cumsum(lens, out=ptr[1:])
    cols = rng.integers(0, n, int(ptr[-1]), dtype=np.int32)
    A = sp.csr_matrix((rng.standard_normal(int(ptr[-1])), cols, ptr.astype(np.int32)), shape=(m, n))
    A.sum_duplicates()
    ax = A @ rng.uniform(0.0, 5.0, n)
    p = pdhcg_amd.QPData(c=rng.standard_normal(n), A=A, con_lb=ax - rng.uniform(0, 1, m),
                         con_ub=ax + rng.uniform(0, 1, m), var_lb=np.zeros(n), var_ub=np.full(n, 5.0))
    if case["objective"] in ("diag", "lowrank"):
        p = replace(p, Q=sp.diags(rng.uniform(0.0, 1.0, n)).tocsr())
    if case["objective"] == "lowrank":
        p = replace(p, R=rng.standard_normal((k, n)) * np.sqrt(1.0 / n), D=rng.uniform(0.5, 2.0, k),
                    fmt={"R": "dense"})
    return p


def _svec_order(k):
    r, c = np.tril_indices(k)
    order = np.lexsort((r, c))  # lower triangle, column by column
    return r[order], c[order]


def _svec(S):
    r, c = _svec_order(S.shape[0])
    return S[r, c] * np.where(r == c, 1.0, np.sqrt(2.0))


def _smat(v, k):
    r, c = _svec_order(k)
    S = np.zeros((k, k))
    S[r, c] = S[c, r] = v * np.where(r == c, 1.0, np.sqrt(0.5))
    return S


def _conic(case, seed):
    layout = np.random.default_rng(1002)  # block sizes and order: the same for every seed
    rng = np.random.default_rng(seed)
    blocks = [("soc", int(k)) for k in layout.integers(1, 63, case["soc"])]
    blocks += [("rsoc", int(k)) for k in layout.integers(1, 31, case["rsoc"])]
    blocks += [("pow", 1)] * case["power"]
    blocks += [("psd", int(k)) for k in layout.integers(case["psd_low"], case["psd_high"] + 1, case["psd"])]
    cones, inner, pos = [], [], 0
    for b in layout.permutation(len(blocks)):
        kind, k = blocks[b]
        if kind == "soc":
            v = rng.standard_normal(k + 1)
            point = np.append(v, np.linalg.norm(v) + 1.0)
            cones.append((capi.CONE_STANDARD_SOC, pos, k))
        elif kind == "rsoc":
            v = rng.standard_normal(k)
            point = np.append(v, np.full(2, np.sqrt(0.5 * v @ v) + 1.0))
            cones.append((capi.CONE_ROTATED_SOC, pos, k))
        elif kind == "pow":
            point = np.array([1.0, 1.0, 0.3])
            cones.append((capi.CONE_POWER, pos, 1, float(rng.uniform(0.1, 0.9))))
        else:
            M = rng.standard_normal((k, k)) / np.sqrt(k)
            point = _svec(M @ M.T + np.eye(k))
            cones.append((capi.CONE_PSD, pos, k))
        inner.append(point)
        pos += point.size
    x = np.concatenate(inner)
    n = x.size
    m = max(2, n // 4)
    A = workloads.random_sparse(rng, m, n, min(4 * n, m * n))
    ax = A @ x
    kb = max(2, n // 30)
    B = sp.csr_matrix((rng.standard_normal(10 * kb), (np.repeat(np.arange(kb), 10), rng.integers(0, n, 10 * kb))),
                      shape=(kb, n))
    Q = (B.T @ B + sp.diags(rng.uniform(0.1, 1.0, n))).tocsr()
    Q.sort_indices()
    acones, rows = [], 0
    while rows < max(3, n // 6):
        k = int(layout.integers(1, 63))
        acones.append((capi.CONE_STANDARD_SOC, rows, k))
        rows += k + 2
    F = workloads.random_sparse(rng, rows, n, min(4 * n, rows * n))
    s0 = np.zeros(rows)
    for _, start, k in acones:
        s0[start + k + 1] = 2.0
    return pdhcg_amd.QPData(c=rng.standard_normal(n), A=A, Q=Q, con_lb=ax - rng.uniform(0, 1, m),
                            con_ub=ax + rng.uniform(0, 1, m), var_lb=np.full(n, -np.inf), var_ub=np.full(n, np.inf),
                            cones=cones, F=F, g=s0 - F @ x, affine_cones=acones)


def _psd_points(case, seed):
    """(cone specs, points): symmetric matrices with spectra on both sides of
    zero, each point a small step (0.1%) from the one before."""
    rng = np.random.default_rng(seed)
    # the same orders for every seed
    orders = np.random.default_rng(1002).integers(case["order_low"], case["order_high"] + 1, case["blocks"])
    specs, pos = [], 0
    for k in orders:
        specs.append((capi.CONE_PSD, pos, int(k)))
        pos += int(k) * (int(k) + 1) // 2
    first = rng.standard_normal(pos)
    steps = 1e-3 * rng.standard_normal((case["points"] - 1, pos))
    return specs, np.vstack([first, first + np.cumsum(steps, axis=0)])


def _problems(case, seed):
    if case["kind"] == "portfolio":
        layout = np.random.default_rng(1003)  # sizes: the same for every seed
        ns = layout.integers(case["n_low"], case["n_high"] + 1, case["count"])
        ks = layout.integers(case["k_low"], case["k_high"] + 1, case["count"])
        return [workloads.portfolio_tracking(int(n), int(k), seed=(seed, i)) for i, (n, k) in enumerate(zip(ns, ks))]
    family = workloads.ParametricFamily(n=case["n"], m=case["m"], nnz=case["nnz"], rank=case["rank"], seed=seed)
    return family.sample(case["count"], seed=seed + 1)[1]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "tiny":
        data = workloads.random_problem(case["objective"], seed=seed, n=case["n"], m=case["m"])
    elif kind == "sparse_q":
        data = workloads.config0(seed=seed, n=case["n"], m=case["m"])
    elif kind == "family":
        data = _family(case, seed)
    elif kind in ("portfolio", "parametric"):
        data = _problems(case, seed)
    elif kind == "conic":
        data = _conic(case, seed)
    elif kind == "psd":
        data = _psd_points(case, seed)
    else:
        rng = np.random.default_rng(seed)
        Z = rng.standard_normal((case["samples"], case["z"])).astype(np.float32)
        W = rng.standard_normal((case["z"], case["out"])) / np.sqrt(case["z"])
        T = np.clip(Z @ W + 0.1 * rng.standard_normal((case["samples"], case["out"])), -1.5, 1.5).astype(np.float32)
        data = (MLP(case["z"], case["hidden"], case["out"], seed=seed % (1 << 31)), Z, T)
    return case, data


def run(state):
    case, data = state
    kind = case["kind"]
    if kind == "psd":
        specs, points = data
        return {"projected": pdhcg_amd.project_cones_seq(specs, points)}
    if kind == "train":
        net, Z, T = data
        loss = net.train(Z, T, epochs=case["epochs"], batch=case["batch"], lr=1e-3, seed=1)
        return {"loss": loss, "weights": net.get_params(), "predicted": net.predict(Z[:256])}
    precision = _PRECISION[case["precision"]]
    if kind in ("portfolio", "parametric"):
        s = pdhcg_amd.solve_batch(data, precision=precision, eps=case["eps"])
        return {"x": np.concatenate([r.x for r in s]), "y": np.concatenate([r.y for r in s]),
                "reduced_cost": np.concatenate([r.reduced_cost for r in s]),
                "objective": np.array([r.pobj for r in s])}
    s = pdhcg_amd.solve(data, precision=precision, eps=case["eps"], iteration_limit=case["iterations"])
    out = {"x": s.x, "y": s.y}
    if kind == "family":  # elsewhere no bound is active and the reduced costs are the stopping residual
        out["reduced_cost"] = s.reduced_cost
    return out


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------

def _solve_work(n, m, nnz, q_bytes, q_flops, iterations):
    """Problem data in and solution out once, and two products with A and one
    with Q per outer iteration."""
    return {"bytes": 12.0 * nnz + q_bytes + 8.0 * (6 * n + 5 * m),
            "flops": float(iterations) * (4.0 * nnz + q_flops + 20.0 * (n + m))}


def work(case):
    kind = case["kind"]
    if kind == "tiny":
        n, m = case["n"], case["m"]
        return _solve_work(n, m, 0.2 * n * m, 8.0 * 6 * n, 4.0 * 6 * n, 200)
    if kind == "sparse_q":
        n, m = case["n"], case["m"]
        q = 0.1 * n * (0.01 * n) ** 2 + n
        return _solve_work(n, m, 0.005 * n * m, 12.0 * q, 2.0 * q, 200)
    if kind == "family":
        n, m, k = case["n"], case["m"], case["rank"]
        return _solve_work(n, m, case["nnz"], 8.0 * k * n, 4.0 * k * n, min(case["iterations"], 200))
    if kind == "portfolio":
        n, k = 0.5 * (case["n_low"] + case["n_high"]), 0.5 * (case["k_low"] + case["k_high"])
        one = _solve_work(n, k + 3, n * (k + 1), 8.0 * k * n, 4.0 * k * n, 200)
        return {key: case["count"] * v for key, v in one.items()}
    if kind == "parametric":
        n, m, k = case["n"], case["m"], case["rank"]
        one = _solve_work(n, m, case["nnz"], 8.0 * k * n, 4.0 * k * n, 200)
        return {key: case["count"] * v for key, v in one.items()}
    if kind == "conic":
        order = 0.5 * (case["psd_low"] + case["psd_high"])
        n = 33.5 * case["soc"] + 17.5 * case["rsoc"] + 3 * case["power"] + case["psd"] * 0.5 * order * (order + 1)
        w = _solve_work(n, 0.42 * n, 8.0 * n, 12.0 * 4 * n, 8.0 * n, case["iterations"])
        w["flops"] += case["iterations"] * case["psd"] * 9.0 * order ** 3
        return w
    if kind == "psd":
        lo, hi = case["order_low"], case["order_high"]
        mean = lambda f: sum(f(k) for k in range(lo, hi + 1)) / (hi - lo + 1)  # noqa: E731
        count = case["blocks"] * case["points"]
        # read and write each svec; a tridiagonal eigensolver with vectors takes about 9 k^3
        return {"bytes": 16.0 * count * mean(lambda k: 0.5 * k * (k + 1)), "flops": 9.0 * count * mean(lambda k: k ** 3)}
    z, h, out = case["z"], case["hidden"], case["out"]
    params = z * h + h * h + h * out
    steps = case["epochs"] * (case["samples"] // case["batch"])
    return {"bytes": 4.0 * case["samples"] * (z + out) + 30.0 * steps * params,
            "flops": 6.0 * steps * case["batch"] * params}


def tolerance(case):
    """About four times the largest difference seen between runs whose sums were
    formed in other orders (lanes per row, threads per problem) or whose
    objective was changed in its last bit, on the listed and on drawn cases.
    Most solves move by 1e-14; where one inner solve of the path ends a step
    earlier or later, by that inner solve's tolerance."""
    kind = case["kind"]
    if kind == "psd":
        return {"rel": 6e-13, "max": 1e-11}  # a tridiagonal eigensolver is 1.5e-13 from the Jacobi sweeps
    if kind == "train":
        return {"rel": 5e-3, "max": 0.05}  # BF16 operands: a rounding changes with its sum
    if kind == "conic":
        return {"rel": 0.014, "max": 0.3}  # stopped well before convergence
    if kind == "family" and case["objective"] == "lowrank":
        return {"rel": 2e-3, "max": 0.5}  # the large one: stopped well before convergence
    if case["precision"] == "mixed":
        return {"rel": 4e-4, "max": 0.06}
    return {"rel": 2.5e-5, "max": 1e-3}


def exact(case, seed):
    """The projections by numpy's eigen-decomposition.  A solve's result is
    where its stopping rule ends it, and the network's steps round to BF16:
    neither has a 64-bit value of its own."""
    if case["kind"] != "psd":
        return None
    specs, points = _psd_points(case, seed)
    out = np.empty_like(points)
    for _, start, k in specs:
        end = start + k * (k + 1) // 2
        for i in range(points.shape[0]):
            w, V = np.linalg.eigh(_smat(points[i, start:end], k))
            out[i, start:end] = _svec((V * np.maximum(w, 0.0)) @ V.T)
    return {"projected": out}
