"""The resident inner solve (dev_inner.hpp) where nothing but its own rules
keeps workgroups from each other's data."""
from threading import Barrier, Thread

import numpy as np
import pytest
import scipy.sparse as sp

import pdhcg_amd
from pdhcg_amd import PRECISION_FP64, PRECISION_MIXED, QPData, capi, workloads
from tests.kkt import kkt
from tests.oracle_lib import oracle_solve

pytestmark = pytest.mark.gpu


def _sparse_q(n, smallest, seed):
    """Box-constrained rows with a sparse symmetric Q whose diagonal starts at
    `smallest`: diagonally dominant elsewhere."""
    rng = np.random.default_rng(seed)
    m = max(1, n // 4)
    A = workloads.random_sparse(rng, m, n, 4 * m)
    ax = A @ rng.uniform(0.0, 5.0, n)
    S = workloads.random_sparse(rng, n, n, 6 * n)
    S = (S + S.T).tocsr()
    diag = rng.uniform(0.6, 1.5, n)
    diag[rng.permutation(n)[: max(1, n // 10)]] = smallest
    Q = (S * (0.05 / abs(S).sum(axis=1).max()) + sp.diags(diag)).tocsr()
    Q.sort_indices()
    return QPData(c=rng.standard_normal(n), A=A, Q=Q, con_lb=ax - rng.uniform(0, 1, m),
                  con_ub=ax + rng.uniform(0, 1, m), var_lb=np.zeros(n), var_ub=np.full(n, 5.0))


@pytest.mark.parametrize("n", [65, 300, 1025, 3000])  # 2, 5, 16 and 16 workgroups
@pytest.mark.parametrize("case", ["indefinite", "limit"])
def test_one_inner_step_is_the_oracles(n, case):
    """One gradient step per inner solve, so no exchange between the
    workgroups: an indefinite Q allows only one, and so may the caller.  The
    iterations are then the oracle's apart from the order of the sums.  What
    that may give: with c changed in its last bit the oracle itself moves by at
    most 5e-12 in 20 iterations of these indefinite problems (by 1e-2 in 200:
    they are not non-expansive) and by 4e-16 in 200 of the convex ones; a sum of
    tens of terms is off by tens of such bits, so 1e-7 is ample, while one stale
    column of x is an error of the size of an iteration's step, 1e-3 and more."""
    count = 20 if case == "indefinite" else 200
    p = _sparse_q(n, -0.5 if case == "indefinite" else 0.3, n)
    kw = dict(eps=1e-14, iteration_limit=count)
    if case == "limit":
        kw["inner_solver_parameters"] = capi.inner_solver_parameters_t(1, 1e-3, 1e-9)
    o = oracle_solve(p, **kw)
    g = pdhcg_amd.solve(p, precision=PRECISION_FP64, **kw)
    assert g.iterations == o.iterations == o.inner_iterations == count
    assert g.inner_iterations == o.inner_iterations
    for a, b in ((g.x, o.x), (g.y, o.y)):
        error = float(np.linalg.norm(a - b) / (1.0 + np.linalg.norm(b)))
        assert error <= 1e-7


def _low_rank(n, k, seed, affine=False):
    rng = np.random.default_rng(seed)
    m = max(1, n // 4)
    A = workloads.random_sparse(rng, m, n, 4 * m)
    x = rng.uniform(0.0, 5.0, n)
    ax = A @ x
    more = {}
    if affine:
        F = workloads.random_sparse(rng, 40, n, 160)
        g = -F @ x
        g[[19, 39]] += 2.0
        more = dict(F=F, g=g, affine_cones=[(capi.CONE_STANDARD_SOC, 0, 18), (capi.CONE_STANDARD_SOC, 20, 18)])
    return QPData(c=rng.standard_normal(n), A=A, Q=sp.diags(rng.uniform(0.8, 1.2, n)).tocsr(),
                  R=rng.standard_normal((k, n)) / np.sqrt(n), D=rng.uniform(0.2, 0.5, k), fmt={"R": "dense"},
                  con_lb=ax - rng.uniform(0, 1, m), con_ub=ax + rng.uniform(0, 1, m), var_lb=np.zeros(n),
                  var_ub=np.full(n, 5.0), **more)


_FORMS = {"rank 12, 2 workgroups": lambda: _low_rank(600, 12, 1), "rank 5, 12 workgroups": lambda: _low_rank(6000, 5, 2),
          "rank 3, 19 workgroups": lambda: _low_rank(9300, 3, 6),
          "affine cones": lambda: _low_rank(700, 9, 4, affine=True), "sparse, 16 workgroups": lambda: _sparse_q(1500, 0.3, 5)}


@pytest.mark.parametrize("form", list(_FORMS))
def test_after_a_wait_that_gives_up_the_solve_goes_on(form, monkeypatch, capfd):
    """An inner solve whose last workgroup gives up at its first wait is
    repeated launch by launch from the state before it: the first one, ones
    between two reads of the scalars, one in a pass with a restart (200, 400)
    and the last one before the iteration limit.  With three inner steps the
    iterates do not depend on a tolerance, and the oracle with c changed in its
    last bit moves by at most 1e-14 on these problems: 1e-9 for the other order
    of the sums."""
    p = _FORMS[form]()
    kw = dict(eps=1e-14, iteration_limit=410, inner_solver_parameters=capi.inner_solver_parameters_t(3, 1e-3, 1e-9))
    o = oracle_solve(p, **kw)
    for launch in (0, 1, 2, 57, 200, 201, 399, 400, 410):
        monkeypatch.setenv("PDHCG_INNER_GIVE_UP", str(launch))
        g = pdhcg_amd.solve(p, precision=PRECISION_FP64, verbose=1, **kw)
        note = capfd.readouterr().err
        assert ("[inner]" in note) == (launch > 0)
        assert launch == 0 or f"launch by launch from iteration {launch - 1}\n" in note
        assert (g.iterations, g.inner_iterations, g.status) == (o.iterations, o.inner_iterations, o.status), launch
        for a, b in ((g.x, o.x), (g.y, o.y)):
            error = float(np.linalg.norm(a - b) / (1.0 + np.linalg.norm(b)))
            assert error <= 1e-9, launch


@pytest.mark.parametrize("precision", [PRECISION_FP64, PRECISION_MIXED])
@pytest.mark.parametrize("form", ["rank 5, 12 workgroups", "sparse, 16 workgroups"])
def test_whole_solve_with_a_wait_that_gives_up(form, precision, monkeypatch):
    p = _FORMS[form]()
    o = oracle_solve(p, eps=1e-5, iteration_limit=20000)
    monkeypatch.setenv("PDHCG_INNER_GIVE_UP", "33")
    g = pdhcg_amd.solve(p, precision=precision, eps=1e-5, iteration_limit=20000)
    assert g.status == o.status == "OPTIMAL"
    assert abs(g.pobj - o.pobj) <= 5e-5 * (1 + abs(o.pobj))
    e = kkt(p, g.x, g.y)
    assert max(e["rel_primal"], e["rel_dual"], e["rel_gap"]) <= 1e-4, e


def test_solves_beside_each_other_wait_for_room(monkeypatch, capfd):
    """Three solvers stepped from three threads at once, whose resident
    workgroups (200, 144 and 16 compute units) do not fit the chip together:
    none of them gives up a wait, and each goes the way it goes alone, bit for
    bit."""
    monkeypatch.setenv("PDHCG_SPMV_SHIFT", "0")  # otherwise picked by timing
    problems = [_low_rank(100000, 6, 11), _low_rank(70000, 20, 12), _sparse_q(1500, 0.3, 13)]
    count = [1500, 1500, 3000]

    def stepper(i):
        return pdhcg_amd.Stepper(problems[i], eps=1e-15, iteration_limit=10 ** 6, verbose=1)

    alone = []
    for i in range(3):
        s = stepper(i)
        s.run(count[i])
        alone.append(s.result())
        s.close()
    steppers = [stepper(i) for i in range(3)]
    gate = Barrier(3)

    def step(i):
        gate.wait()
        for _ in range(10):
            steppers[i].run(count[i] // 10)

    threads = [Thread(target=step, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for a, s in zip(alone, steppers):
        b = s.result()
        s.close()
        assert (a.iterations, a.inner_iterations) == (b.iterations, b.inner_iterations)
        assert a.status == "UNSPECIFIED"  # all the passes asked for
        assert np.array_equal(a.x, b.x) and np.array_equal(a.y, b.y)
    assert "[inner]" not in capfd.readouterr().err


def test_solvers_of_one_thread_in_turn(monkeypatch):
    """Two solvers alive at once, each of more than half the chip, stepped in
    turn: each goes the way it goes alone."""
    monkeypatch.setenv("PDHCG_SPMV_SHIFT", "0")
    problems = [_low_rank(80000, 4, 21), _low_rank(90000, 4, 22)]

    def finish(s):
        r = s.result()
        s.close()
        return r

    alone = []
    for p in problems:
        s = pdhcg_amd.Stepper(p)
        for _ in range(6):
            s.run(7)
        alone.append(finish(s))
    both = [pdhcg_amd.Stepper(p) for p in problems]
    for _ in range(6):
        for s in both:
            s.run(7)
    for a, s in zip(alone, both):
        b = finish(s)
        assert a.iterations == b.iterations == 42
        assert np.array_equal(a.x, b.x) and np.array_equal(a.y, b.y)
