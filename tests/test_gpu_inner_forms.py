"""The resident inner solve (dev_inner.hpp) at the edges of its forms: columns
per workgroup (512), workgroups launched plainly (8 x 512 columns) and
cooperatively, rows of R per wave (8, 16, 32, 56, 80, and the launched form
above), a dense D, and a sparse Q around its 64 variables per workgroup and
16-entry tasks.  Each solve against the oracle's: status, objective within
5 eps, KKT of the returned point."""
import numpy as np
import pytest
import scipy.sparse as sp

import pdhcg_amd
from pdhcg_amd import PRECISION_FP64, PRECISION_MIXED, QPData, capi, workloads
from tests.kkt import kkt
from tests.oracle_lib import oracle_solve

pytestmark = pytest.mark.gpu
EPS = 1e-5


def _rows(rng, n, m, **objective):
    A = workloads.random_sparse(rng, m, n, min(4 * m, m * n))
    ax = A @ rng.uniform(0.0, 5.0, n)
    return QPData(c=rng.standard_normal(n), A=A, con_lb=ax - rng.uniform(0, 1, m), con_ub=ax + rng.uniform(0, 1, m),
                  var_lb=np.zeros(n), var_ub=np.full(n, 5.0), **objective)


def _check(p, precision):
    g = pdhcg_amd.solve(p, precision=precision, eps=EPS, iteration_limit=20000)
    o = oracle_solve(p, eps=EPS, iteration_limit=20000)
    assert g.status == o.status == "OPTIMAL", (g.status, o.status)
    assert abs(g.pobj - o.pobj) <= 5 * EPS * (1 + abs(o.pobj)), (g.pobj, o.pobj)
    e = kkt(p, g.x, g.y)
    assert max(e["rel_primal"], e["rel_dual"], e["rel_gap"]) <= 10 * EPS, e


@pytest.mark.parametrize("precision", [PRECISION_FP64, PRECISION_MIXED])
@pytest.mark.parametrize("n,k", [(1, 1), (63, 8), (512, 9), (513, 16), (1100, 17), (600, 32), (520, 33), (512, 56),
                                 (700, 57), (513, 80), (300, 81), (4096, 3), (4097, 3), (8193, 10)])
def test_low_rank(n, k, precision):
    rng = np.random.default_rng(n + k)
    _check(_rows(rng, n, max(1, n // 4), Q=sp.diags(rng.uniform(0.05, 1.0, n)).tocsr(),
                 R=rng.standard_normal((k, n)) / np.sqrt(n), D=rng.uniform(0.5, 2.0, k), fmt={"R": "dense"}), precision)


@pytest.mark.parametrize("n", [40, 1025, 4200])
def test_low_rank_dense_d(n):
    rng = np.random.default_rng(n)
    M = rng.standard_normal((6, 6))
    _check(_rows(rng, n, n // 4, Q=sp.diags(rng.uniform(0.05, 1.0, n)).tocsr(),
                 R=rng.standard_normal((6, n)) / np.sqrt(n), D=M.T @ M + 0.2 * np.eye(6), fmt={"R": "dense"}),
           PRECISION_FP64)


@pytest.mark.parametrize("precision", [PRECISION_FP64, PRECISION_MIXED])
@pytest.mark.parametrize("n,per_row", [(2, 1), (63, 16), (64, 17), (65, 3), (150, 150), (1024, 5), (1025, 33),
                                       (3000, 4), (2100, 60), (400, 400)])
def test_sparse_q(n, per_row, precision):
    # a diagonally dominant symmetric Q of about per_row entries per row, one
    # row and column full; the last two sizes need more than 512 tasks per workgroup
    rng = np.random.default_rng(n + per_row)
    S = workloads.random_sparse(rng, n, n, max(1, min(n * n, n * per_row // 2)))
    S = sp.triu(S, 1).tolil()
    S[0, 1:] = 0.01
    S = (S + S.T).tocsr()
    Q = (S * (0.5 / max(1.0, abs(S).sum(axis=1).max())) + sp.diags(rng.uniform(0.6, 1.5, n))).tocsr()
    _check(_rows(rng, n, max(1, n // 4), Q=Q), precision)


# 65 workgroups (a lane sums more than one of a row's), all 256 of the chip, and
# the launched form above them
@pytest.mark.parametrize("n,k", [(33000, 80), (131072, 50), (131073, 50)])
def test_low_rank_large_grids(n, k):
    """The oracle's iterates after 16 iterations of three inner steps each.
    With c changed in its last bit the oracle moves by 2e-15 there; the sums of
    up to 131 073 terms in another order are off by at most 1e5 such bits."""
    rng = np.random.default_rng(n)
    p = _rows(rng, n, n // 4, Q=sp.diags(rng.uniform(0.8, 1.2, n)).tocsr(),
              R=rng.standard_normal((k, n)) / np.sqrt(n), D=rng.uniform(0.2, 0.5, k), fmt={"R": "dense"})
    kw = dict(eps=1e-14, iteration_limit=16, inner_solver_parameters=capi.inner_solver_parameters_t(3, 1e-3, 1e-9))
    o = oracle_solve(p, **kw)
    g = pdhcg_amd.solve(p, precision=PRECISION_FP64, **kw)
    assert (g.iterations, g.inner_iterations) == (o.iterations, o.inner_iterations)
    for a, b in ((g.x, o.x), (g.y, o.y)):
        error = float(np.linalg.norm(a - b) / (1.0 + np.linalg.norm(b)))
        assert error <= 1e-10


@pytest.mark.parametrize("n,k", [(33000, 80), (131072, 50)])
def test_low_rank_large_grids_mixed(n, k):
    rng = np.random.default_rng(n)
    p = _rows(rng, n, n // 4, Q=sp.diags(rng.uniform(0.8, 1.2, n)).tocsr(),
              R=rng.standard_normal((k, n)) / np.sqrt(n), D=rng.uniform(0.2, 0.5, k), fmt={"R": "dense"})
    g = pdhcg_amd.solve(p, precision=PRECISION_MIXED, eps=1e-4, iteration_limit=20000)
    assert g.status == "OPTIMAL"
    e = kkt(p, g.x, g.y)
    assert max(e["rel_primal"], e["rel_dual"], e["rel_gap"]) <= 1e-3, e
