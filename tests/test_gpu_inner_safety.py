"""The resident inner solve (dev_inner.hpp) where nothing but its own rules
keeps workgroups from each other's data."""
import numpy as np
import pytest
import scipy.sparse as sp

import pdhcg_amd
from pdhcg_amd import PRECISION_FP64, QPData, capi, workloads
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
