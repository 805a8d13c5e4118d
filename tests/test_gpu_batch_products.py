"""The batched solve's products at the edges of their forms, against the
oracle's solve of the same problem: odd sizes and padding, vectors with and
without room in LDS, all, some and none of R's rows resident, chunks of the
sparse product (4096 entries) with rows that are empty, that span several
chunks and that end on a boundary, and A on both sides of the dense rule."""
import numpy as np
import pytest
import scipy.sparse as sp

import pdhcg_amd
from pdhcg_amd import PRECISION_FP64, PRECISION_MIXED, QPData
from tests.oracle_lib import oracle_solve

pytestmark = pytest.mark.gpu
EPS = 1e-5


def _problem(n, m, k, row_lengths, seed=0):
    rng = np.random.default_rng((n, m, k, seed))
    rows = [np.sort(rng.choice(n, min(int(q), n), replace=False)) for q in row_lengths]
    ptr = np.concatenate([[0], np.cumsum([r.size for r in rows])])
    cols = np.concatenate(rows) if ptr[-1] else np.zeros(0, dtype=int)
    vals = rng.standard_normal(int(ptr[-1])) / np.sqrt(np.maximum(1, np.repeat(np.diff(ptr), np.diff(ptr))))
    A = sp.csr_matrix((vals, cols, ptr), shape=(m, n))
    ax = A @ rng.uniform(0.0, 5.0, n)
    data = dict(c=rng.standard_normal(n), A=A, con_lb=ax - rng.uniform(0.1, 1, m), con_ub=ax + rng.uniform(0.1, 1, m),
                var_lb=np.zeros(n), var_ub=np.full(n, 5.0), Q=sp.diags(rng.uniform(0.2, 1.0, n)).tocsr())
    if k:
        data.update(R=rng.standard_normal((k, n)) / np.sqrt(n), D=rng.uniform(0.5, 2.0, k), fmt={"R": "dense"})
    return QPData(**data)


def _problems():
    out = [_problem(n, m, k, [max(1, n // 6)] * m) for n, m, k in
           [(1, 1, 1), (2, 2, 1), (3, 2, 2), (5, 3, 4), (129, 20, 9), (514, 60, 17), (1023, 50, 40)]]
    out.append(_problem(40, 12, 3, [40] * 10 + [0, 0]))            # dense A
    out.append(_problem(600, 256, 5, [300] * 256))                 # dense, as many rows as its limit
    out.append(_problem(300, 257, 5, [150] * 257))                 # one row too many for the dense form
    out.append(_problem(700, 30, 2, [0, 700, 0, 5, 3] + [230] * 25))
    out.append(_problem(9000, 9, 3, [9000, 0, 4096, 1, 4095, 8192, 2, 0, 33]))   # rows across chunks
    out.append(_problem(4096, 4, 0, [1024] * 4))                   # rows that end on the boundary
    out.append(_problem(2600, 400, 30, [10] * 399 + [2600]))
    out.append(_problem(50, 1500, 2, [3] * 1500))                  # more rows than variables
    return out


@pytest.mark.parametrize("precision", [PRECISION_FP64, PRECISION_MIXED])
@pytest.mark.parametrize("threads", ["256", "512"])
def test_products_match_oracle(threads, precision, monkeypatch):
    monkeypatch.setenv("PDHCG_BATCH_THREADS", threads)
    problems = _problems()
    sols = pdhcg_amd.solve_batch(problems, precision=precision, eps=EPS, iteration_limit=20000, time_limit=60.0)
    for p, g in zip(problems, sols):
        o = oracle_solve(p, eps=EPS, iteration_limit=20000)
        assert g.status == o.status == "OPTIMAL", (p.n, p.A.shape, g.status, o.status)
        assert abs(g.pobj - o.pobj) <= 5 * EPS * (1 + abs(o.pobj)), (p.n, p.A.shape, g.pobj, o.pobj)
        # strongly convex: the points agree as well
        assert np.linalg.norm(g.x - o.x) <= 1e-3 * (1 + np.linalg.norm(o.x)), (p.n, p.A.shape)
