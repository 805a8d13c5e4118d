"""Length of the FP32 sums in the mixed batch's products: R'u and A'y of a dense
A add a column in four sums, R x a lane's columns of a row in four.

Each problem holds one sum of 1 and many t = 0.99 * 2^-24, exactly what FP32
drops when it adds t to 1, so a sum of k terms that is kept as four loses about
k / 4 of them (k / 4 + 4 times 2^-24 bounds it, roundings included) and one
running sum all of them.  The solve is one unscaled FP32 step, whose point is
returned: x1 = -a (Q x0) or a (A'y0), with a in another column."""
import numpy as np
import pytest
import scipy.sparse as sp

import pdhcg_amd
from pdhcg_amd import PRECISION_MIXED, QPData, capi

pytestmark = pytest.mark.gpu
U = 2.0 ** -24
T = 0.99 * U
ONE_STEP = dict(eps=1e-14, iteration_limit=1, l_inf_ruiz_iterations=0, curtis_reid_iterations=0,
                has_pock_chambolle_alpha=False, bound_objective_rescaling=False, diag_jacobi_precond=False,
                termination_evaluation_frequency=1, inner_solver_parameters=capi.inner_solver_parameters_t(1, 1e-3, 1e-9))


def _step(p):
    s = pdhcg_amd.solve_batch([p], precision=PRECISION_MIXED, **ONE_STEP)[0]
    assert s.iterations == 1
    return s.x


def _free(n, x0, **data):
    return QPData(c=np.zeros(n), var_lb=np.full(n, -1e6), var_ub=np.full(n, 1e6), primal_start=x0, **data)


def _no_rows(n):
    return dict(A=sp.csr_matrix((1, n)), con_lb=np.array([-np.inf]), con_ub=np.array([np.inf]))


@pytest.mark.parametrize("n", [64, 2048])  # all rows of R in LDS, few of them
@pytest.mark.parametrize("k", [41, 256])
def test_low_rank_columns(n, k):
    R = np.zeros((k, n))
    R[:, 0] = 1.0          # R x0 = 1 in every row
    R[0, 1], R[1:, 1] = 1.0, T
    R[0, 2] = 1.0
    x0 = np.zeros(n)
    x0[0] = 1.0
    x = _step(_free(n, x0, R=R, fmt={"R": "dense"}, **_no_rows(n)))
    assert x[2] != 0.0
    assert abs(x[1] / x[2] - (1.0 + (k - 1) * T)) <= (k / 4 + 4) * U


@pytest.mark.parametrize("n", [8192, 32768])  # x copied to LDS, read where it is
def test_low_rank_rows(n):
    R = np.zeros((2, n))
    lane = np.arange(0, n, 128)  # what the first element of a lane's pairs meets
    R[0, lane] = T
    R[0, 0] = R[0, 5] = 1.0
    R[1, 0] = R[1, 6] = 1.0
    x0 = np.zeros(n)
    x0[lane] = 1.0
    x = _step(_free(n, x0, R=R, fmt={"R": "dense"}, **_no_rows(n)))
    assert x[6] != 0.0
    assert abs(x[5] / x[6] - (1.0 + (lane.size - 1) * T)) <= (lane.size / 2 + 4) * U


@pytest.mark.parametrize("m", [90, 256])
def test_dense_a_columns(m):
    n = 64
    A = np.ones((m, n))
    A[1:, 1] = T
    A[1:, 2] = 0.0
    x = _step(_free(n, np.zeros(n), A=sp.csr_matrix(A), con_lb=np.full(m, -1.0), con_ub=np.full(m, 1.0),
                    dual_start=np.ones(m)))
    assert x[2] != 0.0
    assert abs(x[1] / x[2] - (1.0 + (m - 1) * T)) <= (m / 4 + 4) * U
