"""Second-order cone projections with a group of lanes per block
(soc_project_group): block sizes on both sides of each lane class (4, 8, 16,
32, 64 lanes), all classes in one call, against the oracle's per-block
routine at 1e-12; and the batched solve with few cones (groups) and many
(one thread per cone)."""
import numpy as np
import pytest
import scipy.sparse as sp

import pdhcg_amd
from pdhcg_amd import QPData, capi, workloads
from tests.oracle_lib import oracle_solve
from tests.test_oracle_cones import project as orc_project

pytestmark = pytest.mark.gpu
SOC, RSOC = capi.CONE_STANDARD_SOC, capi.CONE_ROTATED_SOC
SIZES = (1, 2, 4, 5, 8, 9, 16, 17, 32, 33, 63, 64)


@pytest.mark.parametrize("t", [SOC, RSOC])
@pytest.mark.parametrize("uniform", [True, False])
@pytest.mark.parametrize("copies", [1, 9])
def test_lane_classes_match_oracle(t, uniform, copies):
    rng = np.random.default_rng(17 + copies)
    specs, pos = [], 0
    for vd in rng.permutation(np.repeat(SIZES, copies)):
        specs.append((t, pos, int(vd)))
        pos += int(vd) + 3  # a free slot between blocks
    d = np.ones(pos) if uniform else rng.uniform(0.2, 5.0, pos)
    x = rng.standard_normal(pos)
    for i, (_, st, vd) in enumerate(specs):  # outside, inside and in the polar cone
        x[st + vd + 1] += (0.0, 3.0 * vd, -3.0 * vd)[i % 3]
        if t == RSOC:
            x[st + vd] += (0.0, 3.0 * vd, -3.0 * vd)[i % 3]
    got = pdhcg_amd.project_cones(specs, x, d)
    used = np.zeros(pos, dtype=bool)
    for _, st, vd in specs:
        s = slice(st, st + vd + 2)
        used[s] = True
        want = orc_project(t, x[s], vd, d[s])
        assert np.max(np.abs(got[s] - want)) <= 1e-12 * (1 + np.max(np.abs(x[s]))), (vd, got[s], want)
    assert np.array_equal(got[~used], x[~used])


@pytest.mark.parametrize("count,vdim", [(3, 2), (3, 12), (2, 40), (700, 1), (130, 10)])
def test_batch_cone_forms_match_oracle(count, vdim):
    # count * lanes above 8 * 256 (700 x 4, 130 x 16): one thread per cone
    rng = np.random.default_rng(count)
    n, rows = 60, count * (vdim + 2)
    F = workloads.random_sparse(rng, rows, n, 3 * rows)
    x0 = rng.uniform(-1, 1, n)
    s0 = np.zeros(rows)
    s0[vdim + 1::vdim + 2] = 2.0
    p = QPData(c=rng.standard_normal(n), Q=sp.diags(rng.uniform(0.5, 2.0, n)).tocsr(), var_lb=np.full(n, -10.0),
               var_ub=np.full(n, 10.0), F=F, g=s0 - F @ x0,
               affine_cones=[(SOC, i * (vdim + 2), vdim) for i in range(count)])
    g = pdhcg_amd.solve_batch([p], eps=1e-5, iteration_limit=100000, time_limit=60.0)[0]
    o = oracle_solve(p, eps=1e-5, iteration_limit=100000)
    assert g.status == o.status == "OPTIMAL", (g.status, o.status)
    assert abs(g.pobj - o.pobj) <= 5e-5 * (1 + abs(o.pobj)), (g.pobj, o.pobj)
