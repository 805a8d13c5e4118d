"""PSD projections swept by position (psd_positions_kernel, orders up to 128):
the smallest orders, both sides of a wave of blocks (orders 20 to 24: 55 to 78
blocks of 64 lanes), of the waves that take part (63 to 66) and of the limit
(127 to 129, the last one by index), at entries near 1, 1e-130 and 1e130 (the
rotation scales its inputs by powers of two), cold and warm, against the
oracle's projection."""
import numpy as np
import pytest

import pdhcg_amd
from pdhcg_amd import capi
from tests.test_oracle_cones import project as orc_project

pytestmark = pytest.mark.gpu
ORDERS = (1, 2, 3, 4, 5, 20, 21, 22, 23, 24, 63, 64, 65, 66, 127, 128, 129)


@pytest.mark.parametrize("scale", [1e-130, 1.0, 1e130])
def test_orders_and_scales_match_oracle(scale):
    rng = np.random.default_rng(31)
    specs, pos = [], 0
    for k in ORDERS:
        specs.append((capi.CONE_PSD, pos, k))
        pos += k * (k + 1) // 2
    x = rng.standard_normal(pos)
    points = np.stack([x, x + 1e-3 * rng.standard_normal(pos), -x])
    got = pdhcg_amd.project_cones_seq(specs, scale * points, np.ones(pos)) / scale
    for xs, out in zip(points, got):
        for _, st, k in specs:
            s = slice(st, st + k * (k + 1) // 2)
            want = orc_project(capi.CONE_PSD, xs[s].copy(), k)
            # the bound of the other PSD tests; the scale itself rounds 1 ulp
            assert np.max(np.abs(out[s] - want)) <= 1e-12 * (1.0 + np.max(np.abs(xs[s]))), k
