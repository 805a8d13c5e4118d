"""The round-robin schedule of the PSD projection by position
(psd_positions_kernel in pdhcg_amd/csrc/dev_cones.hpp, orders 2 to 128).

Position L holds an up and a down element, which a round rotates against each
other.  After each round the up elements move one position right, the down
elements one position left, position 0 keeps its up element, position 1 takes
position 0's down element and the last position's up element becomes its down
element (a single pair stays in place); the blocks of the matrix and the rows of
V' are written to where their elements stand next.  This restates those moves
and checks the properties the Jacobi sweep relies on: every round pairs all kp
elements disjointly, every pair meets exactly once in kp - 1 rounds, and the
elements are back at their places after a sweep.  (The rotations themselves are
checked by the GPU PSD tests.)
"""
import itertools


def _move(up, dn):
    np_ = len(up)
    nu = [up[0] if L == 0 else (dn[0] if L == 1 else up[L - 1]) for L in range(np_)]
    nd = [((up[L] if np_ > 1 else dn[L]) if L == np_ - 1 else dn[L + 1]) for L in range(np_)]
    return nu, nd


def test_every_pair_once_per_sweep_and_positions_restored():
    for kp in range(2, 130, 2):
        np_ = kp // 2
        up = [2 * L for L in range(np_)]
        dn = [2 * L + 1 for L in range(np_)]
        seen = set()
        for _ in range(kp - 1):
            assert sorted(up + dn) == list(range(kp)), kp  # a partition of the indices
            for a, b in zip(up, dn):
                pair = (min(a, b), max(a, b))
                assert pair not in seen, (kp, pair)
                seen.add(pair)
            up, dn = _move(up, dn)
        assert seen == set(itertools.combinations(range(kp), 2)), kp
        assert up == [2 * L for L in range(np_)] and dn == [2 * L + 1 for L in range(np_)], kp
