"""Chunk lengths of shapes the line-tile table does not hold, between the
131072-thread lengths and the shortest (no GPU is touched)."""
import numpy as np
import pytest


@pytest.mark.parametrize("n,periodic,want", [
    ((120, 97, 81), True, (16, 16, 16)),     # x: 8 x 15 points even, 16 x 7.5 not
    ((120, 97, 81), False, (8, 16, 16)),     # closed lines have no even split to gain from
    ((96, 96, 96), True, (8, 16, 16)),       # even either way
    ((75, 83, 70), True, (8, 16, 16)),
    ((64, 64, 64), True, (8, 8, 8)),         # 16384 threads at 16
    ((400, 200, 1), True, (8, 8, 0)),        # 400 lines
    ((190, 160, 170), True, (16, 32, 32)),
    ((8, 16384, 1), True, (8, 32, 0)),       # at most 512 chunks per line
])
def test_rule_between(n, periodic, want):
    import compactles_hip as ch
    ch.tune.clear()
    bc = ch.PeriodicBC() if periodic else ch.SlipWallBC()
    prob = ch.Problem(domain=((0.0, 2 * np.pi),) * 3, bcs=((bc, bc),) * 3, ic=lambda X, Y, Z: None)
    assert ch.tune.lookup(ch.SolverSpec(prob, ch.Numerics(n_global=n)))[0] == want
