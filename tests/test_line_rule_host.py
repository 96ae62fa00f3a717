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


PROGRAM = r"""
#include <cstdio>
#include <cstdlib>

#include "cles_internal.h"

// dim nx ny nz periodic -> chunk length of an operator plan
int main(int argc, char **argv)
{
    for (int i = 1; i + 4 < argc; i += 5) {
        const int dim = atoi(argv[i]), periodic = atoi(argv[i + 4]);
        const int64_t n[3] = {atoi(argv[i + 1]), atoi(argv[i + 2]), atoi(argv[i + 3])};
        const int64_t line = n[dim - 1];
        std::printf("%d\n", cles::operator_line_chunk(dim, line, n[0] * n[1] * n[2] / line, n[0], periodic != 0));
    }
}
"""


def test_operator_rule(tmp_path):
    """Chunk lengths of operator plans: lines of up to 256 points within eight
    chunks where the launch is wide, the solver's rule otherwise."""
    from helpers import run_internal
    cases = [((2, 144, 144, 144, 1), 32), ((3, 128, 128, 128, 0), 16), ((2, 129, 129, 129, 1), 32),
             ((2, 64, 20, 64, 1), 16), ((3, 47, 100, 144, 1), 16), ((3, 47, 80, 144, 1), 8), ((2, 64, 300, 63, 1), 8), ((2, 64, 300, 64, 1), 32),
             ((2, 33, 29, 31, 0), 8), ((2, 100, 2000, 1, 1), 32), ((1, 256, 256, 1, 1), 16), ((1, 256, 256, 1, 0), 8),
             ((1, 1000, 20, 20, 1), 16), ((1, 500, 20, 20, 1), 8)]
    out = run_internal(tmp_path, PROGRAM, [str(v) for c, _ in cases for v in c])
    assert [int(x) for x in out.split()] == [w for _, w in cases]
