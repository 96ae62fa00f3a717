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


PLANS = r"""
#include <cstdio>
#include <cstdlib>

#include "cles_internal.h"

using namespace cles;

// a diagonally dominant scheme of half-bandwidth q with nc closure rows
static cles_scheme_desc scheme(int q, int nc)
{
    cles_scheme_desc s{};
    s.q = q;
    s.M = 2;
    s.lhs[0] = 0.3;
    if (q == 2) s.lhs[1] = 0.05;
    s.coeffs[0] = 0.7;
    s.nclosure = nc;
    for (int j = 0; j < nc; j++) {
        s.closure_lhs[j][q] = 1.0;
        s.closure_rhs_len[j] = 1;
    }
    return s;
}

static HostPlan plan(int q, int nc, int dim, const int64_t n[3], int periodic, bool op)
{
    HostPlan hp;
    hp.dim = dim;
    const int64_t line = n[dim - 1], lines = n[0] * n[1] * n[2] / line;
    const int chunk = op ? operator_line_chunk(dim, line, lines, n[0], periodic)
                         : default_line_chunk(dim, line, lines, periodic);
    LineTables t;
    build_line_tables(t, scheme(q, nc), (int)line, periodic, 0.1, chunk, dim, nullptr, 0, 0, n[0]);
    hp.dev = t.dev;
    return hp;
}

// "p" dim nx ny nz periodic q nc -> capacity, whole chunks of an operator plan;
// "s" nx ny nz periodic_y 0 0 nf -> a solver's y and z gradients share a launch
int main(int argc, char **argv)
{
    for (int i = 1; i + 7 < argc; i += 8) {
        int v[8];
        for (int j = 1; j < 8; j++) v[j] = atoi(argv[i + j]);
        if (argv[i][0] == 'p') {
            const int64_t n[3] = {v[2], v[3], v[4]};
            const LineDev p = plan(v[6], v[7], v[1], n, v[5], true).dev;
            std::printf("%d %d\n", p.cap, p.extra == 0 && p.m == p.cap);
        } else {
            const int64_t n[3] = {v[1], v[2], v[3]};
            View3 w;
            for (int d = 0; d < 3; d++) w.n[d] = n[d];
            w.s[0] = 1;
            w.s[1] = n[0];
            w.s[2] = n[0] * n[1];
            std::printf("%d\n", pairable_lines(plan(1, 2, 2, n, v[4], false), plan(1, 2, 3, n, 1, false), w, v[7]));
        }
    }
}
"""


def test_shapes_of_the_gpu_tests(tmp_path):
    """The shapes of the GPU parity tests give the chunk capacities, whole and
    uneven, and the shared launches that those tests are there for."""
    import line_shapes as S
    from helpers import run_internal
    want, args = [], []
    for per in (0, 1):
        for q, nc in ((1, 2), (1, 4), (2, 3)):
            for dim in (2, 3):
                for lanes, outer, lines in ((49, 86, S.WIDE_LINES), (48, 512, S.WIDE_LINES), (49, 7, S.FEW_LINES)):
                    for line, cap, whole in lines:
                        args += ["p", dim, *S.wide(line, dim, lanes, outer), per, q, nc]
                        want.append(f"{cap} {int(whole)}")
            for line, cap, whole in S.X_LINES:
                args += ["p", 1, line, 5, 3, per, q, nc]
                want.append(f"{cap} {int(whole)}")
    for n, per, species, paired in S.PAIRS:
        args += ["s", *n, int(per), 0, 0, 4 if species == 1 else 6]
        want.append(str(int(paired)))
    got = run_internal(tmp_path, PLANS, [str(a) for a in args]).strip().split("\n")
    bad = [(args[8 * i:8 * i + 8], w, g) for i, (w, g) in enumerate(zip(want, got)) if w != g]
    assert len(got) == len(want) and not bad, bad
