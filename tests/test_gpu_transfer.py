"""Host transfers of the state: every interior value arrives and every halo
value of the caller's array is left alone, for states moved in one piece, in
several chunks and by several threads, and for batch instances."""
import numpy as np
import pytest

import cases

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    import compactles_hip as ch
    return ch.Context(0)


@pytest.mark.parametrize("n", [(9, 1, 1), (17, 12, 1), (33, 29, 31), (64, 64, 64), (129, 130, 65)])
def test_state_round_trip(ctx, n):
    import compactles_hip as ch
    prob = ch.Problem(domain=((0.0, 1.0),) * 3, bcs=((ch.PeriodicBC(), ch.PeriodicBC()),) * 3,
                      ic=lambda X, Y, Z: None)
    s = ch.Solver(ctx, prob, ch.Numerics(n_global=n))
    rng = np.random.default_rng(3)
    for _ in range(2):   # the second pass reuses the staging buffers
        Q = np.asfortranarray(rng.standard_normal(s.padded + (s.n_cons,)))
        s.upload(Q)
        R = np.full(Q.shape, 7.0, order="F")
        s.download(R)
        sl = tuple(slice(s.halo[d], s.halo[d] + n[d]) for d in range(3))
        assert np.array_equal(R[sl], Q[sl])
        halo = np.ones(Q.shape, dtype=bool)
        halo[sl] = False
        assert np.all(R[halo] == 7.0)
        assert np.array_equal(s.field("Q[2]"), Q[sl + (1,)])


def test_batch_round_trip(ctx):
    specs = cases.tube_specs(5, nmin=128, nmax=2048)
    b = cases.tube_batch(ctx, specs)
    rng = np.random.default_rng(4)
    want = []
    for i, sp in enumerate(specs):
        Q = np.asfortranarray(rng.standard_normal((sp["n"] + 8, 1, 1, 6)))
        b.upload(i, Q)
        want.append(Q)
    for i in (3, 0, 4, 2, 1):
        got = b.download(i)
        assert np.array_equal(got[4:-4], want[i][4:-4])
        assert np.all(got[:4] == 0) and np.all(got[-4:] == 0)
