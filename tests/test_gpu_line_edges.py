"""GPU parity of the line operators at the sizes where a kernel or a plan
changes form: truncated reductions, chunk capacities, uneven chunks, ragged
lane counts.  Against the oracle's apply_along! on the same seeded inputs, with
the operators' bar: FP64 normwise <= 1e-12, FP32 <= 2e-5."""
import numpy as np
import pytest

import helpers as Hh
import line_shapes as S
from test_gpu_operators import _gpu_apply, _oracle_apply, ctx  # noqa: F401
from test_gpu_solver import _compare_rhs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["lele_d1_6", "lele_d1_10", "compact_filter"])
@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("dim,n", [(1, (1000, 5, 3)), (2, (6, 900, 2)), (3, (7, 2, 520))])
def test_truncated_reduction(ctx, name, periodic, dim, n):  # noqa: F811
    """Lines long enough that the reduction stops before log2(chunks) steps:
    a random line, and one spike of 1e8 over a random line (the interface values
    then span eight decades; the bar is relative to the largest value)."""
    f = Hh.random_field(n, seed=21)
    g = f.copy()
    at = [0, 0, 0]
    at[dim - 1] = n[dim - 1] // 3
    g[tuple(at)] = 1e8
    for a in (f, g):
        ref = _oracle_apply(name, dim, n, periodic, 0.01, a)
        assert Hh.relerr(_gpu_apply(ctx, name, dim, n, periodic, 0.01, a), ref) <= 1e-12


@pytest.mark.parametrize("dtype,bar", [(np.float64, 1e-12), (np.float32, 2e-5)])
@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("lanes,line,outer", [(48, 16, 3), (64, 9, 2), (65, 33, 2), (127, 64, 2), (130, 20, 1),
                                              (50, 33, 512), (128, 64, 513), (130, 11, 300)])
def test_wave_uniform_yz(ctx, dtype, bar, periodic, lanes, line, outer):  # noqa: F811
    """The one-chunk-per-wave y / z sweeps: whole and short chunks of every
    capacity, partial lane blocks, and (FP32, even rows, >= 512 blocks) two
    lines per lane; C6, C10 and the filter."""
    for name in ("lele_d1_6", "lele_d1_10", "compact_filter"):
        for dim in (2, 3):
            n = (lanes, line, outer) if dim == 2 else (lanes, outer, line)
            f = Hh.random_field(n, seed=31)
            if dtype == np.float32:
                f = f.astype(np.float32).astype(np.float64)
            ref = _oracle_apply(name, dim, n, periodic, 0.1, f)
            got = _gpu_apply(ctx, name, dim, n, periodic, 0.1, f, dtype=dtype)
            assert Hh.relerr(got, ref) <= bar, (name, dim)


@pytest.mark.parametrize("dtype,bar", [(np.float64, 1e-12), (np.float32, 2e-5)])
@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("line", [9, 16, 17, 24, 32, 33, 40, 63, 64, 65, 100, 128, 129, 250, 256, 257, 384, 512, 1000,
                                  1024])
def test_wave_local_x(ctx, dtype, bar, periodic, line):  # noqa: F811
    """The wave-local x sweep: 8 to 64 lanes per line, whole and short chunks of
    both capacities, line counts that leave waves partly empty, padded and
    unpadded rows; every scheme."""
    for name in ("lele_d1_6", "pade_d1_4", "lele_d1_10", "compact_filter"):
        for ny, nz, padded in ((5, 3, True), (1, 1, False), (3, 7, False), (67, 2, True)):
            n = (line, ny, nz)
            f = Hh.random_field(n, seed=41)
            if dtype == np.float32:
                f = f.astype(np.float32).astype(np.float64)
            ref = _oracle_apply(name, 1, n, periodic, 0.1, f)
            got = _gpu_apply(ctx, name, 1, n, periodic, 0.1, f, dtype=dtype, padded=padded)
            assert Hh.relerr(got, ref) <= bar, (name, n)


@pytest.mark.parametrize("dtype,bar", [(np.float64, 1e-12), (np.float32, 2e-5)])
@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("line", [1025, 1100, 2048, 4000])
def test_block_x(ctx, dtype, bar, periodic, line):  # noqa: F811
    """The block-wide x sweep: lines of more than 64 chunks, whole and uneven
    chunks, blocks with missing lines, padded and unpadded rows."""
    for name in ("lele_d1_6", "lele_d1_10", "compact_filter"):
        for ny, nz, padded in ((5, 3, True), (1, 1, False), (3, 1, False)):
            n = (line, ny, nz)
            f = Hh.random_field(n, seed=51)
            if dtype == np.float32:
                f = f.astype(np.float32).astype(np.float64)
            ref = _oracle_apply(name, 1, n, periodic, 0.1, f)
            got = _gpu_apply(ctx, name, 1, n, periodic, 0.1, f, dtype=dtype, padded=padded)
            assert Hh.relerr(got, ref) <= bar, (name, n)


@pytest.mark.parametrize("dtype,bar", [(np.float64, 1e-12), (np.float32, 2e-5)])
@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("lanes,line", [(1, 40), (3, 9), (8, 16), (17, 33), (47, 64), (47, 100), (20, 700), (64, 600), (2, 9000)])
def test_narrow_yz(ctx, dtype, bar, periodic, lanes, line):  # noqa: F811
    """The narrow-block y / z sweeps: few lanes, or more chunks than 64 lanes
    leave room for; every chunk capacity, whole and uneven chunks."""
    for name in ("lele_d1_6", "lele_d1_10", "compact_filter"):
        for dim in (2, 3):
            n = (lanes, line, 3) if dim == 2 else (lanes, 2, line)
            f = Hh.random_field(n, seed=61)
            if dtype == np.float32:
                f = f.astype(np.float32).astype(np.float64)
            ref = _oracle_apply(name, dim, n, periodic, 0.1, f)
            got = _gpu_apply(ctx, name, dim, n, periodic, 0.1, f, dtype=dtype)
            assert Hh.relerr(got, ref) <= bar, (name, dim, n)


@pytest.mark.parametrize("n,species", [((24, 20, 20), 1), ((24, 33, 20), 1), ((64, 17, 19), 1), ((50, 40, 36), 2),
                                       ((12, 9, 24), 1)])
def test_paired_gradients(ctx, n, species):  # noqa: F811
    """The y and z gradients of one launch (equal chunk counts, unequal outer
    extents, more fields for two species) and, where the directions differ too
    much, of two: against the oracle's RHS."""
    import cases
    L = (2 * np.pi,) * 3
    X, Y, Z = cases.grid(n, L)
    kw = {}
    if species == 2:
        th = 0.5 * (1 + 0.5 * np.sin(X + Y) * np.cos(Z))
        q = cases.conserved(cases.smooth_prim(X, Y, Z), species=cases.HE_CO2, Y=[1 - th, th])
        kw["species"] = cases.HE_CO2
    else:
        q = cases.conserved(cases.smooth_prim(X, Y, Z))
    gs = cases.gpu_solver(ctx, n, L, q, **kw)
    os_ = cases.oracle_solver(n, L, q, art=True, **kw)
    gs.compute_rhs(False)
    os_.compute_rhs(False)
    _compare_rhs(gs, os_, n)
    for d in (1, 2, 3):
        for j in (1, 2, 3):
            name = f"grad_u[{d}{j}]"
            assert Hh.relerr(gs.field(name), os_.interior(os_.field(name))) <= 1e-12, name
    gs.close()


def _dense(scheme, n, h):
    """The operator of a closed derivative scheme on n points as a dense matrix:
    the left-hand band and the right-hand rows, solved together."""
    q = getattr(scheme, "q", 1)
    lhs = scheme.lhs if q == 2 else [scheme.alpha]
    A, B = np.eye(n), np.zeros((n, n))
    nc = len(scheme.closures)
    for i in range(nc, n - nc):
        for s, a in enumerate(lhs, 1):
            A[i, i - s] = A[i, i + s] = a
        for m, c in enumerate(scheme.coeffs, 1):
            B[i, i + m], B[i, i - m] = c, -c
    for j, row in enumerate(scheme.closures):
        for s in range(-q, q + 1):
            if 0 <= j + s < n:
                A[j, j + s] = A[n - 1 - j, n - 1 - j - s] = row.lhs[q + s]
        for t, w in enumerate(row.rhs):
            B[j, t], B[n - 1 - j, n - 1 - t] = w, -w
    return np.linalg.solve(A, B / h)


@pytest.mark.parametrize("dtype,bar", [(np.float64, 1e-12), (np.float32, 2e-5)])
@pytest.mark.parametrize("half", [1, 2])
@pytest.mark.parametrize("lanes", [6, 50])
def test_long_closures_on_short_chunks(ctx, half, lanes, dtype, bar):  # noqa: F811
    """Closure rows of eight weights reach past the first chunk (four or five
    points on lines of 17 to 20 and 33 to 40) and, for these stencils, past its
    window; every direction, against a dense solve."""
    import compactles_hip as ch
    g = np.random.default_rng(8)
    base = ch.pade_d1_4() if half == 1 else ch.lele_d1_6()
    rows = [ch.ClosureRow(lhs, list(g.uniform(-1, 1, 8))) for lhs in ((0.0, 1.0, 0.5), (0.25, 1.0, 0.25))]
    scheme = ch.CompactScheme("long closures", base.alpha, 0.0, base.coeffs, False, rows)
    for line in (9, 16, 17, 18, 19, 20, 33, 36, 39, 40):
        D = _dense(scheme, line, 0.1)
        for dim in (1, 2, 3):
            n = {1: (line, lanes, 2), 2: (lanes, line, 3), 3: (lanes, 2, line)}[dim]
            f = Hh.random_field(n, seed=71).astype(dtype).astype(np.float64)
            dec = ch.Decomp(n, (False,) * 3)
            plan = ch.plan_direction(ctx, dec, scheme, dim, 0.1, dtype=dtype)
            out = ch.field(ctx, dec, dtype)
            ch.apply_along_(out, plan, ch.DeviceArray.from_numpy(ctx, Hh.pad(f, n), dtype), dec)
            ref = np.moveaxis(np.tensordot(D, f, (1, dim - 1)), 0, dim - 1)
            assert Hh.relerr(Hh.interior(out.numpy().astype(np.float64), n), ref) <= bar, (line, dim)


@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("dim,n", [(1, (256, 6, 5)), (1, (512, 6, 5)), (1, (500, 6, 5)), (1, (768, 3, 2)),
                                   (1, (2000, 5, 3)), (2, (64, 512, 3)), (3, (50, 2, 300)), (2, (6, 900, 2)),
                                   (3, (3, 2, 700)), (2, (128, 128, 512)), (2, (128, 500, 520))])
def test_non_finite_value_spreads_over_its_line(ctx, dim, n, periodic, bad):  # noqa: F811
    """Also where the reduction stops early, a NaN or an infinity leaves no
    finite value on its line, as the sweeps over the whole line would, and
    changes no other line."""
    import compactles_hip as ch
    at = [n[0] // 2, n[1] // 2, n[2] // 2]
    at[dim - 1] = n[dim - 1] // 3
    line = list(at)
    line[dim - 1] = slice(None)
    line = tuple(line)
    f = Hh.random_field(n, seed=81)
    g = f.copy(order="F")
    g[tuple(at)] = bad
    dec = ch.Decomp(n, (periodic,) * 3, n_halo=0)
    for dtype in (np.float64, np.float32):
        for scheme in (ch.lele_d1_6(), ch.lele_d1_10(), ch.compact_filter()):
            plan = ch.plan_direction(ctx, dec, scheme, dim, 0.1, dtype=dtype)
            res = []
            for a in (f, g):
                out = ch.field(ctx, dec, dtype)
                ch.apply_along_(out, plan, ch.DeviceArray.from_numpy(ctx, a, dtype), dec)
                res.append(out.numpy())
            assert not np.isfinite(res[1][line]).any(), (dtype, scheme.name)
            for a in res:
                a[line] = 0
            assert np.array_equal(res[0], res[1]), (dtype, scheme.name)


def _check(ctx, names, dims, n_of, periodic, dtype, bar, seed):
    for dim in dims:
        n = n_of(dim)
        f = Hh.random_field(n, seed=seed).astype(dtype).astype(np.float64)
        for name in names:
            ref = _oracle_apply(name, dim, n, periodic, 0.1, f)
            got = _gpu_apply(ctx, name, dim, n, periodic, 0.1, f, dtype=dtype)
            assert Hh.relerr(got, ref) <= bar, (name, n, dim)


@pytest.mark.parametrize("dtype,bar", [(np.float64, 1e-12), (np.float32, 2e-5)])
@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("line,cap,whole", S.WIDE_LINES)
def test_wide_capacities(ctx, line, cap, whole, periodic, dtype, bar):  # noqa: F811
    """Wide y / z launches at every chunk capacity, whole and uneven chunks, one
    line per lane (which shapes give which: test_line_rule_host)."""
    _check(ctx, ("lele_d1_6", "lele_d1_10", "compact_filter"), (2, 3), lambda d: S.wide(line, d), periodic, dtype, bar, 91)


@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("line", [48, 60, 64, 130, 192, 256])
def test_wide_capacities_two_lines_per_lane(ctx, line, periodic):  # noqa: F811
    """As above in FP32 with even rows and 512 blocks: two lines per lane."""
    _check(ctx, ("lele_d1_6", "compact_filter"), (2,), lambda d: S.wide(line, d, 48, 512), periodic, np.float32, 2e-5, 92)


@pytest.mark.parametrize("dtype,bar", [(np.float64, 1e-12), (np.float32, 2e-5)])
@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("line,cap,whole", S.FEW_LINES)
def test_few_lines_capacity_8(ctx, line, cap, whole, periodic, dtype, bar):  # noqa: F811
    """y / z launches of few lines: 8-point chunks."""
    _check(ctx, ("lele_d1_6", "lele_d1_10", "compact_filter"), (2, 3), lambda d: S.wide(line, d, 49, 7), periodic, dtype,
           bar, 93)


@pytest.mark.parametrize("dtype,bar", [(np.float64, 1e-12), (np.float32, 2e-5)])
@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("line,cap,whole", S.X_LINES)
def test_x_capacity_12(ctx, line, cap, whole, periodic, dtype, bar):  # noqa: F811
    """x lines of 64 chunks at capacity 12: uneven, equal and whole chunks."""
    _check(ctx, ("lele_d1_6", "pade_d1_4", "lele_d1_10", "compact_filter"), (1,), lambda d: (line, 5, 3), periodic, dtype,
           bar, 94)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n,periodic_y,species,paired", S.PAIRS)
def test_paired_gradients_are_the_separate_ones(ctx, n, periodic_y, species, paired, precision):  # noqa: F811
    """The y and z gradients of one launch against the same ones launched
    direction by direction (per-phase timing on): the same bits, also where one
    direction is closed and the other periodic and, on 64^3 FP32, with two lines
    per lane."""
    import cases
    L = (2 * np.pi,) * 3
    X, Y, Z = cases.grid(n, L)
    kw = {} if periodic_y else {"bcs": ((0, 0), (1, 1), (0, 0))}   # slip walls in y
    if species == 2:
        th = 0.5 * (1 + 0.5 * np.sin(X + Y) * np.cos(Z))
        q = cases.conserved(cases.smooth_prim(X, Y, Z), species=cases.HE_CO2, Y=[1 - th, th])
        kw["species"] = cases.HE_CO2
    else:
        q = cases.conserved(cases.smooth_prim(X, Y, Z))
    got = []
    for apart in (False, True):
        s = cases.gpu_solver(ctx, n, L, q, precision=precision, **kw)
        s.profile(apart)
        s.compute_rhs(False)
        got.append([s.field(f"grad_u[{d}{j}]") for d in (1, 2, 3) for j in (1, 2, 3)] +
                   [s.field(f"grad_T[{d}]") for d in (1, 2, 3)])
        s.close()
    for a, b in zip(*got):
        assert np.isfinite(a).all() and np.array_equal(a, b)
