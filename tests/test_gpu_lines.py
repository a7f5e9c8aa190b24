"""Triangular sweeps of 5-point grid factors at the sizes where their strips can
go wrong: fewer lines than a wavefront's, exact multiples and one past them,
lines shorter than the lanes' skew, long lines (7-point grids beside them).
IC(0) and ILU(0), both directions and the adjoint, equal the oracle's bit for
bit (each row's operations run in the reference's order), also with single
precision factors, with infinities and NaN in the right-hand side, after a
refactorisation, and in the r.z partials of the last sweep."""
import numpy as np
import pytest

import oracle_lib as o

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import mtl4gpu
    return mtl4gpu


def star(nx, ny, nz, seed):
    """A 5-point (nz == 1) or 7-point matrix with random nonsymmetric entries, diagonally dominant."""
    rng = np.random.default_rng(seed)
    r = np.arange(nx * ny * nz)
    i, j, k = r % nx, r // nx % ny, r // (nx * ny)
    offs = [(-nx * ny, k > 0), (-nx, j > 0), (-1, i > 0), (0, r >= 0), (1, i < nx - 1), (nx, j < ny - 1),
            (nx * ny, k < nz - 1)]
    keep = np.stack([m for _, m in offs], axis=1)
    cols = np.stack([r + d for d, _ in offs], axis=1)
    vals = -rng.uniform(0.1, 1.0, keep.shape)
    vals[:, 3] = 6.5 + rng.uniform(0.0, 1.0, len(r))
    S = np.concatenate([[0], np.cumsum(keep.sum(axis=1))]).astype(np.int64)
    return S, cols[keep], vals[keep]


SHAPES = [(2, 2, 1), (7, 3, 1), (64, 64, 1), (5, 65, 1), (130, 64, 1), (33, 128, 1), (40, 129, 1), (301, 173, 1),
          (700, 70, 1), (9, 700, 1), (3600, 66, 1), (4, 4, 4), (20, 33, 9)]


def apply(g, P, v, dtype=np.float64, adjoint=False):
    x, y = g.Vector(data=v, dtype=dtype), g.Vector(len(v), dtype=dtype)
    (P.adjoint_solve if adjoint else P.solve)(x, y)
    return y.numpy()


@pytest.mark.parametrize("shape", SHAPES)
def test_line_sweeps_equal_the_oracle(g, shape):
    print(f"line sweeps {shape}", flush=True)
    S, I, V = star(*shape, seed=sum(shape))
    A = o.CSR(S, I, V)
    v = g.rng_uniform(3, 1, A.n)
    Ag = g.Matrix(S, I, V)
    st, L, U = o.ilu0_factor(A)
    P = g.PC(Ag, g.PC_ILU0)
    for _ in range(2):   # the exchange buffers are reset by the sweeps themselves
        np.testing.assert_array_equal(apply(g, P, v), o.ilu0_solve(L, U, v))
        np.testing.assert_array_equal(apply(g, P, v, adjoint=True), o.ilu0_adjoint_solve(L, U, v))
    st, Uc, Lc = o.ic0_factor(A)
    P = g.PC(Ag, g.PC_IC0)
    np.testing.assert_array_equal(apply(g, P, v), o.ic0_solve(Lc, Uc, v))
    P32 = g.PC(Ag, g.PC_IC0, np.float32)
    np.testing.assert_array_equal(apply(g, P32, v), o.ic0_solve(Lc, Uc, v, factor_dtype=np.float32))
    # new values, same pattern
    S, I, V = star(*shape, seed=sum(shape) + 1)
    A = o.CSR(S, I, V)
    Ag.set_values(V)
    P.refactor(Ag)
    st, Uc, Lc = o.ic0_factor(A)
    np.testing.assert_array_equal(apply(g, P, v), o.ic0_solve(Lc, Uc, v))


@pytest.mark.parametrize("shape", [(70, 140, 1), (20, 33, 9)])
def test_line_sweeps_keep_infinities_and_nans_where_they_belong(g, shape):
    print(f"special values {shape}", flush=True)
    S, I, V = star(*shape, seed=1)
    A = o.CSR(S, I, V)
    st, L, U = o.ilu0_factor(A)
    P = g.PC(g.Matrix(S, I, V), g.PC_ILU0)
    for value in (np.inf, -np.inf, np.nan, -0.0):
        v = g.rng_uniform(3, 1, A.n)
        v[[A.n // 3, A.n - 2]] = value
        ref, refa = o.ilu0_solve(L, U, v), o.ilu0_adjoint_solve(L, U, v)
        np.testing.assert_array_equal(apply(g, P, v), ref)
        np.testing.assert_array_equal(apply(g, P, v, adjoint=True), refa)
    z = np.full(A.n, -0.0)
    np.testing.assert_array_equal(np.signbit(apply(g, P, z)), np.signbit(o.ilu0_solve(L, U, z)))


@pytest.mark.parametrize("shape", [(64, 64, 1), (45, 130, 1), (20, 33, 9)])
def test_line_sweeps_single_precision_vectors(g, shape):
    # float factors and vectors: the operations of the double sweeps in float
    print(f"float vectors {shape}", flush=True)
    S, I, V = star(*shape, seed=2)
    A = o.CSR(S, I, V)
    st, U, L = o.ic0_factor(A)
    v = g.rng_uniform(3, 1, A.n).astype(np.float32)
    P = g.PC(g.Matrix(S, I, V), g.PC_IC0, np.float32)
    L32, U32 = [m.data.astype(np.float32) for m in (L, U)]
    y = v.copy()
    for r in range(A.n):
        acc = y[r]
        for p in range(L.starts[r], L.starts[r + 1] - 1):
            acc = np.float32(acc - np.float32(L32[p] * y[L.indices[p]]))
        y[r] = acc * L32[L.starts[r + 1] - 1]
    for r in range(A.n - 1, -1, -1):
        acc = y[r]
        for p in range(U.starts[r] + 1, U.starts[r + 1]):
            acc = np.float32(acc - np.float32(U32[p] * y[U.indices[p]]))
        y[r] = acc * U32[U.starts[r]]
    np.testing.assert_array_equal(apply(g, P, v, dtype=np.float32), y)


def test_a_wait_that_gave_up_is_reported_by_each_direction_and_cleared(g, monkeypatch):
    # one poll per wait: the strips after the first give up, and every wave still ends
    print("line sweeps with a one-poll limit", flush=True)
    S, I, V = star(300, 200, 1, seed=4)
    A = o.CSR(S, I, V)
    st, L, U = o.ilu0_factor(A)
    P = g.PC(g.Matrix(S, I, V), g.PC_ILU0)
    v = g.rng_uniform(3, 1, A.n)
    for adjoint, ref in ((False, o.ilu0_solve(L, U, v)), (True, o.ilu0_adjoint_solve(L, U, v))):
        np.testing.assert_array_equal(apply(g, P, v, adjoint=adjoint), ref)
        with monkeypatch.context() as m:
            m.setenv("M4G_SPIN_LIMIT", "1")
            with pytest.raises(g.M4GError) as e:
                apply(g, P, v, adjoint=adjoint)
            assert e.value.status == g.ERR_TIMEOUT
        for _ in range(2):
            np.testing.assert_array_equal(apply(g, P, v, adjoint=adjoint), ref)


def test_partials_of_the_last_sweep_on_long_lines(g):
    # A = I on a star pattern: alpha of the first CG step is r.z / r.r = 1.  The last cells of each line,
    # which the upper sweep meets first, are 1, the others so small that a float sum that holds a few
    # ones drops their squares: 15 000 of them, 8e-4 of the whole.  Both dots add few products (at most 52)
    # in a row in float and the rest in double: alpha is off by 52 * 2**-24 = 3.1e-6 each at most.
    nx, ny = 15000, 66
    print(f"partials in float {nx} x {ny}", flush=True)
    S, I, V = star(nx, ny, 1, seed=1)
    V = np.where(I == np.repeat(np.arange(nx * ny), np.diff(S)), 1.0, 0.0)
    small = np.float32(np.sqrt(0.45 * 2.0 ** -20))
    b = np.full((ny, nx), small, np.float32)
    b[:, -8:] = 1.0
    Ag = g.Matrix(S, I, V)
    P = g.PC(Ag, g.PC_IC0, np.float32)
    assert P.stats()["tiles_upper"] == 2
    x = g.Vector(nx * ny, dtype=np.float32)
    x.fill(0.0)
    it, _ = g.make_iteration(1, 1e-30, 0.0, float(np.linalg.norm(b.astype(np.float64))))
    g.cg(Ag, x, g.Vector(data=b.ravel(), dtype=np.float32), P, it)
    alpha = x.numpy()[nx - 1]
    print(f"  alpha - 1 = {alpha - 1.0:.2e}", flush=True)
    assert abs(alpha - 1.0) <= 1e-5


@pytest.mark.parametrize("nx,ny,lines", [(2, 139776, True), (2, 139777, False), (41, 128000, False), (42, 128000, True)])
def test_large_narrow_grids_take_the_general_sweep(g, nx, ny, lines):
    # above 256 MB of coefficients a strip may hold 64 bytes a row: 24 * (lanes and steps) / cells.
    # nx = 2: 80 steps, 122 880 bytes a strip, 2184 strips at most; nx = 41 and 42: 112 steps, 65.6 and 64 bytes a row
    print(f"narrow grid {nx} x {ny}", flush=True)
    S, I, V = star(nx, ny, 1, seed=nx)
    A = o.CSR(S, I, V)
    v = g.rng_uniform(3, 1, A.n)
    st, L, U = o.ilu0_factor(A)
    P = g.PC(g.Matrix(S, I, V), g.PC_ILU0)
    s = P.stats()
    assert lines == (s["tiles_lower"] == -(-ny // 64) and s["tile_ny"] == 64), s
    np.testing.assert_array_equal(apply(g, P, v), o.ilu0_solve(L, U, v))
    np.testing.assert_array_equal(apply(g, P, v, adjoint=True), o.ilu0_adjoint_solve(L, U, v))


@pytest.mark.parametrize("nx,ny", [(3722, 66), (3723, 66), (8000, 3), (16010, 3), (16011, 3)])
def test_line_sweeps_on_the_longest_lines(g, nx, ny):
    # a step holds 8 bytes of LDS: above 64 KB (nx = 3 723 on) it is asked for, above 160 KB (nx = 16 010) there
    # is none and the general sweep takes the grid
    print(f"long lines {nx} x {ny}", flush=True)
    S, I, V = star(nx, ny, 1, seed=nx)
    A = o.CSR(S, I, V)
    v = g.rng_uniform(3, 1, A.n)
    Ag = g.Matrix(S, I, V)
    st, L, U = o.ilu0_factor(A)
    P = g.PC(Ag, g.PC_ILU0)
    s = P.stats()
    assert (nx <= 16010) == (s["tiles_lower"] == -(-ny // 64) and s["tile_nx"] == nx and s["tile_ny"] == 64), s
    np.testing.assert_array_equal(apply(g, P, v), o.ilu0_solve(L, U, v))
    np.testing.assert_array_equal(apply(g, P, v, adjoint=True), o.ilu0_adjoint_solve(L, U, v))
    st, Uc, Lc = o.ic0_factor(A)
    P = g.PC(Ag, g.PC_IC0, np.float32)
    np.testing.assert_array_equal(apply(g, P, v), o.ic0_solve(Lc, Uc, v, factor_dtype=np.float32))


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("shape", [(2, 2, 1), (64, 65, 1), (700, 70, 1), (20, 33, 9)])
def test_partials_of_the_last_sweep(g, shape, dtype, monkeypatch):
    # alpha = r.z / p.Ap of the first CG step, from x = alpha z, against a dot kernel's: both add in double what
    # float products and sums of at most 52 in a row give (52 * 2**-24 = 3.1e-6 for float), r.z > 0 without
    # cancellation in the large
    print(f"partials {shape} {np.dtype(dtype).name}", flush=True)
    S, I, V = star(*shape, seed=3)
    rows = np.repeat(np.arange(len(S) - 1), np.diff(S))
    key = np.minimum(rows, I) * len(S) + np.maximum(rows, I)   # one value for both halves
    off = rows != I
    V[off] = -0.1 - (key[off] * 2654435761 % 1000) * 9e-4
    b = 0.5 + g.rng_uniform(5, 1, len(S) - 1) ** 2
    Ag = g.Matrix(S, I, V)
    P = g.PC(Ag, g.PC_IC0, dtype)
    z = apply(g, P, b.astype(dtype), dtype=dtype)
    xs = []
    for separate in (False, True):
        if separate:
            monkeypatch.setenv("M4G_CG_SWEEP_DOT", "0")
        monkeypatch.setenv("M4G_GRID_CG", "0")
        x = g.Vector(len(b), dtype=dtype)
        x.fill(0.0)
        it, _ = g.make_iteration(1, 1e-30, 0.0, 1.0)
        g.cg(Ag, x, g.Vector(data=b, dtype=dtype), P, it)
        xs.append(x.numpy())
    k = np.argmax(z)
    alpha = [float(x[k]) / float(z[k]) for x in xs]
    assert abs(alpha[0] / alpha[1] - 1.0) <= (1e-13 if dtype == np.float64 else 1e-5), alpha
