"""Triangular sweeps of irregular factors on both sides of each compiled piece
width (3, 4, 8, 13, 16 and rows of several pieces): ILU(0) solves in both
directions and with single precision factors equal the oracle's bit for bit, as
each row's operations run in the reference's order."""
import numpy as np
import pytest

import oracle_lib as o

pytestmark = pytest.mark.gpu


def half_rows(n, width, reach, seed):
    """Up to `width` entries below and above the diagonal, within `reach` of it; diagonally dominant."""
    rng = np.random.default_rng(seed)
    S, I, V = [0], [], []
    for r in range(n):
        lo = np.arange(max(0, r - reach), r)
        hi = np.arange(r + 1, min(n, r + reach + 1))
        k = width if r % 3 else rng.integers(0, width + 1)
        c = np.sort(np.concatenate([rng.permutation(lo)[:k], [r], rng.permutation(hi)[:k]]))
        v = -rng.uniform(0.1, 1.0, len(c))
        v[c == r] = 2.5 * width
        S.append(S[-1] + len(c))
        I.append(c)
        V.append(v)
    return np.array(S, np.int64), np.concatenate(I).astype(np.int64), np.concatenate(V)


@pytest.mark.parametrize("width", [3, 4, 5, 8, 9, 12, 13, 14, 16, 17, 40])
def test_sweeps_at_the_piece_widths(width):
    import mtl4gpu as g
    print(f"piece width {width}", flush=True)
    n = 6000
    S, I, V = half_rows(n, width, 300, width)
    A = o.CSR(S, I, V)
    v = g.rng_uniform(3, 1, n)
    st, L, U = o.ilu0_factor(A)
    for dtype in (np.float64, np.float32):
        P = g.PC(g.Matrix(S, I, V), g.PC_ILU0, dtype)
        for _ in range(2):   # the exchange buffers are reset by the sweeps themselves
            x, y = g.Vector(data=v), g.Vector(n)
            P.solve(x, y)
            np.testing.assert_array_equal(y.numpy(), o.ilu0_solve(L, U, v, factor_dtype=dtype))
            if dtype == np.float64:
                P.adjoint_solve(x, y)
                np.testing.assert_array_equal(y.numpy(), o.ilu0_adjoint_solve(L, U, v))
