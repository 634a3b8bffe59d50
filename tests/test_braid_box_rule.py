"""The row rule of the GPU steady ant, checked on the CPU.

With U the union of the children's points of a node of s rows (row -> column,
lo or hi), CI its inverse, and for a row line r
    Y(r) = #{lo rows >= r},  z_r(c) = lo(c) ? CI(c) >= r : CI(c) < r,
    T(r) = min{c : #{c' < c : z_r(c')} >= Y(r)},
the product's point of row r is T(r) - 1 when T(r) > 0 and U(r) is counted at
T(r) (lo ? U >= T : U < T), and U(r) otherwise: no row needs its neighbours'
results.  braid_kernels.hip finds T for all rows of a g x g box from the point
where the ant's path enters it: a row line (T of that line known, delta 0) or
a column line c (delta(rho, c) = -1 at the row rho where the path crosses it).
This restates both forms in numpy and compares them with the oracle's steady
ant.  It runs no GPU code."""
import numpy as np
import pytest

import oracle


def counted(idx, lo, at):
    return np.where(lo, idx >= at, idx < at)


def children(P, Q):
    """The two half products lifted into the node: U (row -> column) and lo."""
    s = len(P)
    h = s // 2
    Qinv = np.empty(s, np.int64)
    Qinv[Q] = np.arange(s)            # column -> shared row
    U, lo = np.empty(s, np.int64), np.zeros(s, bool)
    for half in (0, 1):
        rows = np.nonzero((P >= h) == bool(half))[0]
        cols = np.nonzero((Qinv >= h) == bool(half))[0]
        R = product(P[rows] - half * h, invert(Qinv[cols] - half * h))
        U[rows] = cols[R]
        lo[rows] = half == 0
    return U, lo


def invert(p):
    q = np.empty_like(p)
    q[p] = np.arange(len(p))
    return q


def by_rows(U, lo):
    s = len(U)
    CI = invert(U)
    clo = lo[CI]
    out = U.copy()
    for r in range(s):
        Y = int((lo[r:]).sum())
        Z = np.concatenate([[0], np.cumsum(counted(CI, clo, r))])
        T = int(np.nonzero(Z >= Y)[0][0])
        if T > 0 and counted(U[r], lo[r], T):
            out[r] = T - 1
    return out


def line(E, elo, s, g, j):
    """Boundary j over the entries E: the first position where z_j has been
    counted Y_j times."""
    b = (s - 1 - E) // g
    Y = int((elo & (b < j)).sum())
    Z = np.concatenate([[0], np.cumsum(np.where(elo, b < j, b >= j))])
    return int(np.nonzero(Z >= Y)[0][0])


def by_boxes(U, lo, g):
    s = len(U)
    nb = s // g
    CI = invert(U)
    clo = lo[CI]
    out, seen = U.copy(), np.zeros(s, int)
    row_T = [0] + [line(CI, clo, s, g, j) for j in range(1, nb)]
    col_T = [0] + [line(U, lo, s, g, j) for j in range(1, nb)]
    for q in range(2 * nb - 1):
        if q < nb:
            r_lo, cs, base = s - (q + 1) * g, row_T[q], 0
            rho = r_lo + g - 1
            below = lambda r: r <= rho  # noqa: E731
            cb = 0 if cs == 0 else (cs - 1) // g
        else:
            i = q - nb + 1
            if col_T[nb - i] == 0:
                continue
            rho, cs, base, cb = col_T[nb - i] - 1, i * g, 1, i
            r_lo = s - ((s - 1 - rho) // g + 1) * g
            below = lambda r: r < rho  # noqa: E731
        ce = (cb + 1) * g
        for r in range(r_lo, rho + 1):
            need = base + sum(bool(counted(U[k], lo[k], cs)) for k in range(r, r_lo + g) if below(k))
            Z = np.cumsum(counted(CI[cs:ce], clo[cs:ce], r))
            if need == 0:
                T = cs
            elif len(Z) and Z[-1] >= need:
                T = cs + int(np.nonzero(Z >= need)[0][0]) + 1
            else:
                continue
            seen[r] += 1
            if T > 0 and counted(U[r], lo[r], T):
                out[r] = T - 1
    assert (seen == 1).all()
    return out


def product(P, Q):
    if len(P) == 1:
        return np.zeros(1, np.int64)
    return by_rows(*children(P, Q))


def cases(s):
    rng = np.random.default_rng(s)
    idp = np.arange(s)
    yield "random", rng.permutation(s), rng.permutation(s)
    yield "identity", idp, rng.permutation(s)
    yield "reversal", idp[::-1].copy(), rng.permutation(s)
    yield "shift", np.roll(idp, s // 3), np.roll(idp, -(s // 5))
    swaps = idp.copy()
    for _ in range(3):
        x, y = rng.integers(0, s, 2)
        swaps[x], swaps[y] = swaps[y], swaps[x]
    yield "swaps", swaps, rng.permutation(s)


@pytest.mark.parametrize("s", [2, 4, 8, 16, 32, 64, 128])
def test_rows_are_independent(s):
    for name, P, Q in cases(s):
        want = oracle.steady_ant(P.astype(np.int32), Q.astype(np.int32))
        assert np.array_equal(product(P, Q), want), name


@pytest.mark.parametrize("s,g", [(32, 8), (64, 8), (64, 16), (128, 32), (256, 64)])
def test_boxes_cover_every_row_once(s, g):
    for name, P, Q in cases(s):
        U, lo = children(P, Q)
        assert np.array_equal(by_boxes(U, lo, g), by_rows(U, lo)), name
