"""The block elimination that the time step solves with (csrc/solve.hpp): its
error against extended precision beside that of the banded LU with partial
pivoting, restated in numpy, for the matrices of vel_matrices.

Blocks of four rows are eliminated from both ends towards the block
ceil(N / 4) // 2; rows past N are identity rows; rows are interchanged within a
block's inverse only."""
import numpy as np
import pytest
import scipy.linalg as sl

import opf_oracle as O

KL = 4


def _matrix(me, N, Mp, m, alpha, k, PM, BC, c1, c2):
    r2 = me.rp[-2]
    d = -(r2 * (Mp * m) ** 2) - (alpha * k) ** 2
    if PM:
        d = d - r2 - 2.0 * PM * Mp * m * r2
    A = c2 * O.band_to_dense(me.radLap)
    A[np.arange(N), np.arange(N)] += c2 * d + c1
    A[0] = 0.0
    A[0, :KL + 1] = me.dr0[:, 1 - (m * Mp + abs(PM)) % 2]
    A[N - 1] = 0.0
    A[N - 1, N - KL - 1:] = me.dr1[:, BC]
    return A


def _block_solve(A, b):
    """The solution, and the largest row sum of a subtracted term over that of
    the diagonal block it is subtracted from."""
    N = len(A)
    NB = (N + 3) // 4
    mid = NB // 2
    P = np.eye(4 * NB)
    P[:N, :N] = A
    c = np.zeros((NB, 4, b.shape[1]))
    c.reshape(4 * NB, -1)[:N] = b

    def blk(s, t):
        return P[4 * s:4 * s + 4, 4 * t:4 * t + 4]

    D = np.array([blk(t, t) for t in range(NB)])
    z, E, growth = np.zeros_like(c), np.zeros_like(D), 0.0
    sides = (range(0, mid), 1), (range(NB - 1, mid, -1), -1)
    for ts, dt in sides:
        for t in ts:
            u = t + dt
            E[t] = np.linalg.inv(D[t])
            z[t] = E[t] @ c[t]
            U = blk(u, t) @ (E[t] @ blk(t, u))
            growth = max(growth, (np.abs(U).sum(1) / np.abs(blk(u, u)).sum(1)).max())
            D[u] = D[u] - U
            c[u] = c[u] - blk(u, t) @ z[t]
    x = np.zeros_like(c)
    x[mid] = np.linalg.inv(D[mid]) @ c[mid]
    for ts, dt in sides:
        for t in reversed(ts):
            x[t] = z[t] - E[t] @ (blk(t, t + dt) @ x[t + dt])
    return x.reshape(4 * NB, -1)[:N], growth


def _band_solve(A, b):
    N = len(A)
    ab = np.zeros((3 * KL + 1, N))
    for j in range(N):
        for i in range(max(0, j - KL), min(N, j + KL + 1)):
            ab[2 * KL + i - j, j] = A[i, j]
    lu, ipiv, info = sl.lapack.dgbtrf(ab, KL, KL)
    assert info == 0
    return sl.lapack.dgbtrs(lu, KL, KL, b, ipiv)[0]


def _refined(A, b):
    lu = sl.lu_factor(A)
    x = sl.lu_solve(lu, b).astype(np.longdouble)
    for _ in range(6):
        r = b.astype(np.longdouble) - A.astype(np.longdouble) @ x
        x = x + sl.lu_solve(lu, r.astype(float))
    return x


@pytest.mark.parametrize("N", [9, 10, 15, 16, 32, 33, 64, 96, 127, 128])
@pytest.mark.parametrize("kind", ["pressure", "velocity"])
def test_error_beside_the_banded_lu(N, kind):
    """Over pairs (k, m), the error is that of the banded LU: within three times
    it in the geometric mean (0.3 to 1.8 found) and fifty times for a single
    system, the two errors being of independent roundings.  The subtracted
    terms stay below the diagonal blocks' rows (0.7 found), which is why nothing
    needs to be interchanged between blocks."""
    me = O.build_mesh(N)
    rng = np.random.default_rng(N)
    ratio = []
    for trial in range(40):
        k, m, Mp = int(rng.integers(0, 12)), int(rng.integers(0, 8)), int(rng.integers(1, 4))
        if kind == "pressure":
            k = max(k, 1) if m == 0 else k
            A = _matrix(me, N, Mp, m, 1.25, k, 0, 1, 0.0, 1.0)
        else:
            dt, Re = 10.0 ** rng.uniform(-3, -1.5), 10.0 ** rng.uniform(3, 4)
            A = _matrix(me, N, Mp, m, 1.25, k, int(rng.integers(-1, 2)), 0, 1.0 / dt, -0.51 / Re)
        b = rng.standard_normal((N, 4))
        b[0] = b[-1] = 0.0
        ref = _refined(A, b)
        x, growth = _block_solve(A, b)
        assert growth < 1.0
        scale = np.abs(ref).max()
        e, e_lu = (max(float(np.abs(v - ref).max() / scale), 1e-18) for v in (x, _band_solve(A, b)))
        assert e <= 50.0 * e_lu + 1e-15, (k, m, e, e_lu)
        ratio.append(e / e_lu)
    assert np.exp(np.mean(np.log(ratio))) <= 3.0
