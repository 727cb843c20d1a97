"""Inputs and references of the LU form tests, shared by the CPU emulation's
scenarios and the GPU tests."""
import numpy as np


def uniform(rng, batch, m, n):
    """batch uniform systems, column-major (batch, n, m)."""
    return rng.uniform(-1, 1, (batch, n, m))


def zero_columns_with_nan(rng, n, cols):
    """One uniform system (column-major (1, n, n)), but each of the given
    columns zero except one NaN below the diagonal: its pivot is an exact zero
    with a multiplier that is not."""
    A = rng.uniform(-1, 1, (1, n, n))
    for c in cols:
        A[0, c] = 0.0
        A[0, c, n - 1 - c % 3] = np.nan
    return A


def tied_pairs(rng, n, ulp):
    """One system (column-major (1, n, n)) in which every other column has two
    candidates for its pivot, of magnitude 1 + k ulp, k = 0..3: block upper
    triangular with 2 x 2 diagonal blocks, its rows permuted. Equal candidates
    go to the lowest position, which depends on every interchange before, and
    rounding reaches no candidate of a later pair."""
    M = np.triu(rng.integers(-3, 4, (n, n)).astype(np.float64), 2)
    for j in range(0, n - 1, 2):
        M[j:j + 2, j] = (1 + ulp * rng.integers(0, 4, 2)) * rng.choice([-1.0, 1.0], 2)
        M[j:j + 2, j + 1] = [0.0, rng.integers(1, 5)]
    if n % 2:
        M[n - 1, n - 1] = 2.0
    return np.ascontiguousarray(M[rng.permutation(n)].T)[None]


def dominant_with_zeros(rng, m, n, zeros):
    """m x n with a dominant diagonal, but each of the given rows reaches its
    step unchanged, with a zero on the diagonal."""
    M = rng.uniform(-1, 1, (m, n))
    M[np.arange(n), np.arange(n)] += 2.0 * n
    for z in zeros:
        M[z, :z + 1] = 0.0
    return M


def getf2_nopiv(M):
    """Unblocked LU of M without pivoting; a zero pivot leaves its column
    unscaled and its step is applied all the same (LAPACK dgetf2). Returns
    (LU, info)."""
    M = M.copy()
    info = 0
    for j in range(min(M.shape)):
        if M[j, j] != 0:
            M[j + 1:, j] /= M[j, j]
        elif info == 0:
            info = j + 1
        M[j + 1:, j + 1:] -= np.outer(M[j + 1:, j], M[j, j + 1:])
    return M, info
