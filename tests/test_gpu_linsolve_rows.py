"""LinSolver on systems with long rows, on either side of the non-zeros per row up to which an iteration takes two
launches (640 on average), and on one matrix after another of the same size: each solve takes its own form."""
import numpy as np
import pytest

import shiokaze_amd as S

pytestmark = pytest.mark.gpu


def system(n, per_row, seed):
    """Symmetric, per_row - 1 neighbours on a ring (per_row odd) with weights in [1/2, 1), the diagonal twice their sum: in
    the maximum norm |A| <= 3/2 and 1/|A^-1| >= 1/2 of the largest and smallest diagonal entry, which differ by less
    than 2, so a relative residual of 1e-12 bounds the relative error by 6e-12."""
    r = np.random.default_rng(seed)
    half = (per_row - 1) // 2
    w = r.uniform(0.5, 1.0, size=(half, n))  # w[k, i]: between i and i + k + 1
    i = np.arange(n)
    rows, cols, vals = [i], [i], []
    diag = np.zeros(n)
    for k in range(half):
        j = (i + k + 1) % n
        rows += [i, j]
        cols += [j, i]
        vals += [-w[k], -w[k]]
        diag += w[k]
        diag[j] += w[k]
    rows, cols, vals = np.concatenate(rows), np.concatenate(cols), np.concatenate([2.0 * diag] + vals)
    order = np.lexsort((cols, rows))
    rowptr = np.concatenate([[0], np.cumsum(np.bincount(rows, minlength=n))])
    return rowptr, cols[order], vals[order], r.normal(size=n)


@pytest.mark.parametrize("jacobi", [False, True])
def test_both_forms_one_after_another(jacobi):
    import scipy.sparse as sp
    import scipy.sparse.linalg
    n = 1300
    with S.LinSolver(0) as ls:
        for seed, per_row in enumerate((7, 639, 641, 7, 1025, 511)):
            print(f"[gpu-case] {n} rows of {per_row} jacobi={jacobi}", flush=True)
            rowptr, col, val, b = system(n, per_row, seed)
            x, r = ls.solve(rowptr, col, val, b, residual=1e-12, preconditioner=S.LS_JACOBI if jacobi else S.LS_NONE)
            assert r.status == 0 and r.converged
            ref = sp.linalg.spsolve(sp.csr_matrix((val, col, rowptr), shape=(n, n)).tocsc(), b)
            assert np.abs(x - ref).max() <= 1e-11 * np.abs(ref).max()
