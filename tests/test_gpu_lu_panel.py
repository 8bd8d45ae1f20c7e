"""The register-resident LU panel at the edges of its workgroups (512 rows
each) and column groups (eight columns), against the oracle: the same pivots,
L and U to rounding (entries of PA = LU panels bounded by 2 k eps growth, as
|LU - LU_o| <= 1e-11 max|A| max(1, max(m, n)/100), the factorization tests'
bar), exact ties resolved to the lower row, and NaN and Inf handled as the
sequential scan does (a NaN at the pivot row is kept, elsewhere never
preferred), in one panel and the same entries non-finite."""
import numpy as np
import pytest

import oracle as O
import rnp2_amd as R

pytestmark = pytest.mark.gpu


def check(a):
    lo, po, io = O.lu_factor(a)
    lg, pg, ig = R.lu_factor(a)
    assert np.array_equal(po, pg) and io == ig
    fin = np.isfinite(lo)
    assert np.array_equal(fin, np.isfinite(lg))
    big = np.abs(a[np.isfinite(a)]).max()
    assert np.abs(lg[fin] - lo[fin]).max() <= 1e-11 * big * max(1.0, max(a.shape) / 100.0)


@pytest.mark.parametrize("m,n", [(2, 2), (7, 8), (8, 7), (9, 9), (63, 64), (511, 63), (512, 64), (513, 65), (514, 72),
                                 (1024, 127), (1025, 130), (4097, 9), (33000, 66), (65536, 5)])
def test_panel_edges(m, n):
    check(np.random.default_rng(m + n).standard_normal((m, n)))


@pytest.mark.parametrize("m,n", [(40, 20), (700, 60), (1100, 64)])
def test_exact_ties_take_the_lower_row(m, n):
    """Every row twice: each pivot has an exact rival, in another wave or
    workgroup for the taller ones."""
    b = np.random.default_rng(n).integers(-9, 10, (m // 2, n)).astype(float)
    check(np.vstack([b, b]))
    check(np.vstack([b[::-1], b]))
    p = np.eye(m)[np.random.default_rng(m).permutation(m)][:, :n]
    check(p)


@pytest.mark.parametrize("m,n", [(40, 20), (600, 33), (1300, 64)])
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_nonfinite_entries(m, n, bad):
    rng = np.random.default_rng(m)
    a = rng.standard_normal((m, n))
    b = a.copy()
    b[m - 1, 3] = bad          # below the pivot rows
    check(b)
    b = a.copy()
    b[0, 0] = bad              # at the first pivot row
    check(b)
    b = a.copy()
    b[m // 2, n - 1] = bad     # in the last column
    check(b)
