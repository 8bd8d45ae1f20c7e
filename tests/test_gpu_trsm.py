"""Triangular solves, four right-hand sides to a workgroup: right-hand sides
short of and beyond four, orders around the 64-row block, both triangles,
every operation, unit and other diagonals, against NumPy's solve."""
import numpy as np
import pytest

import rnp2_amd as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("n,nrhs", [(1, 1), (63, 4), (64, 5), (65, 3), (129, 8), (700, 1), (1090, 9)])
@pytest.mark.parametrize("trans", ["N", "T", "C"])
def test_right_hand_sides(n, nrhs, trans, cplx):
    rng = np.random.default_rng(n + nrhs)

    def rand(*shape):
        x = rng.standard_normal(shape)
        return x + 1j * rng.standard_normal(shape) if cplx else x

    # a strong diagonal and multipliers of size 1/n: both triangles well conditioned
    lu = rand(n, n) / n + 2.0 * np.eye(n)
    b = rand(n, nrhs)
    a = (np.tril(lu, -1) + np.eye(n)) @ np.triu(lu)
    want = np.linalg.solve({"N": a, "T": a.T, "C": a.conj().T}[trans], b)
    got = R.lu_solve(trans, np.asfortranarray(lu), np.arange(n, dtype=np.int32), b)
    # n eps |L||U||x| from each side's two solves, the triangles' norms about 2
    tol = 16 * max(n, 8) * np.finfo(np.float64).eps * np.abs(want).max()
    assert np.abs(got - want).max() <= tol
