"""The outer-block kernel (CholeskyQR2 of up to 128 columns with Householder
reconstruction) at the edges of its widths and heights, through QR::Factor
against the oracle: one half and two, ragged ends, square last blocks (whose
last column has no reflector), blocks that need the exact second factorization
or a third pass, rejected blocks, and columns with exact zeros below the
diagonal (tau = 0).  Bar: the factorization tests' (R, tau, V to 1e-11 of the
column scale); for badly conditioned blocks, whose R is only determined to
eps * condition, residual and orthogonality <= 10 n eps."""
import numpy as np
import pytest

import oracle as O
import rnp2_amd as R
from metrics import orth_error, qr_residual, rel_err_colscaled

pytestmark = pytest.mark.gpu


def check(a, elementwise=True):
    m, n = a.shape
    k = min(m, n)
    af, tau = R.factor(a)
    r = np.triu(af[:k])
    q = R.generateq(af[:, :k], tau, n=k)
    assert qr_residual(a, q, r) <= 10 and orth_error(q) <= 10
    if elementwise:
        af_o, tau_o = O.factor(a)
        assert rel_err_colscaled(r, np.triu(af_o[:k])) <= 1e-11
        assert np.max(np.abs(tau - tau_o)) <= 1e-11
        assert np.max(np.abs(np.tril(af, -1) - np.tril(af_o, -1))) <= 1e-9
    return af, tau


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 79, 80, 81, 100, 127, 128, 129, 143, 144, 191, 193, 200])
@pytest.mark.parametrize("extra", [0, 1, 30, 64, 700])
def test_widths_and_heights(n, extra):
    check(np.random.default_rng(n * 1000 + extra).standard_normal((n + extra, n)))


@pytest.mark.parametrize("m,n", [(20, 300), (64, 300), (100, 101), (128, 400), (130, 257)])
def test_wide(m, n):
    check(np.random.default_rng(m + n).standard_normal((m, n)))


@pytest.mark.parametrize("m,n", [(90, 60), (400, 100), (3000, 128)])
@pytest.mark.parametrize("cond", [1e2, 1e4, 1e5, 1e6, 1e8, 1e12])
def test_conditioned_blocks(m, n, cond):
    rng = np.random.default_rng(n)
    u = np.linalg.qr(rng.standard_normal((m, n)))[0]
    v = np.linalg.qr(rng.standard_normal((n, n)))[0]
    check(np.asfortranarray(u * np.logspace(0, -np.log10(cond), n) @ v), elementwise=cond <= 1e4)


@pytest.mark.parametrize("m,n", [(40, 30), (90, 90), (150, 100), (180, 128)])
def test_zero_tails_keep_tau_zero(m, n):
    """Upper triangular input, and one with a zero tail in each half: no
    reflector there (Reflector.hpp:122-125), the entries unchanged."""
    a = np.triu(np.random.default_rng(n).standard_normal((m, n)))
    af, tau = check(a)
    assert np.array_equal(tau, np.zeros_like(tau)) and np.array_equal(af, a)


@pytest.mark.parametrize("n", [60, 100, 128])
def test_repeated_runs_agree(n):
    a = np.random.default_rng(n).standard_normal((900, n))
    f1, t1 = R.factor(a)
    f2, t2 = R.factor(a)
    assert np.array_equal(f1, f2) and np.array_equal(t1, t2)
