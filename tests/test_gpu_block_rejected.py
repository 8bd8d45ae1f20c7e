"""Blocks that the outer-block kernel rejects and refactors column by column
(every workgroup its 64 rows, a grid-wide step per column), against the oracle:
exact zeros below the diagonal in short blocks and ragged halves (tau = 0,
Reflector.hpp:122-125), blocks too ill conditioned for CholeskyQR, zero columns,
and norms that need Generate's scaling.  Bar: the factorization tests' (R, tau, V
to 1e-11 of the column scale); for ill-conditioned blocks, whose R is only
determined to eps * condition, residual and orthogonality <= 10 n eps."""
import time

import numpy as np
import pytest
import torch

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
        assert np.array_equal(tau == 0, tau_o == 0)
        assert rel_err_colscaled(r, np.triu(af_o[:k])) <= 1e-11
        assert np.max(np.abs(tau - tau_o)) <= 1e-11
        assert np.max(np.abs(np.tril(af, -1) - np.tril(af_o, -1))) <= 1e-9


def zero_tails_from(m, n, j):
    """Columns from j on have exact zeros below the diagonal, and still do when
    the reflectors of the columns before, dense in the first j rows, are through."""
    rng = np.random.default_rng(m + n + j)
    a = np.triu(rng.standard_normal((m, n))) / n + 2.0 * np.eye(m, n)
    a[:j, :j] = rng.standard_normal((j, j)) / n + np.eye(j)
    return a


# three workgroups and many; one half and two, short blocks and tall ones
@pytest.mark.parametrize("m,n,j", [(16, 16, 0), (20, 17, 3), (64, 64, 10), (65, 64, 63), (90, 90, 0), (100, 81, 70),
                                   (130, 128, 64), (191, 128, 1), (192, 55, 0), (700, 55, 20), (4000, 33, 32),
                                   (192, 100, 66), (3000, 127, 90), (9001, 100, 70), (16384, 90, 80)])
def test_zero_tails(m, n, j):
    check(zero_tails_from(m, n, j))


@pytest.mark.parametrize("m,n", [(70, 64), (150, 128), (800, 40), (5000, 128), (16384, 128)])
@pytest.mark.parametrize("kind", ["ill", "zero columns", "small", "large"])
def test_other_rejected_blocks(m, n, kind):
    rng = np.random.default_rng(m + n)
    a = rng.standard_normal((m, n))
    if kind == "ill":
        u = np.linalg.qr(a)[0]
        v = np.linalg.qr(rng.standard_normal((n, n)))[0]
        a = u * np.logspace(0, -13, n) @ v
    elif kind == "zero columns":
        a[:, [0, n // 2, n - 1]] = 0.0
    else:  # one column's squared norm leaves [2^-600, 2^600]
        a[:, n // 3] *= 2.0 ** (-330 if kind == "small" else 330)
    check(a, elementwise=kind in ("small", "large"))


def seconds(a):
    m, n = a.shape
    h = R.Handle()
    A0, A = (R.colmajor_empty(m, n, torch.float64) for _ in range(2))
    A0.copy_(torch.from_numpy(a).cuda())
    tau = torch.empty(n, dtype=torch.float64, device="cuda")
    ts = []
    for _ in range(6):
        A.copy_(A0)
        torch.cuda.synchronize()
        t = time.perf_counter()
        h.geqrf(A, tau)
        h.synchronize()
        ts.append(time.perf_counter() - t)
    h.close()
    return min(ts)


@pytest.mark.parametrize("m,n,j", [(10000, 32, 5), (10000, 100, 70), (16384, 127, 64)])
def test_cost_of_a_rejection(m, n, j):
    """A rejected block costs a grid-wide step per column: 30 us each at most (10
    to 15 measured; one workgroup alone took 200 to 1000)."""
    best = [seconds(a) for a in (np.random.default_rng(0).standard_normal((m, n)), zero_tails_from(m, n, j))]
    assert best[1] - best[0] <= 30e-6 * n, best


@pytest.mark.parametrize("m,n,j", [(10000, 100, 20), (3000, 64, 63), (3000, 80, 0)])
def test_short_tail_in_a_full_half_is_no_rejection(m, n, j):
    """One column of the first 64 whose entries below the diagonal are 1e-9 of its
    norm once the columns before are through: a tall matrix keeps the fast path
    (its reflector, tau = 2 to rounding, is what the reference has there)."""
    rng = np.random.default_rng(n)
    a = rng.standard_normal((m, n))
    base = seconds(a)
    af, tau = O.factor(a[:, :j]) if j else (a[:, :0], [])
    x = np.zeros(m)
    x[j] = 1.0
    x[j + 1:] = 1e-9 * rng.standard_normal(m - j - 1) / np.sqrt(m)
    for i in reversed(range(j)):  # column j as the reflectors before it turn into x
        v = np.concatenate([np.zeros(i), [1.0], af[i + 1:, i]])
        x -= tau[i] * v * (v @ x)
    a[:, j] = x
    check(a)
    assert seconds(a) <= 1.5 * base


@pytest.mark.parametrize("m,n", [(130, 128), (200, 100), (3000, 128), (2000, 256), (16384, 128)])
@pytest.mark.parametrize("eps", [1e-5, 1e-7, 1e-9, 1e-12, 1e-15, 0.0])
def test_second_half_near_the_first_halfs_span(m, n, eps):
    """Collinear regressors: the second 64 columns of a block are combinations of
    the first 64 plus eps noise.  Residual and orthogonality at the bar; the block
    takes one or two passes more (50 us each) instead of a column-wise
    refactorization (1 ms and more)."""
    rng = np.random.default_rng(m)
    a = rng.standard_normal((m, n))
    base = seconds(a)
    for i in range(0, n, 128):
        e = min(i + 128, n)
        a[:, i + 64:e] = a[:, i:i + 64] @ rng.standard_normal((64, e - i - 64)) / 8 + eps * a[:, i + 64:e]
    check(a, elementwise=False)
    assert seconds(a) <= 1.7 * base + 100e-6 * (n // 128)


def test_second_half_near_a_badly_conditioned_first_half():
    """The first half at condition 1e4: one projection leaves 1e-8 of the second
    half along it, more than the 1e-11 that is to be found outside."""
    rng = np.random.default_rng(5)
    u = np.linalg.qr(rng.standard_normal((3000, 64)))[0]
    v = np.linalg.qr(rng.standard_normal((64, 64)))[0]
    a1 = u * np.logspace(0, -4, 64) @ v
    check(np.hstack([a1, a1 @ rng.standard_normal((64, 64)) + 1e-11 * rng.standard_normal((3000, 64))]),
          elementwise=False)
