"""Handles with a memory budget: a call that fits panel by panel is not refused
because the block kernel's buffers took the room, nothing is refused after the
matrix has been touched, and the budget holds for the whole handle.  Results
against the FP64 oracle's bars (residual and orthogonality <= 10 n eps)."""
import numpy as np
import pytest
import torch

import rnp2_amd as R
from metrics import orth_error, qr_residual

pytestmark = pytest.mark.gpu


def dev(a):
    t = R.colmajor_empty(a.shape[0], a.shape[1], torch.float64)
    t.copy_(torch.from_numpy(np.ascontiguousarray(a)).cuda())
    torch.cuda.synchronize()
    return t


def factor(h, a):
    A, tau = dev(a), torch.empty(min(a.shape), dtype=torch.float64, device="cuda")
    h.geqrf(A, tau)
    h.synchronize()
    return A.cpu().numpy(), tau.cpu().numpy()


def good(a, f):
    k = min(a.shape)
    q = R.generateq(f[0][:, :k], f[1], n=k)
    assert qr_residual(a, q, np.triu(f[0][:k])) <= 10 and orth_error(q) <= 10


@pytest.mark.parametrize("m,n", [(700, 500), (4000, 128), (8192, 100), (8192, 1024), (16384, 300), (3000, 3000)])
def test_factor_at_the_panel_routes_need(m, n):
    a = np.random.default_rng(m + n).standard_normal((m, n))
    h = R.Handle()
    h.set_tuning(panel=2)
    factor(h, a)
    need = h.workspace_bytes()
    h.close()
    for budget in (need, int(1.3 * need), 2 * need):
        h = R.Handle(budget)
        good(a, factor(h, a))
        assert h.workspace_bytes() <= budget
        good(a, factor(h, a))  # and again with the buffers there
        h.close()


def test_refusal_leaves_the_matrix():
    a = np.random.default_rng(0).standard_normal((4096, 512))
    h = R.Handle(8 << 20)
    A, tau = dev(a), torch.empty(512, dtype=torch.float64, device="cuda")
    with pytest.raises(R.RnpxError):
        h.geqrf(A, tau)
    h.synchronize()
    assert np.array_equal(A.cpu().numpy(), a)
    h.close()


def test_block_buffers_make_room_for_the_next_call():
    """Factor of a tall matrix by blocks, then the solve's and MultQ's buffers."""
    m, n = 16384, 256
    rng = np.random.default_rng(1)
    a, b = rng.standard_normal((m, n)), rng.standard_normal((m, 300))
    h = R.Handle()
    fa, tau = factor(h, a)
    need = h.workspace_bytes()
    h.close()
    h = R.Handle(need)
    dA, dtau = dev(a), torch.empty(n, dtype=torch.float64, device="cuda")
    h.geqrf(dA, dtau)
    C = dev(b)
    h.ormqr("L", "C", dA, dtau, C)
    h.synchronize()
    h2 = R.Handle()
    C2 = dev(b)
    h2.ormqr("L", "C", dA, dtau, C2)
    h2.synchronize()
    assert float((C - C2).norm()) <= 1e-13 * float(C2.norm())
    assert h.workspace_bytes() <= need
    h.close()
    h2.close()


@pytest.mark.parametrize("nq,k,n", [(8192, 64, 256), (20000, 300, 100)])
def test_multq_at_one_blocks_need(nq, k, n):
    """One 64-column block at a time: V, its Gram in 256-row slices (at most 64), T,
    W, Z and W's partial sums over 128-row slices (at most 64), with the 1/8 that
    buffers grow by."""
    ks = min(1024 // ((n + 127) // 128), min(nq // 128, 64))
    need = 8 * (nq * 64 + 2 * 64 * 64 + min(64, nq // 256) * 64 * 64 + (2 + ks) * 64 * n)
    rng = np.random.default_rng(k)
    a, c = rng.standard_normal((nq, k)), rng.standard_normal((nq, n))
    h0 = R.Handle()
    A, tau, C0, C = dev(a), torch.empty(k, dtype=torch.float64, device="cuda"), dev(c), dev(c)
    h0.geqrf(A, tau)
    h0.ormqr("L", "C", A, tau, C0)
    h0.synchronize()
    h0.close()
    h = R.Handle(need + need // 8 + 4096)
    h.ormqr("L", "C", A, tau, C)
    h.synchronize()
    h.close()
    assert float((C - C0).norm()) <= 1e-13 * float(C0.norm())
