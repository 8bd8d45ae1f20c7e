"""MultQ and GenerateQ at the edges of their block plan (T factors formed for
all blocks before the first is applied: 128-column real and 64-column complex
blocks of two 64-column leaves, a narrower last block, 2048-column chunks of
V; the narrow plan of a handle with a memory budget) against torch's products
of the same reflectors on the host.  Unit reflectors tau = 2/(v^H v), so each
block's rounding is bounded by a few eps times the norm: |error|_F <=
10 k eps |C|_F with k reflectors."""
import numpy as np
import pytest
import torch

import rnp2_amd as R

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def stored(q, k, dt, seed):
    g = torch.Generator().manual_seed(seed)
    a = torch.randn(q, k, dtype=dt, generator=g)
    low = a.tril(-1)
    nrm = low.abs().square().sum(0).sqrt()
    want = torch.where(nrm > 0, 0.98, 0.0).to(torch.float64)
    low = low * (want / nrm.clamp_min(1e-30))
    return low + a.triu(), (2.0 / (1.0 + want.square())).to(dt)


def dev(x):
    t = R.colmajor_empty(x.shape[0], x.shape[1], x.dtype)
    t.copy_(x.cuda())
    torch.cuda.synchronize()
    return t


# k across the widths' edges: one leaf, one block, a block and one column,
# a block and more than a leaf, several blocks; 2112 and 2050: two chunks of V
@pytest.mark.parametrize("dt", [torch.float64, torch.complex128])
@pytest.mark.parametrize("q,k", [(40, 1), (70, 63), (130, 64), (131, 65), (300, 128), (301, 129), (500, 193),
                                 (517, 320), (2300, 2112)])
@pytest.mark.parametrize("side,trans", [("L", "N"), ("L", "C"), ("R", "N"), ("R", "C")])
@pytest.mark.parametrize("budget", [0, 64 << 20])
def test_multq_plan_edges(dt, q, k, side, trans, budget):
    if q > 600 and (budget or (side, trans) in (("L", "N"), ("R", "C"))):
        pytest.skip("the large case runs one direction per side, unbudgeted")
    a, tau = stored(q, k, dt, q + k)
    c = torch.randn((q, 37) if side == "L" else (37, q), dtype=dt, generator=torch.Generator().manual_seed(1))
    want = torch.ormqr(a, tau, c, side == "L", trans == "C")
    h = R.Handle(budget)
    try:
        C = dev(c)
        h.ormqr(side, trans, dev(a), tau.cuda(), C)
        h.synchronize()
        assert float((C.cpu() - want).norm()) <= 10 * k * EPS * float(c.norm())
    finally:
        h.close()


@pytest.mark.parametrize("dt", [torch.float64, torch.complex128])
@pytest.mark.parametrize("m,n,k", [(40, 1, 1), (130, 70, 64), (300, 129, 129), (301, 200, 128), (517, 330, 320),
                                   (130, 5, 0)])
@pytest.mark.parametrize("budget", [0, 64 << 20])
def test_generateq_plan_edges(dt, m, n, k, budget):
    a, tau = stored(m, max(k, 1), dt, m + n)
    full = torch.full((m, n), float("nan"), dtype=dt)
    full[:, :k] = a[:, :k]
    want = torch.ormqr(a, tau, torch.eye(m, n, dtype=dt), True, False) if k else torch.eye(m, n, dtype=dt)
    h = R.Handle(budget)
    try:
        A = dev(full)
        h.orgqr(A, tau.cuda(), n=n, k=k)
        h.synchronize()
        assert float((A.cpu() - want).norm()) <= 10 * max(k, 1) * EPS * n ** 0.5
    finally:
        h.close()


@pytest.mark.parametrize("dt,q,k", [(torch.float64, 32768, 1500), (torch.complex128, 20000, 1000)])
def test_multq_copy_of_v_is_bounded(dt, q, k):
    """256 MB of V at a time, whatever the number of reflectors: chunks of 1024
    and 832 columns here, in both directions."""
    a, tau = stored(q, k, dt, q + k)
    A, tau = dev(a), tau.cuda()
    C = dev(torch.randn(q, 5, dtype=dt, generator=torch.Generator().manual_seed(1)))
    C0 = C.clone()
    torch.cuda.synchronize()
    h = R.Handle()
    try:
        h.ormqr("L", "C", A, tau, C)
        h.ormqr("L", "N", A, tau, C)
        h.synchronize()
        assert float((C - C0).norm()) <= 20 * k * EPS * float(C0.norm())
        vbuf = 256 << 20
        assert h.workspace_bytes() <= vbuf + vbuf // 8 + (64 << 20)  # V with its headroom; Grams, T, partial sums
    finally:
        h.close()
