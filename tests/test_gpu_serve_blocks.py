"""The server's pinned request memory: blocks reused by requests of other sizes,
a burst larger than its 1 GiB (the rest in ordinary memory), and a rejected
request, each solution against the FP64 handle's (bar: 1e-9 relative at condition
numbers of a few, the mixed path being refined to working precision)."""
import numpy as np
import pytest
import torch

import rnp2_amd as R

pytestmark = pytest.mark.gpu


def solve(a, b):
    h = R.Handle()
    try:
        A = R.colmajor_empty(*a.shape, torch.float64)
        B = R.colmajor_empty(*b.shape, torch.float64)
        A.copy_(torch.from_numpy(a).cuda())
        B.copy_(torch.from_numpy(b).cuda())
        tau = torch.empty(a.shape[1], dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        h.gels(A, tau, B)
        h.synchronize()
        return B[:a.shape[1]].cpu().numpy()
    finally:
        h.close()


def test_blocks_are_reused_across_sizes():
    rng = np.random.default_rng(0)
    srv = R.Server(workers=2, mode=1)
    try:
        for burst in range(3):
            reqs = [(np.asfortranarray(rng.standard_normal((m, n))), np.asfortranarray(rng.standard_normal((m, q))))
                    for m, n, q in ((900, 300, 2), (80, 20, 1), (1500, 200, 5), (257, 60, 3), (700, 350, 1))]
            ids = [srv.submit(a, b)[1] for a, b in reqs]
            for (a, b), rid in zip(reqs, ids):
                x, info = srv.poll(rid)
                srv.release(rid)
                want = solve(a, b)
                assert info.status == 0 and np.abs(x - want).max() <= 1e-9 * np.abs(want).max()
    finally:
        srv.close()


def test_burst_beyond_the_pinned_memory():
    rng = np.random.default_rng(1)
    m, n = 8192, 1024  # 67 MB each: 20 of them pass 1 GiB
    a = np.asfortranarray(rng.standard_normal((m, n)))
    bs = [np.asfortranarray(rng.standard_normal((m, 1))) for _ in range(20)]
    srv = R.Server(workers=4, mode=0)
    try:
        ids = [srv.submit(a, b)[1] for b in bs]
        xs = [srv.poll(rid)[0] for rid in ids]
    finally:
        srv.close()
    want = solve(a, np.asfortranarray(np.hstack(bs)))
    assert np.abs(np.hstack(xs) - want).max() <= 1e-9 * np.abs(want).max()


def test_rejected_request_takes_no_memory():
    srv = R.Server(hbm_budget=1 << 20, workers=1, mode=1)
    try:
        a, b = np.ones((2000, 500)), np.ones((2000, 1))
        st, rid = srv.submit(a, b)
        assert st == R.RNPX_ERR_NOMEM
        assert srv.stats()["rejected"] == 1
    finally:
        srv.close()
