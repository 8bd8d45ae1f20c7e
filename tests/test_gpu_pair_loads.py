"""The real MFMA products' pair loads at every alignment: operands inside a
larger buffer (odd offset, odd leading dimension), extents of one to three and
odd extents along the pairs, against numpy.  NaN outside the operands shows a
pair read past an extent.  Tolerance: the reduction's rounding,
|error| <= 2 k eps (|A| |B|) + 4 eps |C| per entry."""
import numpy as np
import pytest
import torch

import rnp2_amd as R

pytestmark = pytest.mark.gpu
EPS = np.finfo(np.float64).eps


def dev_inside(x, off, pad):
    """x at (off, 0) of a NaN-filled column-major buffer of off + rows + pad rows."""
    r, c = x.shape
    big = R.colmajor_empty(r + off + pad, c, torch.float64)
    big.fill_(float("nan"))
    v = big[off:off + r, :]
    v.copy_(torch.from_numpy(np.ascontiguousarray(x)).to("cuda"))
    torch.cuda.synchronize()
    return v


@pytest.mark.parametrize("ta", ["N", "T"])
@pytest.mark.parametrize("m,n,k", [(1, 5, 1), (2, 6, 3), (3, 5, 2), (65, 7, 17), (129, 65, 33), (64, 64, 15),
                                   (1931, 77, 128), (128, 131, 1931), (127, 129, 31)])
@pytest.mark.parametrize("off,pad", [(0, 0), (1, 0), (1, 1), (0, 1)])
def test_products_at_any_alignment(ta, m, n, k, off, pad):
    rng = np.random.default_rng(m * 7 + n * 3 + k)
    a = rng.standard_normal((m, k) if ta == "N" else (k, m))
    b, c = rng.standard_normal((k, n)), rng.standard_normal((m, n))
    opa = a if ta == "N" else a.T
    h = R.Handle()
    try:
        for alpha, beta in ((1.0, 0.0), (-1.0, 1.0)):
            A, B, C = (dev_inside(x, off, pad) for x in (a, b, c))
            h.gemm(ta, "N", alpha, A, B, beta, C)
            h.synchronize()
            got = C.cpu().numpy()
            bound = 2 * k * EPS * (np.abs(opa) @ np.abs(b)) + 4 * EPS * np.abs(c)
            assert (np.abs(got - (alpha * (opa @ b) + beta * c)) <= bound).all()
    finally:
        h.close()
