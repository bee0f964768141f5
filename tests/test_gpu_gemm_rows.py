"""gsdft_dgemm with even leading dimensions and 16-byte aligned operands (the LDS-DMA path) at row
counts around the 32, 64, 96 and 128 rows a tile may have, against numpy. Bar: a K-term sum's
round-off, K 2^-53 times the largest sum of magnitudes (a few times sqrt(K) is seen)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = [1, 31, 32, 33, 63, 64, 65, 81, 96, 97, 127, 128, 129, 159, 160, 161, 192, 193, 255, 256, 257]


@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("m", ROWS)
def test_dgemm_row_tiles(g, cuda, ta, tb, m):
    from gs_dft_amd import _lib
    n, k = 150, 83
    rng = np.random.default_rng(1000 * m + 2 * ta + tb)
    even = lambda v: v + v % 2
    ar, ac = (k, m) if ta else (m, k)
    br, bc = (n, k) if tb else (k, n)
    lda, ldb, ldc = even(ar) + 2, even(br), m + 1
    A_buf, B_buf, C_buf = (rng.normal(size=s) for s in (lda * ac, ldb * bc, ldc * n))
    A, B = A_buf.reshape(ac, lda).T[:ar], B_buf.reshape(bc, ldb).T[:br]
    opA, opB = (A.T if ta else A), (B.T if tb else B)
    print(f"[gemm rows] ta={ta} tb={tb} m={m}", flush=True)
    bar = k * 2.0 ** -53 * (np.abs(opA) @ np.abs(opB)).max()
    Ad, Bd, Cd = (torch.tensor(x, device="cuda") for x in (A_buf, B_buf, C_buf))
    _lib.check(_lib.lib().gsdft_dgemm(ta, tb, m, n, k, 1.0, _lib.ptr(Ad), lda, _lib.ptr(Bd), ldb,
                                      0.0, _lib.ptr(Cd), ldc, _lib.stream()), "dgemm")
    out = Cd.cpu().numpy().reshape(n, ldc)
    assert np.abs(out.T[:m] - opA @ opB).max() < bar
    assert np.array_equal(out[:, m:], C_buf.reshape(n, ldc)[:, m:])
