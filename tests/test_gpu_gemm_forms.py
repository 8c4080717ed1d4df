"""FP64 GEMM on both sides of the bounds where K is split over a block's waves: 256, 640
and 1536 tiles of 32 x 32 (and one more), K = 255, 256, 511 and 512, all four operand
orders, ragged edges, alpha and beta, against torch on the CPU.

Tolerance: rounding of a K-term sum whose partial sums, of terms below 1 with random
signs, stay around sqrt(K): K 2^-52 |alpha| sqrt(K)."""
import ctypes

import pytest

from quiqbox_amd import _lib

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


@pytest.mark.parametrize("tiles_m,tiles_n", [(16, 16), (257, 1), (32, 20), (641, 1), (48, 32), (1537, 1)])
@pytest.mark.parametrize("K", [255, 256, 511, 512])
def test_gemm_around_the_split_bounds(tiles_m, tiles_n, K):
    g = torch.Generator().manual_seed(tiles_m + K)
    M, N = 32 * tiles_m - 7, 32 * tiles_n - 3
    A = torch.rand((M, K), generator=g, dtype=torch.float64) * 2 - 1
    B = torch.rand((K, N), generator=g, dtype=torch.float64) * 2 - 1
    C = torch.rand((M, N), generator=g, dtype=torch.float64) * 2 - 1
    ref = 1.25 * (A @ B) - 0.5 * C
    tol = 1.25 * K * 2.0 ** -52 * K ** 0.5
    for ta in (0, 1):
        for tb in (0, 1):
            a = (A.T if ta else A).contiguous().cuda()
            b = (B.T if tb else B).contiguous().cuda()
            c = C.cuda()
            _lib.check(_lib.load().qbx_gemm_f64(ta, tb, M, N, K, 1.25, _p(a), a.shape[1], _p(b), b.shape[1], -0.5,
                                                _p(c), N, None))
            torch.cuda.synchronize()
            assert float((c.cpu() - ref).abs().max()) < tol, (ta, tb)
