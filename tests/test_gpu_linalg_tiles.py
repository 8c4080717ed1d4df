"""The FP64 GEMM with K split over a block's waves and the tiled purification, at
the edges of their tiles, K steps and vector loads."""
import ctypes

import numpy as np
import pytest

import quiqbox_amd as qb
from quiqbox_amd import _lib

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


# K: the threshold of the split (256), one beside it, whole and partial 16-steps;
# M, N: below, at and above the 32 x 32 tile; strides and bases off 16 bytes
@pytest.mark.parametrize("M,N,K", [(1, 1, 256), (31, 33, 255), (32, 32, 257), (33, 65, 271), (100, 7, 272), (5, 64, 1000)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
@pytest.mark.parametrize("pad,off", [(0, 0), (1, 0), (2, 1)])
def test_gemm_split_edges(M, N, K, ta, tb, pad, off):
    rng = np.random.default_rng(M + N + K + pad)
    a, b = ((K, M) if ta else (M, K)), ((N, K) if tb else (K, N))
    A, B = rng.standard_normal(a), rng.standard_normal(b)
    C0 = rng.standard_normal((M, N))

    def place(X):
        t = torch.zeros(X.shape[0] * (X.shape[1] + pad) + off, dtype=torch.float64, device="cuda")
        v = t[off:].view(X.shape[0], X.shape[1] + pad)
        v[:, :X.shape[1]] = torch.tensor(X, device="cuda")
        return v

    dA, dB, dC = place(A), place(B), place(C0)
    _lib.check(_lib.load().qbx_gemm_f64(ta, tb, M, N, K, 1.5, _p(dA), a[1] + pad, _p(dB), b[1] + pad, -0.5, _p(dC),
                                        N + pad, None))
    A, B = A.T if ta else A, B.T if tb else B
    # rounding of a K-term sum
    bound = (K + 4) * 2.0 ** -53 * (1.5 * np.abs(A) @ np.abs(B) + np.abs(C0))
    assert np.all(np.abs(dC[:, :N].cpu().numpy() - (1.5 * A @ B - 0.5 * C0)) <= bound)


# sizes around the 32 x 32 tiles; no, some and all levels occupied
@pytest.mark.parametrize("n,nocc", [(1, 1), (2, 1), (31, 7), (32, 16), (33, 32), (64, 1), (97, 50), (130, 129)])
def test_purified_density(n, nocc):
    rng = np.random.default_rng(n)
    Q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    e = np.concatenate([rng.uniform(-5.0, -1.0, nocc), rng.uniform(0.5, 4.0, n - nocc)])
    U = np.linalg.qr(rng.standard_normal((n, n)))[0]
    w = np.exp(rng.uniform(-0.5, 0.5, n))
    X, Xi = (U * w) @ U.T, (U / w) @ U.T
    F = Xi @ ((Q * e) @ Q.T) @ Xi
    D, it, idem = qb.default_context().purified_density(X, F, nocc)
    O = X @ Q[:, :nocc]
    # the projector settles to rounding: error of X and F times their condition (w within e^1)
    assert np.max(np.abs(D - O @ O.T)) < 1e-11
    assert it > 0 and idem < 1e-9 * max(1, n)


def test_purification_reports_a_missing_gap():
    n = 40
    rng = np.random.default_rng(4)
    Q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    e = np.concatenate([np.full(10, -1.0), np.zeros(4), np.full(26, 1.0)])   # four degenerate levels across the Fermi level
    with pytest.raises(_lib.QbxError):
        qb.default_context().purified_density(np.eye(n), (Q * e) @ Q.T, 12, max_iter=60)
    with pytest.raises(_lib.QbxError):
        e = np.linspace(-1.0, 1.0, n)
        qb.default_context().purified_density(np.eye(n), (Q * e) @ Q.T, 12, max_iter=3)
