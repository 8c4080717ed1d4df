"""The BF16 GEMM's 64 x 64 LDS tiles and its K split over a block's waves at the
edges of tiles, K steps and vector loads, and the fused training pieces, against
numpy.  Products of BF16 values are exact in FP32 and FP32 sums of K terms are
within K 2^-24 of sum |a||b|, which is the tolerance."""
import ctypes

import numpy as np
import pytest

from quiqbox_amd import _lib

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def _bf16(a):
    t = torch.tensor(np.asarray(a, dtype=np.float32)).to(torch.bfloat16)
    return t.cuda(), t.float().numpy().astype(np.float64)


def _p(t):
    return ctypes.c_void_p(t.data_ptr())


def _check(C, ref, A, B, K):
    err = np.abs(C.cpu().numpy().astype(np.float64) - ref)
    assert np.all(err <= (K + 4) * 2.0 ** -24 * (np.abs(A) @ np.abs(B)) + 1e-30)


# (64, 64) tiles: one short, full, one over; K: one step of 8, a partial step of 32,
# the split's threshold (16 waves x 32) and one beside it; many tiles with long K
@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (63, 65, 8), (64, 64, 32), (65, 63, 33), (130, 225, 460),
                                   (464, 256, 511), (464, 256, 512), (33, 31, 1000), (1, 225, 4099), (900, 800, 530)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (1, 0), (0, 1), (1, 1)])
def test_gemm_tile_edges(M, N, K, ta, tb):
    rng = np.random.default_rng(M + N + K)
    dA, A = _bf16(rng.normal(size=(K, M) if ta else (M, K)))
    dB, B = _bf16(rng.normal(size=(N, K) if tb else (K, N)))
    C = torch.full((M, N), 7.0, device="cuda")
    _lib.check(_lib.load().qbx_gemm_bf16(ta, tb, M, N, K, 1.0, _p(dA), dA.shape[1], _p(dB), dB.shape[1], 0.0, _p(C),
                                         N, 0, None, None, None))
    A, B = A.T if ta else A, B.T if tb else B
    _check(C, A @ B, A, B, K)


def test_gemm_unaligned_operands_and_strides():
    """Sub-matrices: a base two bytes off 16-byte alignment and padded strides."""
    rng = np.random.default_rng(3)
    M, N, K = 70, 66, 600
    dA, A = _bf16(rng.normal(size=(M, K + 9)))
    dB, B = _bf16(rng.normal(size=(K, N + 7)))
    C = torch.zeros((M, N + 3), device="cuda")
    a, b = dA.view(-1)[1:], dB.view(-1)[3:]
    _lib.check(_lib.load().qbx_gemm_bf16(0, 0, M, N, K, 1.0, _p(a), K + 9, _p(b), N + 7, 0.0, _p(C), N + 3, 0, None,
                                         None, None))
    A, B = A[:, 1:K + 1], B[:, 3:N + 3]
    _check(C[:, :N], A @ B, A, B, K)
    assert torch.all(C[:, N:] == 0)


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (100, 256, 225), (65, 70, 256)])
def test_relu_back_epilogue(M, N, K):
    rng = np.random.default_rng(M)
    dA, A = _bf16(rng.normal(size=(M, K)))
    dB, B = _bf16(rng.normal(size=(N, K)))
    dH, H = _bf16(np.maximum(rng.normal(size=(M, N)), 0.0))
    C = torch.full((M, N), 7.0, device="cuda")
    Cb = torch.full((M, N), 7.0, device="cuda", dtype=torch.bfloat16)
    _lib.check(_lib.load().qbx_gemm_bf16_relu_back(M, N, K, _p(dA), K, _p(dB), K, _p(dH), _p(C), _p(Cb), N, None))
    _check(C, np.where(H > 0, A @ B.T, 0.0), A, B.T, K)
    assert torch.equal(Cb, C.to(torch.bfloat16))


@pytest.mark.parametrize("rows,cols", [(1, 1), (3, 225), (1000, 16), (65, 17), (4096, 33)])
def test_mse_mean_and_colsum(rows, cols):
    rng = np.random.default_rng(rows)
    Y, T = (rng.normal(size=(rows, cols)).astype(np.float32) for _ in range(2))
    rw = (rng.uniform(size=rows) > 0.2).astype(np.float32)
    cm = (rng.uniform(size=cols) > 0.2).astype(np.float32)
    d = [torch.tensor(v).cuda() for v in (Y, T, rw, cm)]
    dY, dYb = torch.zeros((rows, cols), device="cuda"), torch.zeros((rows, cols), dtype=torch.bfloat16, device="cuda")
    loss = torch.zeros(1, device="cuda")
    L = _lib.load()
    _lib.check(L.qbx_mlp_mse_mean(rows, cols, *(_p(x) for x in d), _p(dY), _p(dYb), _p(loss), None))
    w = rw[:, None].astype(np.float64) * cm / max(float(rw.sum()), 1.0)
    diff = Y.astype(np.float64) - T
    np.testing.assert_allclose(dY.cpu().numpy(), 2 * w * diff, rtol=1e-6, atol=1e-9)
    assert torch.equal(dYb, dY.to(torch.bfloat16))
    assert loss.item() == pytest.approx(float((w * diff ** 2).sum()), rel=1e-5, abs=1e-12)
    out = torch.full((cols,), 7.0, device="cuda")
    _lib.check(L.qbx_mlp_colsum(rows, cols, _p(d[0]), _p(out), None))
    bound = (rows + 1) * 2.0 ** -24 * np.abs(Y).astype(np.float64).sum(0)
    assert np.all(np.abs(out.cpu().numpy() - Y.astype(np.float64).sum(0)) <= bound + 1e-30)


def test_adam_multi_equals_single_tensors():
    rng = np.random.default_rng(1)
    sizes = [1, 255, 256, 257, 1000]
    new = lambda f: [torch.tensor(f(n).astype(np.float32)).cuda() for n in sizes]  # noqa: E731
    w, g = new(lambda n: rng.normal(size=n)), new(lambda n: rng.normal(size=n))
    m, v = new(np.zeros), new(np.zeros)
    wb = [torch.zeros(n, dtype=torch.bfloat16, device="cuda") if n % 2 else None for n in sizes]
    w2, m2, v2 = ([t.clone() for t in ts] for ts in (w, m, v))
    wb2 = [None if t is None else t.clone() for t in wb]
    L = _lib.load()
    arr = lambda ts: (ctypes.c_void_p * len(ts))(*[None if t is None else t.data_ptr() for t in ts])  # noqa: E731
    for step in (1, 2):
        _lib.check(L.qbx_mlp_adam_multi(len(sizes), (ctypes.c_int64 * len(sizes))(*sizes), arr(w), arr(m), arr(v),
                                        arr(g), arr(wb), 1e-2, 0.9, 0.999, 1e-8, step, None))
        for k, n in enumerate(sizes):
            _lib.check(L.qbx_mlp_adam(n, _p(w2[k]), _p(m2[k]), _p(v2[k]), _p(g[k]),
                                      None if wb2[k] is None else _p(wb2[k]), 1e-2, 0.9, 0.999, 1e-8, step, None))
    for a, b in ((w, w2), (m, m2), (v, v2)):
        assert all(torch.equal(x, y) for x, y in zip(a, b))
    assert all(x is None or torch.equal(x, y) for x, y in zip(wb, wb2))
    with pytest.raises(ValueError):
        _lib.check(L.qbx_mlp_adam_multi(17, None, None, None, None, None, None, 1e-2, 0.9, 0.999, 1e-8, 1, None))
