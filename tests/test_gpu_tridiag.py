"""Fock solves through the persistent tridiagonalization (orders of 96 and more):
orders around wave, block and two-elements-a-thread edges and one below the bound,
dense, block-diagonal, diagonal and clustered matrices, small and large scales, and
three contexts at once.

Tolerance: Householder reduction and divide and conquer are backward stable with an
error of a small multiple of n eps |F|; 8 n eps |F|_2 for residual and eigenvalues,
8 n eps for orthogonality.
"""
import threading

import numpy as np
import pytest

from quiqbox_amd.engine import Context, default_context

pytestmark = pytest.mark.gpu


def _matrix(kind, n):
    rng = np.random.default_rng(n)
    A = rng.standard_normal((n, n))
    F = A + A.T
    if kind == "blocks":
        for k in range(0, n, 37):
            F[k:k + 37, k + 37:] = 0.0
            F[k + 37:, k:k + 37] = 0.0
    elif kind == "diagonal":
        F = np.diag(rng.standard_normal(n))
    elif kind == "clustered":
        Q = np.linalg.qr(A)[0]
        F = (Q * np.repeat([-1.0, 0.5, 0.5 + 1e-13, 2.0], (n + 3) // 4)[:n]) @ Q.T
        F = 0.5 * (F + F.T)
    elif kind == "small":
        F = F * 1e-150
    elif kind == "large":
        F = F * 1e120
    return F


def _check(ctx, F):
    n = len(F)
    C, e, D = ctx.fock_solve(np.eye(n), F, n // 2)
    eps, norm = np.finfo(float).eps, np.linalg.norm(F, 2)
    res = np.abs(F @ C - C * e).max() / norm
    orth = np.abs(C.T @ C - np.eye(n)).max()
    val = np.abs(np.sort(e) - np.linalg.eigvalsh(F)).max() / norm
    print("[gpu-test] n %d: residual %.1e, orthogonality %.1e, eigenvalues %.1e (of |F|)" % (n, res, orth, val),
          flush=True)
    assert np.all(np.diff(e) >= 0)
    assert max(res, val, orth) < 8 * n * eps


@pytest.mark.parametrize("kind,n", [("dense", n) for n in (95, 96, 97, 128, 129, 321, 640, 1025)] +
                         [("blocks", 150), ("diagonal", 100), ("clustered", 200), ("small", 130), ("large", 130)])
def test_fock_solve_eigenpairs(kind, n):
    _check(default_context(), _matrix(kind, n))


def test_three_contexts_at_once():
    done = []

    def work(n):
        ctx = Context(0)
        for _ in range(3):
            _check(ctx, _matrix("dense", n))
        ctx.close()
        done.append(n)

    ts = [threading.Thread(target=work, args=(n,)) for n in (200, 300, 400)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert sorted(done) == [200, 300, 400]
