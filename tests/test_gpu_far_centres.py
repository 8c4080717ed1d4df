"""Centres so far apart that the Boys argument p R^2 overflows to infinity: F_m is 0
there, and nothing else may change.  A nucleus and an s function at 1e170 bohr beside an
s/p/d cluster at the origin, against the cluster alone: nuclear attraction, dense tensor,
Fock matrices through the K-row kernels and the one-wave-per-chunk kernels, mixed too.

Tolerances: the same integrals, summed in another order by atomics: 1e-12 of the largest
element; the nuclear matrix (each element one wave's sum, to which the far nucleus adds
zeros) within 1e-13 of its largest, since the lanes hold other items."""
import os

import numpy as np
import pytest

import quiqbox_amd as qb
from helpers import random_spd_basis
from quiqbox_amd.engine import Context

pytestmark = pytest.mark.gpu
FAR = (1e170, 0.0, 0.0)


def _bases(ctx):
    bs = random_spd_basis(4, n_atoms=3)[1]
    far = qb.genGaussTypeOrb(FAR, [1.1, 0.4], [0.6, 0.5], (0, 0, 0))
    return qb.GPUBasis(bs, ctx=ctx), qb.GPUBasis(bs + [far], ctx=ctx)


@pytest.mark.parametrize("rows", ["1", "0"])
def test_far_function(rows):
    old = os.environ.get("QBX_JK_ROWS")
    os.environ["QBX_JK_ROWS"] = rows
    try:
        ctx = Context(0)
    finally:
        if old is None:
            del os.environ["QBX_JK_ROWS"]
        else:
            os.environ["QBX_JK_ROWS"] = old
    near, both = _bases(ctx)
    n = near.n
    rng = np.random.default_rng(2)
    D = rng.uniform(-0.1, 0.1, (n + 1, n + 1))
    D = D + D.T
    D0 = np.ascontiguousarray(D[:n, :n])
    for precision, tol in ((qb.QBX_PREC_FP64, 1e-12), (qb.QBX_PREC_MIXED, 1e-7)):
        G = both.jk(2 * D, D, 0.0, precision)
        R = near.jk(2 * D0, D0, 0.0, precision)
        scale = max(1.0, float(np.abs(R).max()))
        assert np.all(np.isfinite(G))
        assert np.abs(G[:n, :n] - R).max() < tol * scale
        assert np.all(G[:n, n] == 0.0)
    E, E0 = both.eri_dense(), near.eri_dense()
    assert np.all(np.isfinite(E))
    assert np.abs(E[:n, :n, :n, :n] - E0).max() < 1e-12 * np.abs(E0).max()
    assert np.all(E[:n, :n, n, n] == 0.0) and E[n, n, n, n] > 0.0
    del near, both
    ctx.close()


def test_far_nucleus():
    near = _bases(None)[0]
    Z, R = [1.0, 8.0], [[0.1, 0.2, 0.3], [1.5, -0.4, 0.2]]
    V0 = near.nuclear(Z, R)
    V = near.nuclear(Z + [3.0], R + [list(FAR)])
    assert np.all(np.isfinite(V))
    assert np.abs(V - V0).max() < 1e-13 * np.abs(V0).max()
