"""J's ket sums in pair order (bases of 64 functions and more) against the
contraction of the dense tensor, whose kernels do not use them: s, p and d shells,
shells with absent components (lone p_x and d_xy functions), one and two density
sets, K-row kernels and one-wave-per-chunk kernels, and a basis one function below
the bound.

Tolerance: both sides contract the same integrals; an element sums 2 n^2 = 10^4
products, each below 1 in size, in FP64: 10^4 roundings of 1.1e-16 on partial sums
below 10, 1e-11.
"""
import os

import numpy as np
import pytest

import quiqbox_amd as qb
from helpers import random_spd_basis
from quiqbox_amd.engine import Context

pytestmark = pytest.mark.gpu


def _context(**env):
    old = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    try:
        return Context(0)
    finally:
        for k, v in old.items():
            if v is None:
                del os.environ[k]
            else:
                os.environ[k] = v


def _basis(n):
    bs = random_spd_basis(71, n_atoms=6, box=5.0, nprim=(3, 2, 1))[1]
    rng = np.random.default_rng(72)
    lone = [(1, 0, 0), (0, 0, 1), (1, 1, 0), (0, 1, 1), (0, 0, 0), (0, 0, 2), (0, 1, 0)]
    for ijk in lone[:n - len(bs)]:
        bs.append(qb.genGaussTypeOrb(tuple(rng.uniform(0, 5, 3)), [0.4, 1.9], [0.7, 0.4], ijk, outerRenormalize=True))
    return bs


@pytest.mark.parametrize("n,nset,rows", [(67, 1, "1"), (67, 2, "1"), (67, 2, "0"), (64, 1, "1"), (63, 1, "1")])
def test_pair_order_ket_sums_match_dense(n, nset, rows):
    bs = _basis(n)
    ctx = _context(QBX_JK_ROWS=rows)
    gb = qb.GPUBasis(bs, ctx=ctx)
    assert gb.n == n
    E = gb.eri_dense()
    rng = np.random.default_rng(n + nset)
    DJ = rng.uniform(-0.1, 0.1, (nset, n, n))
    DK = rng.uniform(-0.1, 0.1, (nset, n, n))
    DJ, DK = DJ + DJ.transpose(0, 2, 1), DK + DK.transpose(0, 2, 1)
    print("[gpu-test] n %d, %d sets, K rows %s" % (n, nset, rows), flush=True)
    G = gb.jk(DJ, DK, 0.0) if nset > 1 else [gb.jk(DJ[0], DK[0], 0.0)]
    M = E.reshape(n * n, n * n)
    X = E.transpose(0, 2, 1, 3).reshape(n * n, n * n)
    for s in range(nset):
        R = (M @ DJ[s].ravel() - X @ DK[s].ravel()).reshape(n, n)
        err = float(np.abs(G[s] - R).max())
        print("[gpu-test]   set %d: max|dG| %.3e (max|G| %.3e)" % (s, err, float(np.abs(R).max())), flush=True)
        assert err < 1e-11
    del gb
    ctx.close()
