"""J/K tasks of uneven contractions: ket lists that run over several buckets of
primitive-pair counts (merged where more than ten counts occur), chunks of heavy
pairs cut into parts of the bra's primitive pairs (part lengths that do not
divide the count), staged and twin classes, against the one-wave-per-chunk
kernels over a single Schwarz-ordered list (QBX_JK_ROWS=0, QBX_KET_BUCKETS=0,
QBX_TWINS=0).

Tolerances.  FP64: the same integrals summed in another order, 1e-12 of the
largest |G|.  Mixed: the FP32 integrals are below the 1e-5 cut, each within about
100 roundings of 2^-24 (6e-11); a G element sums at most n^2 = 3721 of them with
weights up to 0.2: 5e-8, so 1e-7.
"""
import os

import numpy as np
import pytest

import quiqbox_amd as qb
from helpers import random_spd_basis
from quiqbox_amd.engine import Context

pytestmark = pytest.mark.gpu


def _plain_context():
    env = {"QBX_JK_ROWS": "0", "QBX_KET_BUCKETS": "0", "QBX_TWINS": "0"}
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


def _basis(kind):
    if kind == "uneven":      # 1 .. 169 primitive pairs
        sets = [(1, 13, 2), (7, 5, 1), (13, 1, 3), (2, 3, 5), (11, 2, 1), (5, 7, 2)]
    else:                     # one bucket of 49 pairs, a few chunks
        sets = [(7, 7, 7)] * 3
    bs = []
    for k, nprim in enumerate(sets):
        bs += random_spd_basis(50 + k, n_atoms=1, box=3.0, nprim=nprim)[1]
    return bs


@pytest.mark.parametrize("kind,nset,precision,thr",
                         [("uneven", 1, qb.QBX_PREC_FP64, 0.0), ("uneven", 2, qb.QBX_PREC_FP64, 1e-9),
                          ("uneven", 1, qb.QBX_PREC_MIXED, 1e-10), ("even", 1, qb.QBX_PREC_FP64, 1e-10),
                          ("even", 2, qb.QBX_PREC_MIXED, 0.0)])
def test_task_parts_match_plain_lists(kind, nset, precision, thr):
    bs = _basis(kind)
    gb = qb.GPUBasis(bs)
    ctx = _plain_context()
    plain = qb.GPUBasis(bs, ctx=ctx)
    rng = np.random.default_rng(8)
    n = gb.n
    D = []
    for _ in range(2):
        a = rng.uniform(-0.1, 0.1, (nset, n, n))
        D.append(a + a.transpose(0, 2, 1))
    DJ, DK = (D[0][0], D[1][0]) if nset == 1 else D
    print("[gpu-test] %s: n %d, %d sets, precision %d, thr %g" % (kind, n, nset, precision, thr), flush=True)
    G = gb.jk(DJ, DK, thr, precision)
    R = plain.jk(DJ, DK, thr, precision)
    scale = max(1.0, float(np.abs(R).max()))
    err = float(np.abs(G - R).max())
    print("[gpu-test]   max|dG| %.3e (max|G| %.3e)" % (err, scale), flush=True)
    assert err < (1e-12 if precision == qb.QBX_PREC_FP64 else 1e-7) * scale
    del plain
    ctx.close()
