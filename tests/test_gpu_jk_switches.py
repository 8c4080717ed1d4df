"""Fock builds of contracted water against builds that share none of their lists and
kernels: every switch off (QBX_JK_ROWS, QBX_KET_BUCKETS, QBX_STAGED_SPLIT, QBX_XCD_LOCAL=0)
in a fresh context, so one wave a 64-ket chunk over one Schwarz-ordered list, with all sums
straight to J and K.  One and two density sets, mixed precision, a density-screened
increment, and a converged SCF.

Tolerances: FP64 the same integrals in another order, 1e-12 of the largest |G|; mixed the
FP32 integrals (each below the 1e-5 cut, within about 100 roundings of 2^-24), at most n^2
= 2500 of them with weights up to 0.3, 1e-7; the screened builds drop quartets below 1e-12
in either order alike."""
import os

import numpy as np
import pytest

import oracle
import quiqbox_amd as qb
from quiqbox_amd.engine import Context
from quiqbox_amd.systems import water_box

pytestmark = pytest.mark.gpu
OFF = ("QBX_JK_ROWS", "QBX_KET_BUCKETS", "QBX_STAGED_SPLIT", "QBX_XCD_LOCAL")


def _off_context():
    old = {k: os.environ.get(k) for k in OFF}
    os.environ.update({k: "0" for k in OFF})
    try:
        return Context(0)
    finally:
        for k, v in old.items():
            if v is None:
                del os.environ[k]
            else:
                os.environ[k] = v


@pytest.mark.parametrize("nset,precision,screen", [(1, qb.QBX_PREC_FP64, 0.0), (2, qb.QBX_PREC_FP64, 0.0),
                                                   (1, qb.QBX_PREC_MIXED, 0.0), (2, qb.QBX_PREC_MIXED, 0.0),
                                                   (1, qb.QBX_PREC_FP64, 1e-12)])
def test_water_dimer_against_all_switches_off(nset, precision, screen):
    bs = water_box(2, 11, basis="cc-pVDZ")[1]
    ctx, off = Context(0), _off_context()
    for c in (ctx, off):
        c.set_density_screening(screen)
    a, b = qb.GPUBasis(bs, ctx=ctx), qb.GPUBasis(bs, ctx=off)
    rng = np.random.default_rng(2)
    D = rng.uniform(-0.1, 0.1, (2, nset, a.n, a.n))
    D = (D + D.transpose(0, 1, 3, 2)) * (1e-3 if screen else 1.0)
    G, R = a.jk(D[0], D[1], 1e-12, precision), b.jk(D[0], D[1], 1e-12, precision)
    scale = float(np.abs(R).max()) if screen else max(1.0, float(np.abs(R).max()))
    err = float(np.abs(G - R).max())
    print("[gpu-test] %d sets, precision %d, screen %g: max|dG| %.2e (max|G| %.2e)" % (nset, precision, screen, err,
                                                                                     scale), flush=True)
    assert err < (1e-12 if precision == qb.QBX_PREC_FP64 else 1e-7) * scale
    if not screen and precision == qb.QBX_PREC_FP64:
        E = oracle.Basis(a.flat.as_dict()).eri_dense()
        for s in range(nset):
            assert np.abs(G[s] - oracle.gcore(E, D[0][s], D[1][s])).max() < 1e-10


def test_water_trimer_scf_against_all_switches_off():
    nuc, bs = water_box(3, 21, basis="cc-pVDZ")
    cfg = qb.HFconfig(initial="CoreH", strategy=qb.SCFconfig(("ADIIS", "DIIS"), (1e-4, 1e-10)))
    r = qb.runHartreeFock(nuc, qb.GPUBasis(bs), cfg, printInfo=False)
    s = qb.runHartreeFock(nuc, qb.GPUBasis(bs, ctx=_off_context()), cfg, printInfo=False)
    print("[gpu-test] E %.12f, switches off %.12f" % (r.energy[0], s.energy[0]), flush=True)
    assert r.converged and s.converged
    assert abs(r.energy[0] - s.energy[0]) < 1e-9
