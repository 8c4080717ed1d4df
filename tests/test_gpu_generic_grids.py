"""More quartets with an f shell than one grid holds (2^32 threads, 16,777,215 blocks of
256): one f shell and 323 contracted s shells give 16,901,298 (fs|ss) quartets, in two
launches.  J of a density with a few nonzero elements against sums of the oracle's
integrals: four s-s elements, which every (fs| bra meets, and the f-s elements of the
pair with the smallest Schwarz bound, whose quartets end the list."""
import os

import numpy as np
import pytest

import oracle
import quiqbox_amd as qb
from quiqbox_amd.basis import subshellXYZs

pytestmark = pytest.mark.gpu
THREADS = max(1, min(16, os.cpu_count() or 1))


def test_fock_build_over_two_grids():
    rng = np.random.default_rng(17)
    ns = 323
    cen = rng.uniform(-1.8, 1.8, (ns, 3))
    bs = [qb.genGaussTypeOrb((0.0, 0.0, 0.0), [0.6], [qb.get3DimPGTOrbNormFactor(0.6, ijk)], ijk)
          for ijk in subshellXYZs(3)]
    for c in cen:
        x = np.exp(rng.uniform(np.log(0.3), np.log(1.2), 2))
        w = rng.uniform(0.2, 0.6, 2)
        bs.append(qb.genGaussTypeOrb(tuple(c), list(x), [a * qb.get3DimPGTOrbNormFactor(e, (0, 0, 0))
                                                         for a, e in zip(w, x)], (0, 0, 0)))
    assert ns * ns * (ns + 1) // 2 > (2 ** 32 - 1) // 256
    gb = qb.GPUBasis(bs)
    ob = oracle.Basis(gb.flat.as_dict())
    n = gb.n
    # the f-s pair with the smallest bound, by its diagonal integrals
    f = np.arange(10)
    s = np.arange(10, n)
    q = np.array([(a, b, a, b) for b in s for a in f], dtype=np.int32)
    bound = ob.eri_list(q, threads=THREADS).reshape(ns, 10).max(1)
    last = 10 + int(np.argmin(bound))
    pairs = [(10, 10), (40, 12), (200, 199), (n - 1, 57)] + [(last, int(a)) for a in f]
    D = np.zeros((n, n))
    J = np.zeros((n, n))
    iu, ju = np.tril_indices(n)
    for k, l in pairs:
        w = float(rng.uniform(0.5, 1.5)) * (1.0 if l >= 10 else 10.0)
        D[k, l] = D[l, k] = w
        v = ob.eri_list(np.stack([iu, ju, np.full_like(iu, k), np.full_like(iu, l)], axis=1).astype(np.int32),
                        threads=THREADS)
        J[iu, ju] += (1.0 if k == l else 2.0) * w * v
    J[ju, iu] = J[iu, ju]
    print("[gpu-test] %d functions, Fock build" % n, flush=True)
    G = gb.jk(D, np.zeros_like(D), 0.0)
    err = float(np.abs(G - J).max())
    print("[gpu-test]   max|G - J| %.3e (max|J| %.2f, smallest f-s bound %.1e)" % (err, np.abs(J).max(), bound.min()),
          flush=True)
    assert bound.min() > 1e-8
    assert err < 1e-11 * max(1.0, float(np.abs(J).max()))
