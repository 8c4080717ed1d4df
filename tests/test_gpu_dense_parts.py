"""Dense tensor with chunks shared by a block's waves, and Schwarz bounds with
several lanes a pair, at contractions from 1 to 13 primitives (so 1 to 169 primitive
pairs: fewer than a block has parts, not a multiple of them, many per part).

- s, p and d shells on two centres against the oracle's dense tensor, and bit for bit
  the same on a second call.  1e-12 absolute, as the other dense comparisons: the
  integrals of these normalised functions are below 10.
- s functions alone, where every function is a shell: the number of quartets the
  lists keep at a threshold against the count from sqrt((ij|ij)) of the oracle's
  tensor, at thresholds that no product Q_ij Q_kl comes within 1e-9 of.
"""
import numpy as np
import pytest

import oracle
import quiqbox_amd as qb
from helpers import random_spd_basis

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sets", [[(1, 13, 2), (7, 2, 1)], [(13, 1, 3), (5, 4, 2)], [(2, 3, 5), (1, 1, 1), (8, 1, 1)]])
def test_dense_parts_match_oracle(sets):
    bs = []
    for k, nprim in enumerate(sets):
        bs += random_spd_basis(90 + k, n_atoms=1, box=2.0, nprim=nprim)[1]
    gb = qb.GPUBasis(bs)
    E = gb.eri_dense()
    print("[gpu-test] contractions %s: n %d" % (sets, gb.n), flush=True)
    assert np.array_equal(gb.eri_dense(), E)
    R = oracle.Basis(gb.flat.as_dict()).eri_dense()
    err = float(np.abs(E - R).max())
    print("[gpu-test]   max|dE| %.3e (max|E| %.3e)" % (err, float(np.abs(R).max())), flush=True)
    assert err < 1e-12


def test_dense_with_f_shells_same_on_every_run():
    bs = random_spd_basis(97, n_atoms=2, box=2.0, lmax=3, nprim=(3, 2, 1, 2))[1]
    gb = qb.GPUBasis(bs)
    E = gb.eri_dense()
    print("[gpu-test] s to f shells: n %d" % gb.n, flush=True)
    for _ in range(3):
        assert np.array_equal(gb.eri_dense(), E)
    # the eight permutations of every element are one value
    for p in ((1, 0, 2, 3), (0, 1, 3, 2), (2, 3, 0, 1)):
        assert np.array_equal(E.transpose(p), E)


def test_schwarz_bounds_of_uneven_contractions():
    rng = np.random.default_rng(4)
    bs = []
    for k in (1, 2, 3, 5, 8, 13, 1, 6):
        xp = np.exp(rng.uniform(np.log(0.2), np.log(30.0), k))
        cons = [c * qb.get3DimPGTOrbNormFactor(x, (0, 0, 0)) for x, c in zip(xp, rng.uniform(0.2, 1.0, k))]
        bs.append(qb.genGaussTypeOrb(tuple(rng.uniform(0, 6.0, 3)), list(xp), cons, (0, 0, 0), outerRenormalize=True))
    gb = qb.GPUBasis(bs)
    R = oracle.Basis(gb.flat.as_dict()).eri_dense()
    i, j = np.tril_indices(gb.n)
    Q = np.sqrt(R[i, j, i, j])
    P = np.outer(Q, Q)[np.tril_indices(len(Q))]
    assert len(bs) == gb.n
    tested = 0
    for thr in (1e-10, 3e-7, 1e-5, 1e-3, 0.03):
        if np.any(np.abs(P / thr - 1.0) < 1e-9):
            continue
        got = int(np.sum(gb.jk_stats(thr)["shell_quartets"]))
        print("[gpu-test] threshold %g: %d quartets (oracle %d)" % (thr, got, int((P >= thr).sum())), flush=True)
        assert got == int((P >= thr).sum())
        tested += 1
    assert tested >= 3
