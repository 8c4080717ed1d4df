"""The generic (f and g shell) ERI kernel over its ways of dividing a quartet:
teams over contracted kets, one wide team, one wave; bra contractions longer than
it holds at a time (8); ket components in several parts (two g shells); shells
with missing components.  Dense tensor, Fock matrices (one and two sets, Schwarz
threshold, density screening off) against the oracle."""
import numpy as np
import pytest

import oracle
import quiqbox_amd as qb
from quiqbox_amd.basis import subshellXYZs

pytestmark = pytest.mark.gpu


def _basis(rng, shells):
    bs = []
    for L, nprim, keep in shells:
        c = tuple(rng.uniform(-0.8, 0.8, 3))
        x = np.exp(rng.uniform(np.log(0.3), np.log(4.0), nprim))
        w = rng.uniform(0.2, 1.0, nprim)
        for ijk in subshellXYZs(L)[:keep]:
            cons = [a * qb.get3DimPGTOrbNormFactor(e, ijk) for a, e in zip(w, x)]
            bs.append(qb.genGaussTypeOrb(c, list(x), cons, ijk, outerRenormalize=True))
    return bs


CASES = {
    "f_bare": [(3, 1, 10), (0, 1, 1), (1, 1, 3)],             # one wave, and the wide team for (ff|ff)
    "f_contracted_kets": [(3, 1, 10), (0, 3, 1), (1, 2, 2)],   # shares of 4, 6 and 9 ket primitive pairs
    "f_long_bra": [(3, 9, 4), (0, 2, 1)],                      # 18 and 81 bra primitive pairs, 8 at a time
    "d_f": [(3, 1, 7), (2, 2, 6)],
    "g_g": [(4, 1, 15), (0, 4, 1)],                            # 225 ket components in parts
    "g_f": [(4, 2, 3), (3, 1, 2), (1, 1, 3)],
}


@pytest.mark.parametrize("name", CASES)
def test_generic_kernel_against_oracle(name):
    rng = np.random.default_rng(len(name))
    gb = qb.GPUBasis(_basis(rng, CASES[name]))
    E = oracle.Basis(gb.flat.as_dict()).eri_dense()
    assert np.max(np.abs(gb.eri_dense() - E)) < 1e-12
    n = gb.n
    D = rng.standard_normal((2, n, n))
    D = D + D.transpose(0, 2, 1)
    ref = [oracle.gcore(E, D[0] + D[1], D[s]) for s in range(2)]
    G = gb.jk(np.stack([D[0] + D[1]] * 2), D, 0.0)
    G1 = gb.jk(D[0] + D[1], D[1], 1e-14)
    assert np.max(np.abs(G - ref)) < 1e-11 * max(1.0, np.max(np.abs(ref)))
    assert np.max(np.abs(G1 - ref[1])) < 1e-11 * max(1.0, np.max(np.abs(ref)))
