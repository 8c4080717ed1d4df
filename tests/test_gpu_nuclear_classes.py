"""Nuclear attraction by pair class (one wave per shell pair, its lanes over
(primitive pair, nucleus) items): every pair of s..g shells against the oracle,
with nuclei counts around the lane count and contractions of different lengths."""
import numpy as np
import pytest

import oracle
import quiqbox_amd as qb
from quiqbox_amd.basis import subshellXYZs

pytestmark = pytest.mark.gpu


def _basis(rng, Ls):
    bs = []
    for L, nprim in Ls:
        c = tuple(rng.uniform(-1.0, 1.0, 3))
        x = np.exp(rng.uniform(np.log(0.2), np.log(6.0), nprim))
        w = rng.uniform(0.2, 1.0, nprim)
        for ijk in subshellXYZs(L):
            cons = [a * qb.get3DimPGTOrbNormFactor(e, ijk) for a, e in zip(w, x)]
            bs.append(qb.genGaussTypeOrb(c, list(x), cons, ijk))
    return bs


# item counts below, at and above the 64 lanes, and remainders of the item walk
@pytest.mark.parametrize("nnuc", [1, 2, 7, 63, 64, 65, 131])
@pytest.mark.parametrize("Ls", [[(0, 1), (1, 3), (2, 2)], [(0, 9), (0, 1), (1, 5)], [(3, 1), (4, 2), (0, 2), (2, 1), (1, 1)]])
def test_nuclear_against_oracle(nnuc, Ls):
    rng = np.random.default_rng(nnuc)
    gb = qb.GPUBasis(_basis(rng, Ls))
    Z = rng.uniform(0.5, 3.0, nnuc)
    R = rng.uniform(-3.0, 3.0, (nnuc, 3))
    V = gb.nuclear(Z, R)
    ref = oracle.Basis(gb.flat.as_dict()).nuclear(Z, R)
    # the repository's 1e-11 bar for a few nuclei; rounding grows with the summed charge
    assert np.max(np.abs(V - ref)) < 1e-11 * max(1.0, Z.sum() / 10.0)
    assert np.array_equal(V, V.T)
