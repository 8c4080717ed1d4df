"""Dense tensors of one class or one pair of pair classes (one launch, which stays on the
main stream) and the smallest with two, against the oracle; each twice, with equal bits."""
import numpy as np
import pytest

import oracle
import quiqbox_amd as qb
from quiqbox_amd.basis import subshellXYZs

pytestmark = pytest.mark.gpu


def _shell(c, L, x):
    return [qb.genGaussTypeOrb(c, list(x), [0.7 * qb.get3DimPGTOrbNormFactor(e, ijk) for e in x], ijk)
            for ijk in subshellXYZs(L)]


CASES = {
    "s": _shell((0.0, 0.1, 0.0), 0, (0.8, 0.3)),
    "ss": _shell((0.0, 0.1, 0.0), 0, (0.8, 0.3)) + _shell((0.9, 0.0, 0.4), 0, (1.7,)),
    "p": _shell((0.0, 0.1, 0.0), 1, (0.8, 0.3)),
    "sp": _shell((0.0, 0.1, 0.0), 0, (0.8,)) + _shell((0.9, 0.0, 0.4), 1, (0.5, 1.7)),
    "d": _shell((0.0, 0.1, 0.0), 2, (0.8,)),
    "f": _shell((0.0, 0.1, 0.0), 3, (0.8, 0.3)),
    "sf": _shell((0.0, 0.1, 0.0), 0, (0.8,)) + _shell((0.9, 0.0, 0.4), 3, (0.5,)),
}


@pytest.mark.parametrize("name", CASES)
def test_small_tensor_against_oracle(name):
    gb = qb.GPUBasis(CASES[name])
    E = oracle.Basis(gb.flat.as_dict()).eri_dense()
    for _ in range(2):
        G = gb.eri_dense()
        assert np.abs(G - E).max() < 1e-12 * max(1.0, float(np.abs(E).max()))
    assert np.array_equal(G, gb.eri_dense())
