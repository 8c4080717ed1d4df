"""The gradient kernels' two accumulation forms (a block's LDS copy of the
outputs, and global atomics where the copy does not fit) and ragged primitive
counts, against central differences of the energy functional
sum D H - sum W S + 1/2 sum D (J[D] - K[D]/2) at fixed weights and densities."""
import dataclasses

import numpy as np
import pytest

import quiqbox_amd as qb
from quiqbox_amd.basis import flatten_basis, subshellXYZs

pytestmark = pytest.mark.gpu


def _basis(n_sites, spacing, shells):
    side = int(np.ceil(n_sites ** (1.0 / 3.0)))
    bs, cen = [], []
    rng = np.random.default_rng(n_sites)
    for k in range(n_sites):
        c = spacing * np.array([k % side, k // side % side, k // side ** 2], float) + 0.1 * rng.uniform(-1, 1, 3)
        cen.append(c)
        for L, nprim in shells[k % len(shells)]:
            x = np.exp(rng.uniform(np.log(0.3), np.log(4.0), nprim))
            w = rng.uniform(0.2, 1.0, nprim)
            for ijk in subshellXYZs(L):
                cons = [a * qb.get3DimPGTOrbNormFactor(e, ijk) for a, e in zip(w, x)]
                bs.append(qb.genGaussTypeOrb(tuple(c), list(x), cons, ijk))
    return flatten_basis(bs), np.array(cen)


# LDS copy: 2 x radial + 3 x shells doubles; 300 shells of 8 primitives need
# 45.6 KB beside 23 KB of Boys rows, beyond the 64 KB of a block
@pytest.mark.parametrize("n_sites,spacing,shells", [
    (4, 1.6, [[(0, 1), (1, 3)], [(0, 8)], [(1, 5)]]),
    (300, 30.0, [[(0, 8)]]),
])
def test_gradient_against_central_differences(n_sites, spacing, shells):
    flat, cen = _basis(n_sites, spacing, shells)
    n = flat.n_bf
    rng = np.random.default_rng(7)
    D = rng.standard_normal((n, n))
    D = 0.1 * (D + D.T) + np.diag(rng.uniform(0.5, 1.5, n))
    W = rng.standard_normal((n, n))
    W = 0.1 * (W + W.T)
    Z, R = np.array([1.0, 2.0]), np.array([[0.2, -0.3, 0.4], [1.5, 0.1, -0.2]])

    def energy(fl):
        gb = qb.GPUBasis(fl)
        H = gb.core_hamiltonian(Z, R)
        return float(np.sum(D * H) - np.sum(W * gb.overlap()) + 0.5 * np.sum(D * gb.jk(D, 0.5 * D, 0.0)))

    gb = qb.GPUBasis(flat)
    gx, gl, gc, sh = gb.rhf_gradient(D, W, Z, R, 0.0)
    for shell in (0, len(sh["L"]) - 1):
        x = sh["xpn"][sh["poff"][shell]]
        at = np.all(np.asarray(flat.prim_cen) == sh["center"][shell], axis=1)
        prim = at & (np.asarray(flat.prim_xpn) == x)
        h = 1e-4
        E = []
        for s in (1, -1):
            xp = np.array(flat.prim_xpn, float)
            xp[prim] += s * h * x
            E.append(energy(dataclasses.replace(flat, prim_xpn=xp)))
        fd = (E[0] - E[1]) / (2 * h * x)
        # truncation O(h^2) and the energies' rounding over h
        scale = max(1.0, abs(E[0]))
        assert gx[sh["poff"][shell]] == pytest.approx(fd, rel=2e-6, abs=2e-10 * scale)
    # centre of the first site, all its shells together
    on = np.all(sh["center"] == cen[0], axis=1)
    E = []
    for s in (1, -1):
        pc = np.array(flat.prim_cen, float)
        pc[np.all(pc == cen[0], axis=1), 2] += s * 1e-4
        E.append(energy(dataclasses.replace(flat, prim_cen=pc)))
    scale = max(1.0, abs(E[0]))
    assert gc[on, 2].sum() == pytest.approx((E[0] - E[1]) / 2e-4, rel=2e-6, abs=2e-10 * scale)
