"""Schwarz bounds of more shell pairs than one grid of the bound kernel takes (65536 blocks,
four pairs each at 64 lanes a pair), and than 2^32 threads would (11,700 functions, 68
million pairs): the number of shell quartets that single-primitive s functions keep at
several thresholds, against the count from the closed form (ab|ab) =
2 pi^(5/2) K^2 / (p^2 sqrt(2p)).  Pairs whose product lies within rounding of the threshold
may fall on either side: 1e-6 of the count."""
import dataclasses

import numpy as np
import pytest

import quiqbox_amd as qb

pytestmark = pytest.mark.gpu


def closed_form(x, w, cen):
    i, j = np.tril_indices(len(x))
    p = x[i] + x[j]
    K = w[i] * w[j] * np.exp(-x[i] * x[j] / p * ((cen[i] - cen[j]) ** 2).sum(1))
    Q = np.sqrt(2 * np.pi ** 2.5 * K * K / (p * p * np.sqrt(2 * p)))
    Q[np.abs(K / p) < 1e-20] = 0.0      # pairs without a primitive pair
    return np.sort(Q)[::-1]


def kept(Q, thr):
    """pairs (a, b), b up to a in descending order, with Q_a Q_b >= thr"""
    Q = Q[Q > 0.0]
    n = np.searchsorted(-Q, -(thr / Q), side="right")
    return int(np.minimum(n, np.arange(1, len(Q) + 1)).sum())


@pytest.mark.parametrize("n,box,thrs", [(800, 60.0, (1e-4, 1e-8, 1e-12)), (11700, 400.0, (1e-8,))])
def test_bounds_beyond_one_grid(n, box, thrs):
    rng = np.random.default_rng(9)
    cen = rng.uniform(0.0, box, (n, 3))
    x = np.exp(rng.uniform(np.log(0.2), np.log(3.0), n))
    w = (2.0 * x / np.pi) ** 0.75
    one = qb.flatten_basis([qb.genGaussTypeOrb((0.0, 0.0, 0.0), [1.0], [1.0], (0, 0, 0))])
    index = np.arange(n + 1, dtype=np.asarray(one.bf_ptr).dtype)
    flat = dataclasses.replace(one, prim_cen=cen, prim_xpn=x, bf_ptr=index, bf_prim=index[:-1], bf_w=w,
                               prim_ang=np.zeros((n, 3), dtype=np.asarray(one.prim_ang).dtype))
    gb = qb.GPUBasis(flat)
    assert n * (n + 1) // 2 > 65536 * 4
    Q = closed_form(x, w, cen)
    for thr in thrs:
        got = int(gb.jk_stats(thr)["shell_quartets"].sum())
        ref = kept(Q, thr)
        print("[gpu-test] %d functions, thr %g: %d quartets, closed form %d" % (n, thr, got, ref), flush=True)
        assert abs(got - ref) <= 1e-6 * ref
