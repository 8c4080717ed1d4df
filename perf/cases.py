"""Timed cases: what a program built on quiqbox_amd asks of the GPU, one entry
point each.

  fock      the two-electron matrix G = J[DJ] - K[DK] of one SCF step (GPUBasis.jk
            with host densities, GPUBasis.jk_device with densities on the GPU):
            one or two density sets, FP64 or mixed precision, full builds and
            density-screened increments, from a ten-function hydrogen chain to
            600 functions, s to f shells
  dense     the dense (ij|kl) tensor (GPUBasis.eri_dense)
  nuclear   the nuclear-attraction matrix (GPUBasis.nuclear)
  gradient  the energy derivatives of the basis parameters (GPUBasis.rhf_gradient,
            uhf_gradient)
  orbitals  one SCF step's eigenvectors and density (Context.fock_solve)
  purify    the same density by purification (Context.purified_density)
  basis_change  AO to MO two-electron integrals (Context.mo_transform)
  train     one training step of the learned guess (LearnedGuess.train_step)

The molecules are those of quiqbox_amd.systems, placed by the seed.  Densities
are synthetic: symmetric, the diagonal near an occupation, off-diagonal blocks
falling with the distance of the functions' centres, as converged ones do.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.abspath("quiqbox.jl_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import quiqbox_amd as qb  # noqa: E402
from quiqbox_amd import learned_guess, systems  # noqa: E402
from quiqbox_amd.basis import flatten_basis  # noqa: E402
from quiqbox_amd.particles import NuclearCluster  # noqa: E402

THR = 1e-12          # Schwarz threshold of every Fock build and gradient


def listed():
    return [
        _fock("fock_h10_host", "h_chain", 10),
        _fock("fock_water8_uhf_host", "water", 8, sets=2),
        _fock("fock_cluster64_sp_mixed", "cluster_sp", 64, mixed=True, host=False),
        _fock("fock_water24", "water", 24, host=False),
        _fock("fock_cluster160_spd", "cluster_spd", 160, host=False),
        {"name": "dense_n2_pvtz", "kind": "dense", "system": "n2_tz", "size": 2},
        {"name": "nuclear_cluster160_spd", "kind": "nuclear", "system": "cluster_spd", "size": 160},
        {"name": "gradient_h32_sp", "kind": "gradient", "size": 32, "sets": 1},
        {"name": "orbitals_600", "kind": "orbitals", "n": 600},
        {"name": "purify_600", "kind": "purify", "n": 600},
        {"name": "basis_change_70", "kind": "basis_change", "n": 70, "n_mo": 70},
        {"name": "train_water_4096", "kind": "train", "layout": "water", "rows": 4096},
    ]


def _fock(name, system, size, sets=1, mixed=False, increment=False, host=True):
    return {"name": name, "kind": "fock", "system": system, "size": size, "sets": sets, "mixed": mixed,
            "increment": increment, "host": host}


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["fock"] * 6 + ["dense", "nuclear", "nuclear", "gradient", "orbitals", "purify", "basis_change",
                                      "train"])
    if kind == "fock":
        system = rng.choice(["h_chain", "water", "water", "cluster_sp", "cluster_spd", "n2_tz"])
        hi = {"h_chain": 40, "water": 18, "cluster_sp": 96, "cluster_spd": 120, "n2_tz": 2}[system]
        lo = {"h_chain": 2, "water": 1, "cluster_sp": 4, "cluster_spd": 10, "n2_tz": 2}[system]
        c = _fock("", system, _log_int(rng, lo, hi), sets=rng.choice([1, 1, 2]), mixed=rng.random() < 0.25,
                  increment=rng.random() < 0.25, host=rng.random() < 0.5)
        del c["name"]
        return c
    if kind == "dense":
        system = rng.choice(["h_chain", "water", "cluster_spd", "n2_tz"])
        hi = {"h_chain": 64, "water": 3, "cluster_spd": 16, "n2_tz": 2}[system]
        return {"kind": kind, "system": system, "size": _log_int(rng, 2, hi)}
    if kind == "nuclear":
        system = rng.choice(["h_chain", "water", "cluster_sp", "cluster_spd"])
        hi = {"h_chain": 64, "water": 24, "cluster_sp": 128, "cluster_spd": 160}[system]
        return {"kind": kind, "system": system, "size": _log_int(rng, 2, hi)}
    if kind == "gradient":
        return {"kind": kind, "size": _log_int(rng, 2, 32), "sets": rng.choice([1, 2])}
    if kind in ("orbitals", "purify"):
        return {"kind": kind, "n": _log_int(rng, 40, 600)}
    if kind == "basis_change":
        n = _log_int(rng, 8, 70)
        return {"kind": kind, "n": n, "n_mo": rng.choice([n, max(1, n // 2), max(1, n - 3)])}
    return {"kind": "train", "layout": rng.choice(["water", "cho"]), "rows": _log_int(rng, 100, 4096)}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _system(case, seed):
    """(nuclei, basis) of a case, placed by the seed."""
    kind, n = case["system"], case["size"]
    rng = np.random.default_rng([seed, 1])
    if kind == "h_chain":
        return systems.h10_sto3g(n, float(1.4 + 0.1 * rng.uniform(-1.0, 1.0)))
    if kind == "water":
        return systems.water_box(n, seed, basis="cc-pVDZ")
    if kind == "n2_tz":
        z = float(1.0 + 0.05 * rng.uniform(-1.0, 1.0))
        cen = [(0.0, 0.0, -z), (0.0, 0.0, z)]
        bs = []
        for c in cen:
            bs += qb.genGaussTypeOrbSeq(c, "N", "cc-pVTZ")
        return NuclearCluster(["N", "N"], cen, pairwiseSort=False), bs
    # the 64- and 160-atom clusters fill a 20-bohr cube; smaller ones keep the
    # density of the 64-atom cube
    box = 20.0 * min(1.0, (n / 64.0) ** (1.0 / 3.0)) + 2.0 * (n < 64)
    return systems.random_cluster(n, seed, with_d=kind == "cluster_spd", box=box)


def _densities(flat, sets, seed, scale):
    """(DJ, DK), each (sets, n, n): symmetric, falling with distance."""
    rng = np.random.default_rng([seed, 2])
    cen = np.asarray(flat.prim_cen)[np.asarray(flat.bf_prim)[np.asarray(flat.bf_ptr)[:-1]]]
    d = np.sqrt(((cen[:, None, :] - cen[None, :, :]) ** 2).sum(-1))
    n = len(cen)
    D = []
    for _ in range(sets):
        M = rng.standard_normal((n, n))
        M = 0.3 * (M + M.T) * np.exp(-0.7 * d)
        M[np.arange(n), np.arange(n)] = rng.uniform(0.2, 1.0, n)
        D.append(scale * M)
    DK = np.stack(D)
    DJ = np.stack([2.0 * D[0]] if sets == 1 else [D[0] + D[1]] * 2)
    return DJ, DK


def _fock_in_basis(n, seed):
    """X, F of one SCF step with a gap at the Fermi level, and the
    eigenvectors and eigenvalues of X F X that went into them."""
    rng = np.random.default_rng([seed, 3])
    nocc = max(1, n // 5)
    e = np.concatenate([np.linspace(-20.0, -0.5, nocc), np.linspace(0.2, 8.0, n - nocc)])
    e = e + 0.3 * np.concatenate([[0.0], np.diff(e)]) * rng.uniform(-1.0, 0.0, n)
    Q = np.linalg.qr(rng.standard_normal((n, n)))[0]
    U = np.linalg.qr(rng.standard_normal((n, n)))[0]
    w = np.exp(rng.uniform(-0.7, 1.0, n))
    X, Xi = (U * w) @ U.T, (U / w) @ U.T
    F = Xi @ ((Q * e) @ Q.T) @ Xi
    return 0.5 * (X + X.T), 0.5 * (F + F.T), Q, e, nocc


def _tensor(case, seed):
    rng = np.random.default_rng([seed, 4])
    n, m = case["n"], case["n_mo"]
    T = rng.random((n, n, n, n)) - 0.3
    C = np.linalg.qr(rng.standard_normal((n, n)))[0][:, :m]
    return T, np.ascontiguousarray(C)


def _layout(case):
    return learned_guess.WATER if case["layout"] == "water" else learned_guess.CHO_SP


def _batch(case, seed):
    """Normalized features and padded density blocks of `rows` atom pairs."""
    rng = np.random.default_rng([seed, 5])
    lay = _layout(case)
    x = np.zeros((case["rows"], lay.n_in), dtype=np.float32)
    x[:, :lay.n_feat] = rng.standard_normal((case["rows"], lay.n_feat))
    y = 0.2 * rng.standard_normal((case["rows"], lay.n_out)).astype(np.float32)
    return x, y


def _gradient_inputs(case, seed):
    nuc, bs = systems.h_cluster_sp(case["size"], seed, box=10.0 * (case["size"] / 32.0) ** (1.0 / 3.0) + 1.0)
    flat = flatten_basis(bs)
    _, D = _densities(flat, 2, seed, 0.6)
    W = -0.4 * _densities(flat, 1, seed + 1, 0.6)[1][0]
    return nuc, flat, D, W


def prepare(case, seed):
    kind = case["kind"]
    s = dict(case)
    if kind in ("fock", "dense", "nuclear"):
        nuc, bs = _system(case, seed)
        gb = s["gb"] = qb.GPUBasis(bs)
        s["Z"], s["R"] = nuc.charges, nuc.coord_array
        if kind == "fock":
            DJ, DK = _densities(gb.flat, case["sets"], seed, 1e-3 if case["increment"] else 1.0)
            s["precision"] = qb.QBX_PREC_MIXED if case["mixed"] else qb.QBX_PREC_FP64
            if not case["host"]:
                DJ, DK = (torch.tensor(x, device="cuda") for x in (DJ, DK))
                s["G"] = torch.empty_like(DJ)
            s["DJ"], s["DK"] = DJ, DK
    elif kind == "gradient":
        nuc, flat, D, s["W"] = _gradient_inputs(case, seed)
        s["gb"] = qb.GPUBasis(flat)
        s["Z"], s["R"], s["D"], s["Dt"] = nuc.charges, nuc.coord_array, D, D[0] + D[1]
    elif kind in ("orbitals", "purify"):
        s["ctx"] = qb.default_context()
        s["X"], s["F"], _, _, s["nocc"] = _fock_in_basis(case["n"], seed)
    elif kind == "basis_change":
        s["ctx"] = qb.default_context()
        s["T"], s["C"] = _tensor(case, seed)
    else:
        x, y = _batch(case, seed)
        s["model"] = learned_guess.LearnedGuess(seed=seed, layout=_layout(case))
        s["xb"] = torch.tensor(x, device="cuda").to(torch.bfloat16)
        s["yt"] = torch.tensor(y, device="cuda")
        s["rw"] = torch.ones(case["rows"], dtype=torch.float32, device="cuda")
    return s


def run(s):
    kind = s["kind"]
    if kind == "fock":
        gb = s["gb"]
        if s["increment"]:
            gb.ctx.set_density_screening(THR)
        try:
            if s["host"]:
                return gb.jk(s["DJ"], s["DK"], THR, s["precision"])
            gb.jk_device(s["DJ"].data_ptr(), s["DK"].data_ptr(), s["G"].data_ptr(), s["sets"], THR, s["precision"])
            return s["G"]
        finally:
            if s["increment"]:
                gb.ctx.set_density_screening(0.0)
    if kind == "dense":
        return s["gb"].eri_dense()
    if kind == "nuclear":
        return s["gb"].nuclear(s["Z"], s["R"])
    if kind == "gradient":
        if s["sets"] == 2:
            return s["gb"].uhf_gradient(s["Dt"], s["D"][0], s["D"][1], s["W"], s["Z"], s["R"], THR)[:3]
        return s["gb"].rhf_gradient(s["Dt"], s["W"], s["Z"], s["R"], THR)[:3]
    if kind == "orbitals":
        return s["ctx"].fock_solve(s["X"], s["F"], s["nocc"])
    if kind == "purify":
        return s["ctx"].purified_density(s["X"], s["F"], s["nocc"])[0]
    if kind == "basis_change":
        return s["ctx"].mo_transform(s["T"], s["C"])
    m = s["model"]
    loss = m.train_step(s["xb"], s["yt"], s["rw"], s["rows"])
    return {"loss": loss, "W": list(m.dev.W), "b": list(m.dev.b)}


# ---------------------------------------------------------------------------
# least bytes and operations
# ---------------------------------------------------------------------------
def _ncart(L):
    return (L + 1) * (L + 2) // 2


def _quartet_flops(la, lb, lc, ld):
    """(per primitive quartet, per contracted quartet): geometry, Boys values
    and about 11 operations for each [e0|f0] value; transfer and digest of each
    Cartesian integral."""
    ne = sum(_ncart(l) for l in range(la, la + lb + 1))
    nf = sum(_ncart(l) for l in range(lc, lc + ld + 1))
    return 58 + 4 * (la + lb + lc + ld) + 11 * ne * nf, 15 * _ncart(la) * _ncart(lb) * _ncart(lc) * _ncart(ld)


@functools.lru_cache(maxsize=None)
def _screened_flops(system, size):
    """Operations of the Schwarz-screened unique quartets (s, p, d shells)."""
    st = qb.GPUBasis(_system({"system": system, "size": size}, 0)[1]).jk_stats(THR)
    f = 0.0
    for c, l in enumerate(qb.class_table()):
        fp, fc = _quartet_flops(*(int(x) for x in l))
        f += float(st["prim_quartets"][c]) * fp + float(st["shell_quartets"][c]) * fc
    return f


def _unscreened_flops(L, nprim):
    """Operations of all unique shell quartets of shells (L, primitives)."""
    pairs = {}
    for a in range(len(L)):
        for b in range(a + 1):
            k = (max(L[a], L[b]), min(L[a], L[b]))
            n, p = pairs.get(k, (0, 0))
            pairs[k] = n + 1, p + nprim[a] * nprim[b]
    f = 0.0
    for x, (nx, px) in pairs.items():
        for y, (ny, py) in pairs.items():
            fp, fc = _quartet_flops(*x, *y)
            f += 0.5 * (px * py * fp + nx * ny * fc)
    return f


def _shells(flat):
    """(L, primitives) of every shell: the functions of one centre, one
    exponent list and one L, every Cartesian component once."""
    seen = {}
    for f in range(flat.n_bf):
        p = flat.bf_prim[flat.bf_ptr[f]:flat.bf_ptr[f + 1]]
        L = int(np.sum(flat.prim_ang[p[0]]))
        w = flat.bf_w[flat.bf_ptr[f]:flat.bf_ptr[f + 1]]
        key = (tuple(flat.prim_cen[p[0]]), tuple(flat.prim_xpn[q] for q in p), L, round(float(w[0] / w[-1]), 9))
        seen[key] = (L, len(p))
    return [v[0] for v in seen.values()], [v[1] for v in seen.values()]


def work(case):
    kind = case["kind"]
    if kind in ("fock", "dense", "nuclear"):
        nuc, bs = _system(case, 0)
        flat = flatten_basis(bs)
        n = flat.n_bf
        L, npr = _shells(flat)
        if kind == "nuclear":
            pp = sum(a * b for a in npr for b in npr) / 2.0
            return {"bytes": 8 * n * n + 32 * len(nuc.charges) + 40 * flat.n_prim,
                    "flops": float(len(nuc.charges)) * pp * 60.0}
        if kind == "dense":
            return {"bytes": 8 * n ** 4 + 40 * flat.n_prim, "flops": _unscreened_flops(L, npr)}
        f = _unscreened_flops(L, npr) if max(L) > 2 else _screened_flops(case["system"], case["size"])
        return {"bytes": 24 * case["sets"] * n * n + 40 * flat.n_prim, "flops": f}
    if kind == "gradient":
        n, m = 4 * case["size"], case["size"]
        return {"bytes": 8 * (2 + (case["sets"] == 2) * 2) * n * n + 8 * (20 * m + 6 * m),
                "flops": 4.0 * _unscreened_flops([0, 1] * m, [4, 4] * m)}
    if kind == "orbitals":
        # two congruence products, tridiagonal form, its eigenvectors and their back-transformation, C and D
        n = case["n"]
        return {"bytes": 8 * (4 * n * n + n), "flops": (4.0 + 4.0 / 3 + 4.0 / 3 + 2.0 + 2.0 + 0.4) * n ** 3}
    if kind == "purify":
        # two congruence products, about 30 squarings
        n = case["n"]
        return {"bytes": 8 * 3 * n * n, "flops": 2.0 * 34 * n ** 3}
    if kind == "basis_change":
        n, m = case["n"], case["n_mo"]
        return {"bytes": 8 * (n ** 4 + m ** 4 + n * m),
                "flops": 2.0 * sum(n ** (4 - q) * m ** (q + 1) for q in range(4))}
    lay, r = _layout(case), case["rows"]
    sizes = [(lay.n_in, learned_guess.WIDTH), (learned_guess.WIDTH,) * 2, (learned_guess.WIDTH, lay.n_out)]
    p = sum(a * b + b for a, b in sizes)
    mul = sum(a * b for a, b in sizes)
    return {"bytes": r * (2 * lay.n_in + 4 * lay.n_out) + 24 * p + 2 * p,
            "flops": 2.0 * r * (2 * mul + mul - sizes[0][0] * sizes[0][1])}


# ---------------------------------------------------------------------------
# results in 64 bits
# ---------------------------------------------------------------------------
def _boys(n, T):
    """F_0..F_n of an array of arguments: the top order from the incomplete
    gamma function (a power series near zero), then downward."""
    T = torch.as_tensor(T, dtype=torch.float64)
    big = torch.clamp(T, min=0.5)
    top = torch.special.gammainc(torch.full_like(T, n + 0.5), big) * (0.5 * math.gamma(n + 0.5)) * big ** -(n + 0.5)
    ser, term = torch.zeros_like(T), torch.full_like(T, 1.0 / (2 * n + 1))
    for k in range(1, 22):
        ser = ser + term
        term = term * 2.0 * torch.clamp(T, max=0.5) / (2 * n + 2 * k + 1)
    e = torch.exp(-T)
    F = [torch.where(T < 0.5, e * ser, top)]
    for m in range(n - 1, -1, -1):
        F.insert(0, (2.0 * T * F[0] + e) / (2 * m + 1))
    return [f.numpy() for f in F]


def _functions(flat):
    """(centre, exponents, weights, Cartesian powers) of every function."""
    out = []
    for f in range(flat.n_bf):
        p = flat.bf_prim[flat.bf_ptr[f]:flat.bf_ptr[f + 1]]
        out.append((np.asarray(flat.prim_cen[p[0]], float), np.asarray(flat.prim_xpn)[p],
                    np.asarray(flat.bf_w[flat.bf_ptr[f]:flat.bf_ptr[f + 1]], float),
                    tuple(int(x) for x in flat.prim_ang[p[0]])))
    return out


def _hermite(i, j, a, b, XA, XB):
    """Hermite expansion E_t, t <= i + j, of x_A^i x_B^j on one axis, without
    the exponential of the pair (XA = P - A, XB = P - B)."""
    p = a + b

    def up(row, X):
        n = len(row)
        get = lambda t: row[t] if 0 <= t < n else 0.0 * p  # noqa: E731
        return [get(t - 1) / (2.0 * p) + X * get(t) + (t + 1) * get(t + 1) for t in range(n + 1)]

    row = [np.ones_like(p)]
    for _ in range(i):
        row = up(row, XA)
    for _ in range(j):
        row = up(row, XB)
    return row


def _exact_nuclear(flat, Z, R):
    """McMurchie-Davidson nuclear attraction, one function pair at a time."""
    fn = _functions(flat)
    n = len(fn)
    Z, R = np.asarray(Z, float), np.asarray(R, float).reshape(-1, 3)
    V = np.zeros((n, n))
    for i in range(n):
        Ai, xa, wa, la = fn[i]
        for j in range(i + 1):
            Bj, xb, wb, lb = fn[j]
            a, b = (v.ravel() for v in np.meshgrid(xa, xb, indexing="ij"))
            p = a + b
            w = np.outer(wa, wb).ravel() * np.exp(-a * b / p * ((Ai - Bj) ** 2).sum()) * 2.0 * math.pi / p
            P = (a[:, None] * Ai + b[:, None] * Bj) / p[:, None]
            E = [_hermite(la[t], lb[t], a, b, P[:, t] - Ai[t], P[:, t] - Bj[t]) for t in range(3)]
            PC = P[:, None, :] - R[None, :, :]
            L = sum(la) + sum(lb)
            F = _boys(L, (p[:, None] * (PC ** 2).sum(-1)).ravel())
            G = [((-2.0 * p[:, None]) ** m) * F[m].reshape(len(p), -1) for m in range(L + 1)]
            memo = {}

            def herm(t, u, v, m):
                if (t, u, v, m) in memo:
                    return memo[t, u, v, m]
                if t + u + v == 0:
                    r = G[m]
                else:
                    ax = 0 if t else 1 if u else 2
                    k = [t, u, v]
                    k[ax] -= 1
                    r = PC[:, :, ax] * herm(*k, m + 1)
                    if k[ax]:
                        k2 = list(k)
                        k2[ax] -= 1
                        r = r + k[ax] * herm(*k2, m + 1)
                memo[t, u, v, m] = r
                return r

            s = 0.0
            for t, et in enumerate(E[0]):
                for u, eu in enumerate(E[1]):
                    for v, ev in enumerate(E[2]):
                        s = s + (et * eu * ev * w) @ (herm(t, u, v, 0) @ Z)
            V[i, j] = V[j, i] = -s
    return V


def _exact_s_tensor(flat):
    """(ij|kl) of s functions in closed form."""
    fn = _functions(flat)
    n = len(fn)
    iu, ju = np.tril_indices(n)
    p, K, P = [], [], []
    for i, j in zip(iu, ju):
        (A, xa, wa, _), (B, xb, wb, _) = fn[i], fn[j]
        a, b = (v.ravel() for v in np.meshgrid(xa, xb, indexing="ij"))
        p.append(a + b)
        K.append(np.outer(wa, wb).ravel() * np.exp(-a * b / (a + b) * ((A - B) ** 2).sum()) / (a + b))
        P.append((a[:, None] * A + b[:, None] * B) / (a + b)[:, None])
    p, K, P = np.stack(p), np.stack(K), np.stack(P)
    E = np.zeros((n, n, n, n))
    for r, (i, j) in enumerate(zip(iu, ju)):
        pq = p[r][:, None, None] + p[None]
        T = p[r][:, None, None] * p[None] / pq * ((P[r][:, None, None, :] - P[None]) ** 2).sum(-1)
        v = 2.0 * math.pi ** 2.5 * K[r][:, None, None] * K[None] / np.sqrt(pq)
        v = (v * _boys(0, T.ravel())[0].reshape(T.shape)).sum((0, 2))
        M = np.zeros((n, n))
        M[iu, ju] = v
        M[ju, iu] = v
        E[i, j] = E[j, i] = M
    return E


def _bf(x):
    """Storage in bfloat16, as the layer's activations are kept."""
    return torch.tensor(x).to(torch.float32).to(torch.bfloat16).to(torch.float64).numpy()


def _exact_train(case, seed):
    """One Adam step from the seed's weights: products in 64 bits, activations
    and their gradients kept in bfloat16."""
    x, y = _batch(case, seed)
    lay, r, wd = _layout(case), case["rows"], learned_guess.WIDTH
    rng = np.random.default_rng(seed)
    sizes = [(lay.n_in, wd), (wd, wd), (wd, lay.n_out)]
    W = [(rng.uniform(-1.0, 1.0, size=s) / np.sqrt(s[0])).astype(np.float32).astype(np.float64) for s in sizes]
    Wb = [_bf(w) for w in W]
    h = [_bf(x.astype(np.float64))]
    for l in range(2):
        h.append(_bf(np.maximum(h[l] @ Wb[l], 0.0)))
    d = h[2] @ Wb[2] - y.astype(np.float64)
    loss = float((d * d).sum() / r)
    g = 2.0 * d / r
    outW, outb = [None] * 3, [None] * 3
    for l in (2, 1, 0):
        gw, gbias = h[l].T @ _bf(g), g.sum(0)
        adam = lambda v: 1e-3 * v / (np.abs(v) + 1e-8)  # noqa: E731  (first step: moments are the gradient)
        outW[l], outb[l] = W[l] - adam(gw), -adam(gbias)
        if l:
            g = (_bf(g) @ Wb[l].T) * (h[l] > 0.0)
    return {"loss": np.array([loss]), "W": outW, "b": outb}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("fock", "dense") and case["system"] == "h_chain" and case["size"] <= 40:
        flat = flatten_basis(_system(case, seed)[1])
        E = _exact_s_tensor(flat)
        if kind == "dense":
            return E
        DJ, DK = _densities(flat, case["sets"], seed, 1e-3 if case["increment"] else 1.0)
        G = np.einsum("ijkl,skl->sij", E, DJ) - np.einsum("iljk,skl->sij", E, DK)
        return G
    if kind == "nuclear":
        nuc, bs = _system(case, seed)
        flat = flatten_basis(bs)
        if flat.n_bf ** 2 * len(nuc.charges) > 60000:
            return None
        return _exact_nuclear(flat, nuc.charges, nuc.coord_array)
    if kind in ("orbitals", "purify"):
        X, F, Q, e, nocc = _fock_in_basis(case["n"], seed)
        if kind == "orbitals":
            C = X @ Q
            C = C * np.where(C[0] < 0, -1.0, 1.0)
            return C, e, C[:, :nocc] @ C[:, :nocc].T
        O = X @ Q[:, :nocc]
        return O @ O.T
    if kind == "basis_change":
        T, C = _tensor(case, seed)
        for _ in range(4):
            T = np.tensordot(T, C, (0, 0))
        return T
    if kind == "train":
        return _exact_train(case, seed)
    return None
