"""The generated adjoint recurrences in the form that the gradient kernels are built with
(EriAdj::vrr_adj_grp<GR>: one group of bra components each, three for (pp|pp)), evaluated
on the CPU from the emitted statements.  Each group's derivatives against central
differences of its own seeded sum, exact up to O(h^2) truncation; the groups' forward
values against the one-group form's, component by component, and their seeded sums against
the sum over all components (the same statements in another order: 1e-13)."""
import re

import numpy as np
import pytest

import test_gen_adjoint as base
from test_gen_adjoint import CLASSES, gen_eri

IDS = ["".join(map(str, c)) for c in CLASSES]


def _groups(cls):
    """(programs of the groups, NACC) of the emitted vrr_adj_grp"""
    n = gen_eri.GRAD_GROUPS.get(cls, 1)
    code = gen_eri.gen_adjoint(*cls, n)[0]
    assert int(re.search(r"NGRP = (\d+)", code).group(1)) == n
    body = base._body(code, "double vrr_adj_grp(")
    head, *parts = re.split(r"(?:else )?if constexpr \(GR == \d+\) \{\n", body)
    assert len(parts) == n
    progs = [base._to_python(head + p[:p.rindex("}")] if "}" in p else head + p) for p in parts]
    return progs, int(re.search(r"NACC = (\d+)", code).group(1))


def _inputs(cls, nacc):
    rng = np.random.default_rng(sum(cls) + 7)
    inputs = {k: float(rng.uniform(-1.0, 1.0)) for k in gen_eri.VRR_INPUTS}
    for k in ("inv2p", "inv2q", "inv2pq", "rho_p", "rho_q"):
        inputs[k] = float(rng.uniform(0.1, 0.9))
    return inputs, [float(x) for x in rng.uniform(0.1, 1.0, sum(cls) + 1)], [float(x) for x in rng.normal(size=nacc)]


def _run(prog, cls, nacc, F, inp, g):
    env = dict(inp, F=list(F), g=list(g), acc=[0.0] * nacc, Fb=[0.0] * (sum(cls) + 1),
               bin=[0.0] * len(gen_eri.VRR_INPUTS), NACC=nacc)
    return base._run(prog, env)


@pytest.mark.parametrize("cls", CLASSES, ids=IDS)
def test_group_adjoints_match_central_differences(cls):
    progs, nacc = _groups(cls)
    inputs, F, g = _inputs(cls, nacc)
    h = 1e-5
    for gr, prog in enumerate(progs):
        r = _run(prog, cls, nacc, F, inputs, g)
        for m in range(len(F)):
            L = []
            for s in (h, -h):
                Fs = list(F)
                Fs[m] += s
                L.append(_run(prog, cls, nacc, Fs, inputs, g)["__ret"])
            assert r["Fb"][m] == pytest.approx((L[0] - L[1]) / (2 * h), rel=1e-7, abs=1e-9), (gr, "F", m)
        for k, name in enumerate(gen_eri.VRR_INPUTS):
            L = [_run(prog, cls, nacc, F, dict(inputs, **{name: inputs[name] + s}), g)["__ret"] for s in (h, -h)]
            assert r["bin"][k] == pytest.approx((L[0] - L[1]) / (2 * h), rel=1e-7, abs=1e-9), (gr, name)


@pytest.mark.parametrize("cls", CLASSES, ids=IDS)
def test_groups_share_out_the_components(cls):
    progs, nacc = _groups(cls)
    inputs, F, g = _inputs(cls, nacc)
    one = base._to_python(base._body(gen_eri.gen_adjoint(*cls)[0], "double vrr_adj("))
    # [e0|f0]_k: the seeded sum with the k-th unit seed
    ref = [_run(one, cls, nacc, F, inputs, np.eye(nacc)[k])["__ret"] for k in range(nacc)]
    runs = [_run(p, cls, nacc, F, inputs, g) for p in progs]
    acc = np.array([r["acc"] for r in runs])
    assert np.all(np.count_nonzero(acc, axis=0) == 1)      # every component in one group
    assert acc.sum(0) == pytest.approx(ref, rel=1e-13, abs=1e-13)
    assert sum(r["__ret"] for r in runs) == pytest.approx(float(np.dot(g, ref)), rel=1e-12)
    total = _run(one, cls, nacc, F, inputs, g)
    for key in ("Fb", "bin"):
        assert np.sum([r[key] for r in runs], axis=0) == pytest.approx(total[key], rel=1e-12, abs=1e-12)
