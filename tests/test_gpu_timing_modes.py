"""Per-class times of the concurrent builds (timing mode 2).  A basis of one class runs on
one stream, so its per-class times add up to no more than the build; a basis of several
classes forks, and each class still reports a time.  The elapsed times are differences of
event stamps of 40 ns resolution (and a class's end precedes the build's), so 1% is
allowed."""
import numpy as np
import pytest

import quiqbox_amd as qb
from quiqbox_amd.engine import Context
from quiqbox_amd.systems import h10_sto3g, water_box

pytestmark = pytest.mark.gpu


def _times(bs):
    ctx = Context(0)
    gb = qb.GPUBasis(bs, ctx=ctx)
    D = np.eye(gb.n)
    gb.jk(2 * D, D, 0.0)
    ctx.set_timing(2)
    for _ in range(5):
        gb.jk(2 * D, D, 0.0)
    ms, total = ctx.last_timing()
    quartets = gb.jk_stats(0.0)["shell_quartets"]
    ctx.set_timing(0)
    del gb
    ctx.close()
    return ms, total, quartets


def test_one_class():
    ms, total, quartets = _times(h10_sto3g(160)[1])
    print("[gpu-test] one class: classes %.3f ms, build %.3f ms" % (ms.sum(), total), flush=True)
    assert np.count_nonzero(quartets) == 1
    assert ms[np.argmax(quartets)] > 0.0
    assert ms.sum() <= 1.01 * total


def test_several_classes():
    ms, total, quartets = _times(water_box(2, 3, basis="cc-pVDZ")[1])
    print("[gpu-test] %d classes: build %.3f ms" % (np.count_nonzero(quartets), total), flush=True)
    assert np.all(ms[quartets > 0] > 0.0)
    assert ms.max() <= 1.01 * total
