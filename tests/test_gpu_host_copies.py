"""Large host arrays through the staged copies: the two-body transform with the
identity returns its input bit for bit (every product is x 1 or x 0), at sizes below
and above the staged bound (16 MiB) and with a ragged last chunk; repeated calls on
one context, and three contexts at once."""
import numpy as np
import pytest

from quiqbox_amd.engine import Context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [37, 39, 41, 52])
def test_identity_transform_returns_its_input(n):
    ctx = Context(0)
    rng = np.random.default_rng(n)
    for rep in range(3):
        A = rng.uniform(-1, 1, (n,) * 4)
        keep = A.copy()
        out = ctx.mo_transform(A, np.eye(n))
        print("[gpu-test] n %d (%.1f MiB), call %d" % (n, A.nbytes / 2**20, rep), flush=True)
        assert np.array_equal(out, keep)
        assert np.array_equal(A, keep)
    ctx.close()


def test_two_contexts_at_once():
    import threading
    n, res = 45, {}

    def work(k):
        ctx = Context(0)
        A = np.random.default_rng(k).uniform(-1, 1, (n,) * 4)
        res[k] = all(np.array_equal(ctx.mo_transform(A, np.eye(n)), A) for _ in range(3))
        ctx.close()

    ts = [threading.Thread(target=work, args=(k,)) for k in range(3)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert res == {0: True, 1: True, 2: True}
