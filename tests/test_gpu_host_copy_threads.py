"""Threads of the staged host copies: no more than the CPUs that the calling thread may use,
and the plain copy (no thread) where that is one.  The calls run in a thread bound to one,
two and three CPUs while the process's threads are counted; the transform with the identity
returns its input bit for bit at every count."""
import os
import threading

import numpy as np
import pytest

from quiqbox_amd.engine import Context

pytestmark = pytest.mark.gpu


def _tasks():
    return len(os.listdir("/proc/self/task"))


@pytest.mark.parametrize("cpus", [1, 2, 3])
def test_no_more_threads_than_cpus(cpus):
    allowed = sorted(os.sched_getaffinity(0))
    if len(allowed) < cpus:
        pytest.skip("the process may use fewer CPUs")
    n, res = 60, {}
    A = np.random.default_rng(n).uniform(-1, 1, (n,) * 4)     # 104 MB
    ctx = Context(0)
    ctx.mo_transform(A, np.eye(n))                            # the runtime's own threads are there
    started, go = threading.Event(), threading.Event()

    def work():
        os.sched_setaffinity(0, set(allowed[:cpus]))
        res["mask"] = len(os.sched_getaffinity(0))
        started.set()
        go.wait()
        res["equal"] = all(np.array_equal(ctx.mo_transform(A, np.eye(n)), A) for _ in range(4))
        res["done"] = True

    t = threading.Thread(target=work)
    t.start()
    started.wait()
    before, most = _tasks(), 0
    go.set()
    while not res.get("done"):
        most = max(most, _tasks())
    t.join()
    ctx.close()
    print("[gpu-test] %d CPUs: %d threads before, at most %d during the copies" % (cpus, before, most), flush=True)
    assert res["mask"] == cpus
    assert res["equal"]
    assert most - before <= cpus - 1
