"""Orders of the persistent tridiagonalization that the LDS of a block decides: the
first of 256 blocks, the largest that fits (1850) and the first that does not (1851,
solved by the library's own reduction); and what a solve beyond them allocates.

Tolerances as in test_gpu_tridiag: 8 n eps |F|_2."""
import numpy as np
import pytest

from quiqbox_amd.engine import Context, default_context
from test_gpu_tridiag import _check, _matrix

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1536, 1850, 1851])
def test_fock_solve_eigenpairs_of_large_orders(n):
    _check(default_context(), _matrix("dense", n))


def test_no_exchange_buffer_for_an_order_that_does_not_fit():
    """A solve of order 2304 must not hold the exchange buffer (2 n^2 values) that it
    cannot use: the first solve of an order that fits still has to allocate its own."""
    ctx = Context(0)
    _check(ctx, _matrix("dense", 2304))
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    _check(ctx, _matrix("dense", 1600))
    torch.cuda.synchronize()
    grown = before - torch.cuda.mem_get_info()[0]
    print("[gpu-test] allocated by the solve of order 1600: %.1f MB" % (grown / 1e6), flush=True)
    assert grown >= 2 * 1600 * 1600 * 8
    ctx.close()
