"""The dense tensor right after a Fock build that is still running on a caller's
stream: both use the basis's staged-class workspaces, so the tensor has to wait for
the build.  A sleep on the side stream holds the build back until the tensor's call
has begun.  Checked against the same calls made one at a time: the tensor's elements
each have one writer and a fixed summation order (equal bits), G is summed by atomics
(1e-12 of its largest element)."""
import numpy as np
import pytest

import quiqbox_amd as qb
from quiqbox_amd.engine import Context
from quiqbox_amd.systems import water_box

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nset", [1, 2])
def test_dense_tensor_waits_for_a_build_on_another_stream(nset):
    bs = water_box(2, 11, basis="cc-pVDZ")[1]
    ctx = Context(0)
    gb = qb.GPUBasis(bs, ctx=ctx)
    n = gb.n
    rng = np.random.default_rng(3)
    D = rng.uniform(-0.1, 0.1, (2, nset, n, n))
    D = D + D.transpose(0, 1, 3, 2)
    dJ, dK = (torch.tensor(x, device="cuda") for x in D)
    dG = torch.zeros_like(dJ)
    G0 = gb.jk(D[0], D[1], 0.0)
    E0 = gb.eri_dense()
    side = torch.cuda.Stream()
    torch.cuda.synchronize()
    for rep in range(3):
        print("[gpu-test] %d sets, call %d" % (nset, rep), flush=True)
        dG.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            torch.cuda._sleep(10_000_000)
        gb.jk_device(dJ.data_ptr(), dK.data_ptr(), dG.data_ptr(), nset, 0.0, stream=side.cuda_stream)
        E = gb.eri_dense()
        side.synchronize()
        assert np.array_equal(E, E0)
        assert np.max(np.abs(dG.cpu().numpy() - G0)) < 1e-12 * max(1.0, float(np.abs(G0).max()))
    del gb
    ctx.close()
