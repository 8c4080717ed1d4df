"""Column sums of more columns than a grid of 64 threads a column holds (67 million), around
the walk of 65536 blocks of 16 columns and around the bound of few rows (16): sums of
small whole numbers, exact in FP32."""
import ctypes

import pytest

from quiqbox_amd import _lib

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(2, 70_000_003), (17, 70_000_003), (17, 16 * 65536), (17, 16 * 65536 + 1),
                                       (16, 33), (0, 5), (70, 17)])
def test_wide_column_sums(rows, cols):
    X = (torch.arange(rows * cols, device="cuda", dtype=torch.int64) % 1013).to(torch.float32).view(rows, cols)
    X = X if rows else torch.zeros(1, device="cuda")
    out = torch.full((cols,), -1.0, dtype=torch.float32, device="cuda")
    print("[gpu-test] %d x %d" % (rows, cols), flush=True)
    _lib.check(_lib.load().qbx_mlp_colsum(rows, cols, ctypes.c_void_p(X.data_ptr()), ctypes.c_void_p(out.data_ptr()),
                                          None))
    torch.cuda.synchronize()
    ref = torch.zeros(cols, dtype=torch.float32, device="cuda")
    for r in range(rows):
        ref += X[r]
    assert torch.equal(out, ref)
