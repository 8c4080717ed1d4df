"""The gradient kernels' sums straight to the outputs, where a block's LDS copy of them
does not fit: the same central differences as test_gpu_gradient_sinks, on a basis whose
outputs exceed the copy's limit by themselves, whatever the Boys rows beside it take.  The
limit is read from the kernels' header, so that the case stays on that path."""
import os
import re

import pytest

import test_gpu_gradient_sinks as sinks

pytestmark = pytest.mark.gpu
HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "quiqbox.jl_amd", "csrc",
                      "qbx_grad.h")


def test_gradient_with_outputs_beyond_the_lds_copy():
    with open(HEADER) as f:
        text = f.read()
    limit = 1024 * int(re.search(r"GRAD_LDS_MAX = (\d+) \* 1024;", text).group(1))
    assert "shm <= (size_t)GRAD_LDS_MAX ? (int)n : 0" in text
    per_shell = 8 * (2 * 8 + 3)           # 8 primitives: two sums each, three of the centre
    n = limit // per_shell + 10
    print("[gpu-test] %d shells, %d B of outputs, limit %d B" % (n, n * per_shell, limit), flush=True)
    sinks.test_gradient_against_central_differences(n, 30.0, [[(0, 8)]])
