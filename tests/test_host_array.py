"""Device-to-host copy of a statevector through pinned chunks."""
import os
import sys

import numpy as np
import pytest
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (ROOT, os.path.join(ROOT, "qiskit-blackwell_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, (1 << 17) - 1, 1 << 17, (1 << 21) + 3, (1 << 22) + (1 << 20) + 7, 1 << 23])
def test_host_array_is_the_tensor(n):
    """Below and at the first chunked size, one chunk, a ragged last one and
    more chunks than staging buffers: every amplitude, in an array of its own."""
    from blackwell_backend.simulator import host_array
    g = torch.Generator(device="cuda:0").manual_seed(n)
    t = torch.view_as_complex(torch.randn(n, 2, device="cuda:0", generator=g))
    a = host_array(t)
    t2 = t * 2
    b = host_array(t2)
    assert a.dtype == np.complex64 and a.shape == (n,) and a.flags.writeable
    assert np.array_equal(a, t.cpu().numpy()) and np.array_equal(b, t2.cpu().numpy())
