"""A device allocation that fails is reported by the call that needed it, and by no later
one: the runtime keeps its last error until it is read, and the kernels' launch checks
would take it for their own."""
import numpy as np
import pytest

from pydensecrf_amd import capi
from tests.helpers import image_case

pytestmark = pytest.mark.gpu


def test_failed_allocation_leaves_no_error_behind():
    import torch
    W, H, L = 64, 48, 21
    img, U, _ = image_case(W, H, L, seed=2)
    m = capi.Model.create_2d(W, H, L)
    m.set_unary(U)
    m.add_gaussian(3.0, 3.0, 3.0)
    ref = m.inference(2)
    Q = torch.empty(W * H * L, device="cuda")
    with pytest.raises(MemoryError):  # 10^7 stored iterates: 2.6 TB
        m.forward_device(10 ** 7, None, Q.data_ptr())
    m.add_bilateral(40.0, 40.0, 13.0, 13.0, 13.0, img, 10.0)
    got = m.inference(2)
    assert got.shape == ref.shape and np.isfinite(got).all()
