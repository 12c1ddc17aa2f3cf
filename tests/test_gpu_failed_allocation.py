"""A device allocation that fails is reported by the call that needed it, and by no later
one: the runtime keeps its last error until it is read, and the kernels' launch checks
would take it for their own.  What the failed call had begun to replace is gone."""
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


def test_backward_after_a_forward_that_failed():
    import torch
    W, H, L = 64, 48, 21
    _, U, _ = image_case(W, H, L, seed=2)
    m = capi.Model.create_2d(W, H, L)
    m.set_unary(U)
    m.add_gaussian(3.0, 3.0, 3.0)
    Q, dU = (torch.ones(W * H * L, device="cuda") for _ in range(2))
    m.forward_device(2, None, Q.data_ptr())
    m.backward_device(Q.data_ptr(), dU.data_ptr())
    with pytest.raises(MemoryError):
        m.forward_device(10 ** 7, None, Q.data_ptr())
    with pytest.raises(capi.DCRFError, match="preceding training forward"):
        m.backward_device(Q.data_ptr(), dU.data_ptr())
