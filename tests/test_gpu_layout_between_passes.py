"""A layout rebuilt between a training forward and its backward: where the LDS-tiled splat
stops or starts fitting, the stride of the gathered rows changes (19 labels: 19 or 20),
and the forward's stored iterates move to the new one."""
import numpy as np
import pytest

from pydensecrf_amd import capi
from tests.helpers import image_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("matrix", [False, True])
@pytest.mark.parametrize("before,after", [(0, 1), (1, 0)])
@pytest.mark.parametrize("n", [1, 5])
def test_row_stride_changes_between_forward_and_backward(n, before, after, matrix):
    import torch
    W, H, L = 60, 45, 19
    img, U, _ = image_case(W, H, L, seed=4)
    rng = np.random.default_rng(5)
    cb = 10.0 * np.eye(L, dtype=np.float32) + rng.random((L, L), dtype=np.float32) if matrix else 10.0
    m = capi.Model.create_2d(W, H, L)
    m.set_splat_tile(26)
    m.add_gaussian(3.0, 3.0, 3.0)
    m.add_bilateral(40.0, 40.0, 13.0, 13.0, 13.0, img, cb)
    U = torch.from_numpy(np.ascontiguousarray(U.T)).cuda()
    dQ = torch.from_numpy(rng.standard_normal((W * H, L)).astype(np.float32)).cuda()
    stream = torch.cuda.current_stream().cuda_stream

    def forward(chunk):
        m.set_splat_chunk(chunk)
        Q = torch.empty(W * H, L, device="cuda")
        m.forward_device(n, U.data_ptr(), Q.data_ptr(), stream=stream)
        return m.splat_layout()["tiled"]

    def backward():
        dU = torch.full((W * H, L), float("nan"), device="cuda")
        dc = torch.full((1 + (L * L if matrix else 1),), float("nan"), device="cuda")  # raw layout
        m.backward_device(dQ.data_ptr(), dU.data_ptr(), dc.data_ptr(), stream=stream)
        torch.cuda.synchronize()
        return dU.cpu().numpy(), dc.cpu().numpy()

    tiled = forward(before)
    ref = backward()
    forward(before)
    m.set_splat_chunk(after)
    assert m.splat_layout()["tiled"] == 1 - tiled
    got = backward()
    # the bar of the gradients against the oracle, whose order of summation differs too
    for a, b in zip(got, ref):
        assert np.abs(a - b).max() <= 1e-4 * np.abs(b).max()
