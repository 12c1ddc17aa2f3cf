"""Calls on a layout that splat_layout() alone has built: the allocation-free inference
needs every buffer of it, the iterate of padded rows (19 labels: rows of 20) among them."""
import numpy as np
import pytest

from pydensecrf_amd import capi
from tests.helpers import image_case

pytestmark = pytest.mark.gpu


def _model(W, H, L, img, tile=None):
    m = capi.Model.create_2d(W, H, L)
    if tile:
        m.set_splat_tile(tile)
    m.add_gaussian(3.0, 3.0, 3.0)
    m.add_bilateral(40.0, 40.0, 13.0, 13.0, 13.0, img, 10.0)
    return m


def _run(m, U, n, noalloc):
    import torch
    Q = torch.full((m.N * m.L,), -1.0, device="cuda", dtype=torch.float32)
    f = m.inference_device_noalloc if noalloc else m.inference_device
    f(n, Q.data_ptr(), U.data_ptr(), torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return Q.cpu().numpy().view(np.int32)


@pytest.mark.parametrize("L", [5, 10, 19, 21, 131])
def test_noalloc_after_splat_layout(L):
    import torch
    W, H = 50, 37
    img, U, _ = image_case(W, H, L, seed=L)
    U = torch.from_numpy(np.ascontiguousarray(U.T)).cuda()
    m = _model(W, H, L, img)
    m.splat_layout()
    got = [_run(m, U, n, True) for n in (0, 1, 3)]
    other = _model(W, H, L, img)
    for n, q in zip((0, 1, 3), got):
        assert np.array_equal(q, _run(other, U, n, False)), n


def test_noalloc_after_the_tiled_splat_no_longer_fits():
    import torch
    W, H, L, tile = 60, 45, 19, 26
    img, U, _ = image_case(W, H, L, seed=1)
    U = torch.from_numpy(np.ascontiguousarray(U.T)).cuda()
    m = _model(W, H, L, img, tile)
    _run(m, U, 2, False)
    assert m.splat_layout()["tiled"] == 1
    m.set_splat_chunk(1)  # a segment per entry: more than the LDS holds
    assert m.splat_layout()["tiled"] == 0
    got = _run(m, U, 2, True)
    other = _model(W, H, L, img, tile)
    other.set_splat_chunk(1)
    assert np.array_equal(got, _run(other, U, 2, False))
