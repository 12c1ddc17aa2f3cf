"""dcrf_get_lattice reads a model: its normalisers do not build the layout, and are those
the layout has (bit for bit), for every normalisation, segment length and blur form."""
import numpy as np
import pytest

from pydensecrf_amd import capi
from tests.helpers import image_case

pytestmark = pytest.mark.gpu


def _model(W, H, L, img, ntype, chunk=0):
    m = capi.Model.create_2d(W, H, L)
    m.set_splat_chunk(chunk)
    m.add_gaussian(3.0, 3.0, 3.0, ntype=ntype)
    m.add_bilateral(40.0, 40.0, 13.0, 13.0, 13.0, img, 10.0, ntype=ntype)
    return m


@pytest.mark.parametrize("ntype", range(4))
@pytest.mark.parametrize("chunk", [0, 1, 1 << 20])
def test_normalisers_without_a_layout(ntype, chunk):
    W, H, L = 150, 131, 4
    img, _, _ = image_case(W, H, L, seed=3)
    m = _model(W, H, L, img, ntype, chunk)
    before = [m.lattice(k)["norm"] for k in range(2)]
    m.splat_layout()
    for pairs in (1, 0):
        m.set_blur_pairs(pairs)
        m.splat_layout()
        for k in range(2):
            assert np.array_equal(m.lattice(k)["norm"].view(np.int32), before[k].view(np.int32))


def test_lattice_query_leaves_the_layout_unbuilt():
    import torch
    W, H, L = 64, 48, 21  # (21 labels: rows without padding)
    img, _, _ = image_case(W, H, L, seed=3)
    m = _model(W, H, L, img, capi.NORMALIZE_SYMMETRIC)
    m.lattice(0)
    with pytest.raises(capi.DCRFError, match="layout is not built"):
        m.inference_device_noalloc(1, torch.zeros(W * H * L, device="cuda").data_ptr())
