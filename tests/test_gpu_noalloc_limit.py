"""The limit of the allocation-free inference does not depend on the splat's form: 8
labels, segments of one entry (a quad per segment: a partial row per 8 of them, 69 MB of
rows; one per 32 without quads, 17 MB) is taken."""
import numpy as np
import pytest

from pydensecrf_amd import capi

pytestmark = pytest.mark.gpu


def test_quad_rows_do_not_count():
    import torch
    W = H = 2400
    L = 8
    m = capi.Model.create_2d(W, H, L)
    m.set_splat_chunk(1)
    m.add_gaussian(30.0, 30.0, 3.0)
    lay = m.splat_layout()
    _, V = m.term_info(0)
    assert (lay["partials"] + 2 * (V + 1)) * L * 4 > 64 << 20
    g = torch.Generator(device="cuda").manual_seed(0)
    U = torch.rand(W * H, L, device="cuda", generator=g)
    Q = [torch.full((W * H, L), float("nan"), device="cuda") for _ in range(2)]
    stream = torch.cuda.current_stream().cuda_stream
    m.inference_device_noalloc(2, Q[0].data_ptr(), U.data_ptr(), stream)
    m.inference_device(2, Q[1].data_ptr(), U.data_ptr(), stream)
    torch.cuda.synchronize()
    assert torch.equal(Q[0].view(torch.int32), Q[1].view(torch.int32))
    assert bool(torch.isfinite(Q[0]).all())
