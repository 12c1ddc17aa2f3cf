"""64-bit row offsets at three and four labels per lane: the splat of whole lane groups, the
fused mean-field and adjoint kernels, with and without a Matrix compatibility.  An instance
of a batch past the 24-bit row number or the 4 GiB of 32-bit offsets gives the bits it gives
alone, below both, in the inference, the training forward and the backward."""
import pytest

from pydensecrf_amd import capi

pytestmark = pytest.mark.gpu


def _model(shapes, L, sxy, compat):
    m = capi.Model.create_batch_2d([w for w, _ in shapes], [h for _, h in shapes], L)
    m.add_gaussian(sxy, sxy, compat)
    return m


def _run(m, U, dQ):
    import torch
    stream = torch.cuda.current_stream().cuda_stream
    Q, F, dU = (torch.full_like(U, float("nan")) for _ in range(3))
    m.inference_device(2, Q.data_ptr(), U.data_ptr(), stream)
    m.forward_device(1, U.data_ptr(), F.data_ptr(), stream=stream)
    m.backward_device(dQ.data_ptr(), dU.data_ptr(), stream=stream)
    torch.cuda.synchronize()
    return Q, F, dU


@pytest.mark.parametrize("shapes,L,sxy,what,matrix", [
    ([(4096, 4096), (45, 31)], 9, 200.0, "pixels", False),        # 2^24 pixels before the last instance
    ([(4096, 4096), (45, 31)], 9, 200.0, "pixels", True),
    ([(450, 450)] * 28 + [(45, 31)], 9, 0.2, "vertices", False),  # 2^24 vertices (three to a pixel)
    ([(450, 450)] * 28 + [(45, 31)], 9, 0.2, "vertices", True),
    ([(2100, 2050), (45, 31)], 256, 100.0, "pixels", False),      # 4 GiB of rows
    ([(450, 450)] * 8 + [(45, 31)], 256, 0.2, "vertices", False),
])
def test_wide_rows_bitwise(shapes, L, sxy, what, matrix):
    import torch
    g = torch.Generator(device="cuda").manual_seed(L)
    compat = 2.0
    if matrix:
        compat = (torch.eye(L) + 0.1 * torch.rand(L, L, generator=torch.Generator().manual_seed(1))).numpy()
    N = sum(w * h for w, h in shapes)
    U, dQ = (torch.randn(N, L, device="cuda", generator=g) for _ in range(2))
    both = _model(shapes, L, sxy, compat)
    rows = N if what == "pixels" else both.term_info(0)[1]
    assert rows > 1 << 24 or rows * L * 4 > 1 << 32
    got = _run(both, U, dQ)
    both.close()
    at = [0]
    for w, h in shapes:
        at.append(at[-1] + w * h)
    for i in (0, len(shapes) - 1):
        alone = _model([shapes[i]], L, sxy, compat)
        assert alone.N <= 1 << 24 and alone.term_info(0)[1] < 1 << 24
        part = slice(at[i], at[i + 1])
        ref = _run(alone, U[part].contiguous(), dQ[part].contiguous())
        alone.close()
        for a, b in zip(got, ref):
            assert torch.equal(a[part].view(torch.int32), b.view(torch.int32)), i
            assert bool(torch.isfinite(b).all())
