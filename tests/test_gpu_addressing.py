"""Row addressing of the splat and the fused per-pixel kernels: 24-bit row numbers and
32-bit byte offsets where they fit, 64-bit offsets above.  The two forms do the same
arithmetic, so an instance of a batch that is past the limit gives the bits it gives
alone, below it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _model(shapes, L, sxy, unaries):
    from pydensecrf_amd import capi
    m = capi.Model.create_batch_2d([w for w, _ in shapes], [h for _, h in shapes], L)
    for i, U in enumerate(unaries):
        m.set_unary_instance(i, U)
    m.add_gaussian(sxy, sxy, 2.0)
    return m


@pytest.mark.parametrize("shapes,sxy,what", [
    # 2^24 pixels in the first instance: the second starts past the limit
    ([(4096, 4096), (45, 31)], 200.0, "pixels"),
    # isolated pixels, three vertices each: more than 2^24 vertex rows in all
    ([(450, 450)] * 28 + [(45, 31)], 0.2, "vertices"),
])
def test_wide_rows_bitwise(shapes, sxy, what):
    L = 1 if what == "vertices" else 2
    rng = np.random.default_rng(len(shapes))
    U = [rng.standard_normal((L, w * h), dtype=np.float32) for w, h in shapes]
    both = _model(shapes, L, sxy, U)
    _, V = both.term_info(0)
    assert both.N > 1 << 24 if what == "pixels" else V > 1 << 24
    Q = both.inference(2)
    both.close()
    at = np.cumsum([0] + [w * h for w, h in shapes])
    for i in (0, len(shapes) - 1):
        alone = _model([shapes[i]], L, sxy, [U[i]])
        assert alone.N <= 1 << 24 and alone.term_info(0)[1] < 1 << 24
        got = np.ascontiguousarray(Q[:, at[i]:at[i + 1]])
        assert np.array_equal(got.view(np.int32), np.ascontiguousarray(alone.inference(2)).view(np.int32)), i
        alone.close()
