"""The splat of rows of one or two lanes (up to 8 labels), where several lanes share a
segment: segment lengths around the lane count and the batch (chunks of 1, 3, 4, 5, 31 to
33 and 100,000 contributors), against the oracle, forward and transposed; the LDS-tiled
form of the same sums as well."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [1, 2, 3, 4, 6, 8])
def test_split_splat_segments(L):
    from oracle import pyoracle as po
    from pydensecrf_amd import capi, synthetic as syn
    W, H = 61, 47
    img, U, _ = syn.make_image(W, H, L=L, sites=5, seed=700 + L)

    def model(tile):
        g = capi.Model.create_2d(W, H, L)
        if tile:
            g.set_splat_tile(tile)
        g.set_unary(U)
        g.add_gaussian(3.0, 3.0, 3.0)
        g.add_bilateral(20.0, 20.0, 13.0, 13.0, 13.0, img, 10.0)
        return g

    o = po.OracleCRF(W=W, H=H, L=L)
    o.set_unary(U)
    o.add_gaussian(3.0, 3.0, 3.0)
    o.add_bilateral(20.0, 20.0, 13.0, 13.0, 13.0, img, 10.0)
    Qo, S = o.inference(3), o.start()
    g = model(0)
    for chunk in (1, 3, 4, 5, 31, 32, 33, 100000):
        g.set_splat_chunk(chunk)
        assert g.splat_layout()["tiled"] == 0
        assert np.abs(g.inference(3) - Qo).max() <= 1e-5, chunk
        np.testing.assert_allclose(g.apply(1, S, True), o.apply(1, S, True), rtol=1e-5, atol=1e-5)
    t = model(16)
    for chunk in (3, 32):
        t.set_splat_chunk(chunk)
        assert t.splat_layout()["tiled"] == 1
        assert np.abs(t.inference(3) - Qo).max() <= 1e-5, chunk
