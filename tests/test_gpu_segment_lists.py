"""The splat's segment and recombination lists, built on the device with the layout.

They are rebuilt whenever a term, a parameter or the segment length changes, also when the
lattices are asked for before any inference.  Segment lengths 1 (a partial row per
entry: vertices of thousands of them), the default and one above every run; row shapes
with in-wave runs, with four lanes per segment, padded, and with groups wider than a wave;
four tiles, the last ones ragged, and padding lanes' vertices without entries.
"""
import numpy as np
import pytest

from oracle import pyoracle as po
from pydensecrf_amd import capi
from tests.helpers import image_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chunk", [1, 32, 1 << 20])
@pytest.mark.parametrize("L", [2, 5, 21, 300])
def test_lists_follow_the_terms(L, chunk):
    W, H = 150, 131
    img, U, _ = image_case(W, H, L, seed=17)

    def bilateral(m):
        m.add_bilateral(60.0, 60.0, 20.0, 20.0, 20.0, img, 4.0)

    g = capi.Model.create_2d(W, H, L)
    o = po.OracleCRF(W=W, H=H, L=L)
    g.set_splat_chunk(chunk)
    for m in (g, o):
        m.set_unary(U)
        m.add_gaussian(3.0, 3.0, 3.0)
    norm = g.lattice(0)["norm"]  # before any inference
    # sums of positive products in another order: the bar of the other normaliser tests
    assert np.abs(norm - o.norm(0)).max() <= 2e-6 * np.abs(o.norm(0)).max()
    assert np.abs(g.inference(1) - o.inference(1)).max() <= 1e-5
    for m in (g, o):
        bilateral(m)
    got = g.inference(2)
    assert np.abs(got - o.inference(2)).max() <= 1e-5
    assert np.array_equal(g.lattice(0)["norm"].view(np.int32), norm.view(np.int32))
    fresh = capi.Model.create_2d(W, H, L)
    fresh.set_unary(U)
    fresh.add_gaussian(3.0, 3.0, 3.0)
    bilateral(fresh)
    fresh.inference(1)
    fresh.set_splat_chunk(chunk)  # the lists are rebuilt
    assert np.array_equal(np.asarray(fresh.inference(2)).view(np.int32), np.asarray(got).view(np.int32))
