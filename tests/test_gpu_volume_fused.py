"""The fused kernels for two terms of d + 1 = 4 and 5 (volumes: position, position and
intensity), in both orders: the same bits as the generic kernels (inference, step,
gradients), sizes around a wave's pixels, and the oracle's results."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [(3, 4), (4, 3)])
@pytest.mark.parametrize("L", [2, 4, 5, 21])
@pytest.mark.parametrize("N", [1, 63, 65, 1009])
def test_volume_terms_bitwise(order, L, N):
    from oracle import pyoracle as po
    from pydensecrf_amd import capi
    rng = np.random.default_rng(N + L)
    U = rng.standard_normal((L, N)).astype(np.float32)
    gt = rng.integers(0, L, N).astype(np.int16)
    feats = [(rng.standard_normal((d, N)) * 1.5).astype(np.float32) for d in order]
    compat = [3.0, (-np.eye(L) + rng.normal(0, 0.1, (L, L))).astype(np.float32)]
    norms = [capi.NORMALIZE_SYMMETRIC, capi.NORMALIZE_AFTER]
    outs = []
    for mode in (0, 1):
        g = capi.Model.create(N, L)
        g.set_unary(U)
        for f, c, nt in zip(feats, compat, norms):
            g.add_pairwise(f, c, ntype=nt)
        g.set_meanfield_kernel(mode)
        assert g.splat_layout()["meanfield"] == (1 if mode == 0 else 0)
        outs.append([g.inference(3)] + list(g.gradient(3, gt, kernel=True)))
    for a, b in zip(*outs):
        assert np.array_equal(np.asarray(a), np.asarray(b))
    o = po.OracleCRF(N=N, L=L)
    o.set_unary(U)
    for f, c, nt in zip(feats, compat, norms):
        o.add_pairwise(f, c, ntype=nt)
    assert np.abs(outs[0][0] - o.inference(3)).max() <= 1e-5
