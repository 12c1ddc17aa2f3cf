"""Label counts that neither 4 nor 3 divides: gathered rows are padded to four labels per
lane (5 -> 8, 19 -> 20, 257 -> 260, ...), the caller's rows are not.  Every path that
reads one kind and writes the other: inference with the fused, the generic and the
pixel-run kernels and Q in blocks (the same bits), step, the allocation-free form, KL,
messages and gradients, against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _models(W, H, L, seed):
    from oracle import pyoracle as po
    from pydensecrf_amd import capi, synthetic as syn
    img, U, gt = syn.make_image(W, H, L=L, sites=6, seed=seed)
    rng = np.random.default_rng(seed)
    c1 = rng.uniform(1, 4, L).astype(np.float32)
    c2 = (-2 * np.eye(L) + rng.normal(0, 0.05, (L, L))).astype(np.float32)
    g = capi.Model.create_2d(W, H, L)
    o = po.OracleCRF(W=W, H=H, L=L)
    for m in (g, o):
        m.set_unary(U)
        m.add_gaussian(3.0, 3.0, -c1)
        m.add_bilateral(20.0, 20.0, 13.0, 13.0, 13.0, img, c2)
    return g, o, gt


@pytest.mark.parametrize("L", [5, 7, 10, 13, 19, 22, 65, 257])
def test_padded_labels(L):
    import torch
    W, H, n = 29, 18, 3
    g, o, gt = _models(W, H, L, 500 + L)
    Q = np.ascontiguousarray(g.inference(n))
    Qo = o.inference(n)
    assert np.abs(Q - Qo).max() <= 1e-5
    S = g.start()
    for _ in range(n):
        S, t1, t2 = g.step(S)
    assert np.array_equal(Q.view(np.int32), np.ascontiguousarray(S).view(np.int32))
    assert np.isfinite(t1).all() and np.isfinite(t2).all()
    dev = torch.full((W * H, L), -1.0, device="cuda")
    dev2 = torch.full((W * H + 1, L), -1.0, device="cuda")
    g.inference_device(n, dev.data_ptr())
    g.inference_device_noalloc(n, dev2.data_ptr())
    torch.cuda.synchronize()
    assert np.array_equal(dev.cpu().numpy().T.copy().view(np.int32), Q.view(np.int32))
    assert torch.equal(dev2[:-1], dev) and bool((dev2[-1] == -1.0).all())  # nothing written past Q
    for mode in (3, 1):
        g.set_meanfield_kernel(mode)
        assert np.array_equal(np.ascontiguousarray(g.inference(n)).view(np.int32), Q.view(np.int32)), mode
    g.set_meanfield_kernel(0)
    g.set_q_blocks(True)
    assert np.array_equal(np.ascontiguousarray(g.inference(n)).view(np.int32), Q.view(np.int32))
    g.set_q_blocks(False)
    assert abs(g.kl(Qo) - o.kl(Qo)) <= 1e-5 * max(1.0, abs(o.kl(Qo)))
    for k in (0, 1):
        np.testing.assert_allclose(g.apply(k, Qo, True), o.apply(k, Qo, True), rtol=1e-5, atol=1e-5)
    r, ug, cg, kg, kp = g.gradient(n, gt, kernel=True)
    ro, ugo, cgo, kpo = o.gradient(n, gt, kernel=True)
    assert abs(r - ro) <= 1e-5 * abs(ro)
    for a, b, bar in ((ug, ugo, 1e-4), (cg, cgo, 1e-4), (kp, kpo, 1e-3)):  # the configuration sweep's bars
        assert np.abs(a - b).max() <= bar * np.abs(b).max() + 1e-6
