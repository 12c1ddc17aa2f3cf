"""Cases for measuring the framework: what its users run, over the sizes they run it on.

A case is a dict of plain values.  ``kind`` says how the framework is called:

  infer   mean-field inference of a prepared 2-D model on device tensors
          (``capi.Model.inference_device``): the serving loop, one image's model in hand
  dropin  a new ``DenseCRF2D`` per image through the drop-in module, host arrays in and
          out: what a program written for the original API does
  batch   inference of a batch of images of uneven size (``BatchedDenseCRF2D``)
  train   a training step's forward and backward through ``CRFLayer`` (cross-entropy of
          the labels; gradients of the unary, the compatibilities and the term weights)
  volume  the same for a batch of 3-D volumes with explicit features (``BatchedDenseCRF``)
  learn   two learning steps that also move the kernel parameters: each sets new feature
          scales (the lattices are rebuilt) and runs forward and backward

All 2-D models have the Gaussian (sxy = 3) and the bilateral (sxy = 80, srgb = 13) term.
Images and unaries follow ``pydensecrf_amd.synthetic``: Voronoi regions of one colour
with pixel noise, -log softmax of noisy logits that favour the region's label, 30 % of
the regions mislabelled; here they are made on the GPU from the seed.

``exact`` evaluates the same model in 64 bits with plain torch.  The lattice (which
simplex a point falls into, its barycentric weights) is defined by float32 arithmetic,
so that part is done in float32 with the operations in their defined order; everything
from the splat on is in 64 bits.
"""
import math

import numpy as np
import torch

SXY_G, SXY_B, SRGB = 3.0, 80.0, 13.0
W_G, W_B = 3.0, 10.0
NORMS = {"no": 0, "before": 1, "after": 2, "symmetric": 3}


# ---------------------------------------------------------------- the cases
def listed():
    def infer(name, W, H, L, iters, compat="potts", norm="symmetric"):
        return dict(name=name, kind="infer", W=W, H=H, L=L, iters=iters, compat=compat, norm=norm)

    def dropin(name, W, H, L, iters):
        return dict(name=name, kind="dropin", W=W, H=H, L=L, iters=iters)

    def train(name, W, H, L, iters, compat):
        return dict(name=name, kind="train", W=W, H=H, L=L, iters=iters, compat=compat)

    return [
        # a thumbnail or a crop around a detection: launches and latency count
        infer("infer_64x48x21", 64, 48, 21, 5),
        # an ordinary photograph at the resolution segmentation networks put out
        infer("infer_320x213x21", 320, 213, 21, 5),
        # the benchmark's image: a full-size photograph, the label set of PASCAL VOC
        infer("infer_1024x768x21", 1024, 768, 21, 10),
        # foreground / background on a video frame: few labels, many pixels
        infer("infer_1920x1080x2", 1920, 1080, 2, 10),
        # odd sides and a prime label count, one weight per label, another normalisation
        infer("infer_1021x511x19", 1021, 511, 19, 10, "diagonal", "after"),
        # a folder of photographs of all sizes processed together
        dict(name="batch_16x21", kind="batch", n=16, lo=256, hi=1024, pick=1002, L=21, iters=10),
        # training with the CRF as a network's last layer, Potts terms, full-size image
        train("train_1024x768x21_potts", 1024, 768, 21, 10, "potts"),
        # the same with a learned label-pair matrix, on a training crop
        train("train_512x512x21_matrix", 512, 512, 21, 5, "matrix"),
        # training on 3-D scans: few labels, explicit features of 3 and 4 dimensions
        dict(name="volume_4x96x96x4", kind="volume", n=4, lo=32, hi=64, side=96, pick=1004, L=4, iters=10),
        # scripts of the original API: a new model per image, small and full size
        dropin("dropin_320x213x21", 320, 213, 21, 5),
        dropin("dropin_1024x768x21", 1024, 768, 21, 10),
        # learning the feature scales as well
        dict(name="learn_512x512x21", kind="learn", W=512, H=512, L=21, iters=5),
    ]


LABELS = (2, 3, 4, 5, 6, 7, 8, 11, 12, 16, 19, 21, 21, 27, 32, 40, 59, 80, 150)


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sides(rng, lo, hi, most):
    """Two sides between lo and hi, of at most `most` pixels together."""
    while True:
        W, H = _spread(rng, lo, hi), _spread(rng, lo, hi)
        if 1 / 3 <= W / H <= 3 and W * H <= most:
            return W, H


def draw(rng):
    kind = rng.choices(("infer", "dropin", "train", "volume", "batch", "learn"), (8, 3, 4, 2, 1, 1))[0]
    compat = rng.choice(("potts", "potts", "diagonal", "matrix"))
    if kind == "volume":
        return dict(kind=kind, n=rng.randint(1, 4), lo=16, hi=64, side=rng.randint(24, 96), pick=rng.randrange(1 << 20),
                    L=rng.choice((2, 3, 4, 5)) if compat == "potts" else 4, iters=rng.choice((5, 10)))
    if kind == "batch":
        return dict(kind=kind, n=rng.randint(2, 16), lo=100, hi=rng.randint(200, 1000), pick=rng.randrange(1 << 20),
                    L=rng.choice((2, 5, 19, 21)), iters=rng.choice((5, 10)))
    iters = rng.choice((5, 10))
    L = rng.choice(LABELS)
    # variables times labels within the full-size image's, so that none is larger
    most = 1024 * 768 * 21 // L
    if kind == "learn":
        L = rng.choice((2, 5, 12, 21))
        W, H = _sides(rng, 60, 512, 512 * 512)
        return dict(kind=kind, W=W, H=H, L=L, iters=5)
    if kind == "infer":
        W, H = _sides(rng, 40, 1920, most)
        return dict(kind=kind, W=W, H=H, L=L, iters=iters, compat=compat,
                    norm=rng.choice(("symmetric", "symmetric", "symmetric", "before", "after")))
    W, H = _sides(rng, 100, 1024, most)
    if kind == "train":
        return dict(kind=kind, W=W, H=H, L=L, iters=iters, compat=compat)
    return dict(kind=kind, W=W, H=H, L=L, iters=iters)


def _shapes(case):
    """The (W, H) or depths of a batch, from the case alone."""
    r = np.random.default_rng(case["pick"])
    if case["kind"] == "batch":
        return [(int(w), int(h)) for w, h in zip(r.integers(case["lo"], case["hi"] + 1, case["n"]),
                                                 r.integers(case["lo"], case["hi"] + 1, case["n"]))]
    return [int(z) for z in r.integers(case["lo"], case["hi"] + 1, case["n"])]


def work(case):
    """Inputs once, outputs once; the multiply-adds of splat, slice and compatibility and
    the softmax, per iteration (the blur depends on the lattice and is left out)."""
    kind, L, it = case["kind"], case["L"], case["iters"]
    if kind == "batch":
        N, d1 = sum(w * h for w, h in _shapes(case)), 9
    elif kind == "volume":
        N, d1 = sum(z * case["side"] ** 2 for z in _shapes(case)), 9
    else:
        N, d1 = case["W"] * case["H"], 9
    row = N * L * 4
    flops = it * N * L * (4 * d1 + 10 + (4 * L if case.get("compat") == "matrix" or kind == "learn" else 4))
    if kind == "dropin":
        return {"bytes": 2 * row + 3 * N, "flops": flops}
    if kind in ("infer", "batch"):
        return {"bytes": 2 * row + N * d1 * 8, "flops": flops}
    # training: unary in, Q and the unary's gradient out, labels; forward and adjoint
    one = {"bytes": 3 * row + N * 8 + N * d1 * 8, "flops": 2 * flops}
    if kind == "learn":
        return {"bytes": 2 * one["bytes"], "flops": 4 * one["flops"]}
    return one


# ---------------------------------------------------------------- inputs
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _regions(g, shape, sites):
    """Index of the nearest of `sites` random sites per grid cell, flat."""
    axes = [torch.arange(s, device="cuda", dtype=torch.float32) for s in shape]
    pos = [torch.rand(sites, generator=g, device="cuda") * s for s in shape]
    best = bestd = None
    for k in range(sites):
        dist = 0.0
        for i, (a, p) in enumerate(zip(axes, pos)):
            dist = dist + ((a - p[k]) ** 2).reshape([-1 if j == i else 1 for j in range(len(shape))])
        if best is None:
            best, bestd = torch.zeros(dist.shape, dtype=torch.int64, device="cuda"), dist
        else:
            best = torch.where(dist < bestd, k, best)
            bestd = torch.minimum(dist, bestd)
    return best.reshape(-1)


def _unary(g, region, sites, L):
    """Unary (N, L) and the true labels (N,) int64: 30 % of the regions show another label."""
    true = torch.randint(0, L, (sites,), generator=g, device="cuda")
    wrong = torch.rand(sites, generator=g, device="cuda") < 0.3
    other = torch.randint(0, max(L - 1, 1), (sites,), generator=g, device="cuda")
    shown = torch.where(wrong, other + (other >= true).long(), true).clamp_(max=L - 1)
    logits = torch.randn((region.numel(), L), generator=g, device="cuda")
    logits.scatter_add_(1, shown[region][:, None], torch.full((region.numel(), 1), 3.0, device="cuda"))
    return -torch.log_softmax(logits, 1), true[region]


def _image(W, H, L, seed):
    """Image (H, W, 3) uint8, unary (N, L) float32, labels (N,) int64, on the GPU."""
    g = _generator(seed)
    sites = min(48, max(12, W * H // 16384))
    region = _regions(g, (H, W), sites)
    colour = torch.randint(0, 256, (sites, 3), generator=g, device="cuda").float()
    noise = torch.randn((W * H, 3), generator=g, device="cuda")
    img = (colour[region] + 8.0 * noise).round_().clamp_(0, 255).to(torch.uint8).reshape(H, W, 3)
    U, gt = _unary(g, region, sites, L)
    return img, U, gt


def _volume(Z, side, L, seed):
    """Gaussian features (3, N) and bilateral features (4, N), host float32; unary, labels."""
    g = _generator(seed)
    region = _regions(g, (Z, side, side), 20)
    level = torch.rand(20, generator=g, device="cuda")
    vol = level[region] + 0.05 * torch.randn(region.numel(), generator=g, device="cuda")
    U, gt = _unary(g, region, 20, L)
    pos = np.stack(np.meshgrid(np.arange(Z), np.arange(side), np.arange(side), indexing="ij"))
    pos = pos.reshape(3, -1).astype(np.float32)
    inten = vol.cpu().numpy().reshape(1, -1)
    fg = np.ascontiguousarray(pos / np.float32(3))
    fb = np.ascontiguousarray(np.concatenate([pos / np.float32(40), inten / np.float32(0.1)]))
    return fg, fb, U, gt


def _compat(case, seed):
    """The two terms' compatibilities as a user gives them, and the term weights."""
    L, kind = case["L"], case.get("compat", "potts")
    r = np.random.default_rng(seed)
    if case["kind"] == "learn":
        kind = "matrix"
    if kind == "matrix":
        c = [(-np.eye(L) + r.normal(0, 0.1, (L, L))).astype(np.float32) for _ in range(2)]
        return c, [W_G, W_B]
    if case["kind"] == "volume":
        c = (-1 - r.random(L)).astype(np.float32)
        return [c, c - np.float32(0.5)], [1.0, 2.0]
    if kind == "diagonal":
        return [(-w * (0.75 + 0.5 * r.random(L))).astype(np.float32) for w in (W_G, W_B)], [1.0, 1.0]
    return [W_G, W_B], [1.0, 1.0]


def _folded(case, seed):
    """The compatibilities with the term weights multiplied in (inference has no others)."""
    c, w = _compat(case, seed)
    return [a * np.float32(b) if isinstance(a, np.ndarray) else a * b for a, b in zip(c, w)]


def _host(t):
    return np.ascontiguousarray(t.cpu().numpy())


# ---------------------------------------------------------------- prepare and run
def prepare(case, seed):
    kind, L, it = case["kind"], case["L"], case["iters"]
    if kind == "dropin":
        img, U, _ = _image(case["W"], case["H"], L, seed)
        return dict(kind=kind, W=case["W"], H=case["H"], L=L, iters=it, img=_host(img), U=_host(U.t().contiguous()))
    from pydensecrf_amd import capi
    if kind == "infer":
        img, U, _ = _image(case["W"], case["H"], L, seed)
        c = _folded(case, seed)
        norm = NORMS[case["norm"]]
        m = capi.Model.create_2d(case["W"], case["H"], L)
        m.add_gaussian(SXY_G, SXY_G, c[0], ntype=norm)
        m.add_bilateral(SXY_B, SXY_B, SRGB, SRGB, SRGB, _host(img), c[1], ntype=norm)
        return dict(kind=kind, model=m, U=U, Q=torch.empty_like(U), iters=it)
    if kind == "batch":
        from pydensecrf_amd.batched import BatchedDenseCRF2D
        shapes = _shapes(case)
        imgs, Us = [], []
        for i, (w, h) in enumerate(shapes):
            img, U, _ = _image(w, h, L, seed * 64 + i)
            imgs.append(_host(img))
            Us.append(_host(U.t().contiguous()))
        b = BatchedDenseCRF2D(shapes, L)
        b.setUnaryEnergy(Us)
        b.addPairwiseGaussian(sxy=SXY_G, compat=W_G)
        b.addPairwiseBilateral(sxy=SXY_B, srgb=SRGB, rgbims=imgs, compat=W_B)
        return dict(kind=kind, batch=b, Q=torch.empty((b.N, L), device="cuda"), iters=it)
    from pydensecrf_amd.autograd import CRFLayer
    c, w = _compat(case, seed)
    if kind == "volume":
        from pydensecrf_amd.batched import BatchedDenseCRF
        vols = [_volume(z, case["side"], L, seed * 64 + i) for i, z in enumerate(_shapes(case))]
        b = BatchedDenseCRF([v[2].shape[0] for v in vols], L)
        b.addPairwiseEnergy([v[0] for v in vols], c[0])
        b.addPairwiseEnergy([v[1] for v in vols], c[1])
        model, U, gt = b.model, torch.cat([v[2] for v in vols]), torch.cat([v[3] for v in vols])
    else:
        img, U, gt = _image(case["W"], case["H"], L, seed)
        model = capi.Model.create_2d(case["W"], case["H"], L)
        model.add_gaussian(SXY_G, SXY_G, c[0])
        model.add_bilateral(SXY_B, SXY_B, SRGB, SRGB, SRGB, _host(img), c[1])
    layer = CRFLayer(model, it, c, kweights=w, learn_kernel=kind == "learn")
    s = dict(kind=kind, layer=layer, U=U.requires_grad_(True), gt=gt)
    if kind == "learn":
        s["scales"] = torch.from_numpy(_scales(seed)).cuda()
    return s


def _scales(seed):
    """Two vectors of feature scales, as a minimiser's steps from the unit scales."""
    r = np.random.default_rng(seed + 1)
    return (1 + 0.02 * r.standard_normal((2, 7))).astype(np.float32)


def _loss(Q, gt):
    """Cross-entropy of the labels, with the usual guard against the log of nothing."""
    return -torch.log(Q.gather(1, gt[:, None]) + 1e-12).mean()


def _step(s):
    s["U"].grad = None
    s["layer"].zero_grad(set_to_none=True)
    Q = s["layer"](s["U"])
    _loss(Q, s["gt"]).backward()
    return [Q.detach(), s["U"].grad, s["layer"].compat.grad, s["layer"].kweights.grad]


def run(s):
    kind = s["kind"]
    if kind == "infer":
        s["model"].inference_device(s["iters"], s["Q"].data_ptr(), s["U"].data_ptr(), torch.cuda.current_stream().cuda_stream)
        return s["Q"]
    if kind == "batch":
        s["batch"].inference_device(s["iters"], s["Q"].data_ptr(), torch.cuda.current_stream().cuda_stream)
        return s["Q"]
    if kind == "dropin":
        import pydensecrf_amd.densecrf as dcrf
        d = dcrf.DenseCRF2D(s["W"], s["H"], s["L"])
        d.setUnaryEnergy(s["U"])
        d.addPairwiseGaussian(sxy=SXY_G, compat=W_G)
        d.addPairwiseBilateral(sxy=SXY_B, srgb=SRGB, rgbim=s["img"], compat=W_B)
        return np.asarray(d.inference(s["iters"]))
    if kind != "learn":
        return _step(s)
    out = []
    for scales in s["scales"]:
        with torch.no_grad():
            s["layer"].kparams.copy_(scales)
        out += _step(s) + [s["layer"].kparams.grad]
    return out


# ---------------------------------------------------------------- the same in 64 bits
class _Lattice:
    """The permutohedral lattice of features f (d, N), float32 on the host."""

    def __init__(self, f):
        d, N = f.shape
        d1 = d + 1
        f = torch.from_numpy(np.ascontiguousarray(f))
        pad = -N % 4  # points come in blocks of four, the missing ones at the origin
        f = torch.cat([f, torch.zeros((d, pad))], 1)
        inv_std = np.float32(math.sqrt(2.0 / 3.0) * d1)
        scale = [torch.tensor(np.float32(1.0 / math.sqrt((i + 2.0) * (i + 1.0)) * float(inv_std))) for i in range(d)]
        inv_d1 = torch.tensor(np.float32(1.0) / np.float32(d1))
        # onto the plane, the nearest remainder-0 point, the ranks of the differences
        elev, sm = [None] * d1, torch.zeros(N + pad)
        for j in range(d, 0, -1):
            cf = f[j - 1] * scale[j - 1]
            elev[j] = sm - cf * torch.tensor(float(j))
            sm = sm + cf
        elev[0] = sm
        rem0, total = [], torch.zeros(N + pad)
        for i in range(d1):
            v = torch.round(elev[i] * inv_d1)
            rem0.append(v * torch.tensor(float(d1)))
            total = total + v
        diff = [elev[i] - rem0[i] for i in range(d1)]
        rank = [torch.zeros(N + pad) for _ in range(d1)]
        for i in range(d):
            for j in range(i + 1, d1):
                less = (diff[i] < diff[j]).float()
                rank[i] = rank[i] + less
                rank[j] = rank[j] + (1.0 - less)
        for i in range(d1):
            rank[i] = rank[i] + total
            move = (rank[i] < 0).float() * d1 - (rank[i] >= d1).float() * d1
            rank[i] = rank[i] + move
            rem0[i] = rem0[i] + move
        rank = torch.stack(rank, 1).long()
        rem0 = torch.stack(rem0, 1)
        # barycentric weights: v by rank, then differences
        v = (torch.stack(elev, 1) - rem0) * inv_d1
        by = torch.zeros_like(v).scatter_(1, rank, v)
        bary = torch.empty_like(v)
        for r in range(1, d1):
            bary[:, r] = by[:, d - r] - by[:, d - r + 1]
        bary[:, 0] = by[:, d] + (1.0 + (0.0 - by[:, 0]))
        rem0, rank = rem0.long().cuda(), rank.cuda()
        keys = torch.stack([rem0[:, :d] + torch.where(rank[:, :d] <= d - r, r, r - d1) for r in range(d1)], 1)
        # one number per key, with room for the neighbours' moves
        lo = keys.reshape(-1, d).amin(0) - d1
        span = keys.reshape(-1, d).amax(0) + d1 - lo + 1
        stride = [1]
        for s in span.tolist():
            stride.append(stride[-1] * s)
        assert stride[-1] < 1 << 62
        stride = torch.tensor(stride[:-1], device="cuda")
        uniq, off = torch.unique(((keys - lo) * stride).sum(-1), return_inverse=True)
        V = uniq.numel()
        self.d, self.N, self.V = d, N, V
        self.off = off[:N]
        self.rank = rank[:N]
        self.bary = bary[:N].cuda().double()
        # neighbours along each axis; V is the row of zeros of an absent vertex
        self.nbr = []
        one = stride.sum()
        for j in range(d1):
            move = stride[j] * d1 - one if j < d else -one
            pair = []
            for m in (move, -move):
                at = torch.searchsorted(uniq, uniq + m).clamp_(max=V - 1)
                at = torch.where(uniq[at] == uniq + m, at, V)
                pair.append(torch.cat([at, torch.tensor([V], device="cuda")]))
            self.nbr.append(pair)
        self.alpha = 1.0 / (1.0 + 2.0 ** -d)

    def rows(self, x, reverse=False):
        """x splatted and blurred: one row per vertex, and the row of zeros."""
        v = torch.zeros((self.V + 1, x.shape[1]), dtype=torch.float64, device="cuda")
        for j in range(self.d + 1):
            v = v.index_add(0, self.off[:, j], self.bary[:, j:j + 1] * x)
        for j in range(self.d, -1, -1) if reverse else range(self.d + 1):
            a, b = self.nbr[j]
            v = v + 0.5 * (v[a] + v[b])
        return v

    def filter(self, x, reverse=False):
        v, out = self.rows(x, reverse), 0.0
        for j in range(self.d + 1):
            out = out + self.bary[:, j:j + 1] * v[self.off[:, j]]
        return self.alpha * out

    def slice_gradient(self, v, c):
        """The gradient of sum c . slice(v) over the features, with the simplices fixed."""
        d, d1 = self.d, self.d + 1
        s = torch.stack([(c * v[self.off[:, r]]).sum(1) for r in range(d1)], 1)
        r0 = d - self.rank
        ra = (self.alpha / d1) * (s.gather(1, r0) - s.gather(1, (r0 + 1) % d1))
        sm, out = ra[:, 0], []
        for j in range(1, d1):
            sf = math.sqrt(2.0 / 3.0) * d1 / math.sqrt((j + 1.0) * j)
            out.append(sf * (sm - j * ra[:, j]))
            sm = sm + ra[:, j]
        return torch.stack(out, 1)

    def gradient(self, a, c):
        return self.slice_gradient(self.rows(a), c) + self.slice_gradient(self.rows(c, True), a)


class _Term:
    def __init__(self, f, norm):
        self.lat = _Lattice(f)
        k1 = self.lat.filter(torch.ones((self.lat.N, 1), dtype=torch.float64, device="cuda")) + 1e-20
        self.n = k1.rsqrt() if norm == 3 else 1.0 / k1
        self.pre, self.post = norm in (1, 3), norm in (2, 3)

    def message(self, Q):
        m = self.lat.filter(Q * self.n if self.pre else Q)
        return m * self.n if self.post else m


def _apply(c, m):
    if c.ndim == 2:
        return m @ (0.5 * (c + c.t())).t()
    return m * c if c.numel() > 1 else -c * m


def _mean_field(U, terms, compat, kw, iters, keep=None):
    """Q after the iterations; keep takes (Q_t, E_{t+1}) of every iteration."""
    Q = torch.softmax(-U, 1)
    for _ in range(iters):
        E = U
        for t, c, w in zip(terms, compat, kw):
            E = E + _apply(c, w * t.message(Q))
        if keep is not None:
            E.retain_grad()
            keep.append((Q, E))
        Q = torch.softmax(-E, 1)
    return Q


def _features_2d(img, scales=None):
    H, W = img.shape[:2]
    y, x = np.divmod(np.arange(W * H, dtype=np.int64), W)
    x, y = x.astype(np.float32), y.astype(np.float32)
    rgb = img.reshape(-1, 3).T.astype(np.float32)
    fg = np.stack([x / np.float32(SXY_G), y / np.float32(SXY_G)])
    fb = np.concatenate([np.stack([x / np.float32(SXY_B), y / np.float32(SXY_B)]), rgb / np.float32(SRGB)])
    if scales is None:
        return fg, fb
    return (scales[:2, None] * fg).astype(np.float32), (scales[2:, None] * fb).astype(np.float32)


def _double(c):
    return torch.as_tensor(c, dtype=torch.float32).double().reshape(np.shape(c)).cuda()


def _exact_inference(img, U, c, norm, iters):
    with torch.no_grad():
        terms = [_Term(f, norm) for f in _features_2d(_host(img))]
        return _mean_field(U.double(), terms, [_double(a) for a in c], [1.0, 1.0], iters)


def _exact_step(U, gt, terms, c, w, iters, bases=None):
    """[Q, and the gradients of U, the compatibilities, the term weights (and the scales)]."""
    U = U.detach().double().requires_grad_(True)
    c = [_double(a).requires_grad_(True) for a in c]
    kw = torch.tensor(w, dtype=torch.float64, device="cuda", requires_grad=True)
    keep = []
    Q = _mean_field(U, terms, c, kw, iters, keep)
    _loss(Q, gt).backward()
    out = [Q.detach(), U.grad, torch.cat([a.grad.reshape(-1) for a in c]), kw.grad]
    if bases is None:
        return out
    with torch.no_grad():  # the symmetric normalisation's feature gradient, as the framework defines it
        dk = []
        for k, (t, f) in enumerate(zip(terms, bases)):
            n, total = t.n, 0.0
            for Qt, E in keep:
                b, lbl = E.grad, _apply(c[k], kw[k] * Qt)
                x = 0.5 * (b * t.lat.filter(lbl * n) + t.lat.filter(b * n, True) * lbl) * n ** 3
                fg = t.lat.gradient(b * n, lbl * n) - t.lat.gradient(x, torch.ones_like(x))
                total = total + (torch.from_numpy(f).cuda().double().t() * fg).sum(0)
            dk.append(total)
    return out + [torch.cat(dk)]


class _Joined:
    """The terms of several instances as one: messages of their slices side by side."""

    def __init__(self, parts, sizes):
        self.parts, self.sizes = parts, sizes

    def message(self, Q):
        return torch.cat([p.message(q) for p, q in zip(self.parts, Q.split(self.sizes))])


def exact(case, seed):
    kind, L, it = case["kind"], case["L"], case["iters"]
    if kind in ("infer", "dropin"):
        img, U, _ = _image(case["W"], case["H"], L, seed)
        c = _folded(case, seed) if kind == "infer" else [W_G, W_B]
        Q = _exact_inference(img, U, c, NORMS[case.get("norm", "symmetric")], it)
        return Q if kind == "infer" else Q.t().cpu().numpy()
    if kind == "batch":
        out = []
        for i, (w, h) in enumerate(_shapes(case)):
            img, U, _ = _image(w, h, L, seed * 64 + i)
            out.append(_exact_inference(img, U, [W_G, W_B], 3, it))
        return torch.cat(out)
    c, w = _compat(case, seed)
    if kind == "volume":
        vols = [_volume(z, case["side"], L, seed * 64 + i) for i, z in enumerate(_shapes(case))]
        sizes = [v[2].shape[0] for v in vols]
        terms = [_Joined([_Term(v[k], 3) for v in vols], sizes) for k in (0, 1)]
        return _exact_step(torch.cat([v[2] for v in vols]), torch.cat([v[3] for v in vols]), terms, c, w, it)
    img, U, gt = _image(case["W"], case["H"], L, seed)
    if kind == "train":
        return _exact_step(U, gt, [_Term(f, 3) for f in _features_2d(_host(img))], c, w, it)
    out = []
    for scales in _scales(seed):
        terms = [_Term(f, 3) for f in _features_2d(_host(img), scales)]
        out += _exact_step(U, gt, terms, c, w, it, _features_2d(_host(img)))
    return out
