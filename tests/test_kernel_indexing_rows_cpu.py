"""Host emulation of the index arithmetic of padded rows, the quad splat, the staged slice
pairs and the device-built lists (no GPU).

Restated for every thread, and checked to stay inside every buffer and to touch each item
exactly once, at the edges of the shapes (one lane per row, a lane group as wide as a wave,
padding labels, a last wave with one pixel, waves without any):

* dcrf_device.h: LaneGroup's division by a reciprocal, load_row / store_row's shifted last
  piece, row_piece's 24- and 32-bit offsets; filter.hip: padded_labels;
* dcrf_fused.h, meanfield.hip, adjoint_fused.hip: WavePixels, wave_pairs and
  stage_wave_pairs (rounds of 128 pairs, the last pair repeated), message rows and the
  statistic's slots of padded rows;
* filter.hip: k_splat's entry windows, k_splat_split's quads;
* segments.hip: group_first, the run and head counts, k_emit's three ranges,
  k_ones_segments and k_ones_vertices, against lists built one segment after another;
* kgrad.hip: k_kg_relayout (x layout to paired layout), stage_words;
* lattice.hip: the chains of k_hash_insert;
* capi.hip: the shares of a downloaded window.
"""
import numpy as np
import pytest

WAVE_BLOCK, XCDS, K_WIN, K_BATCH, K_SPLIT, K_SPLIT_BATCH, SPLIT = 256, 8, 512, 8, 4, 8, 16
LABELS = [1, 2, 3, 4, 5, 7, 8, 10, 11, 13, 14, 19, 21, 22, 26, 64, 65, 85, 130, 131, 251, 256]


def labels_per_lane(L):
    return next((R for R in (4, 3, 2) if L % R == 0), 1)


def padded_labels(L):
    R = labels_per_lane(L)
    return (L + 3) & ~3 if (R == 1 and L >= 5) or (R == 2 and L >= 14) else L


def shape(Lv):
    R = labels_per_lane(Lv)
    return R, Lv // R


def xcd_block(b, nb):
    x, i = b % XCDS, b // XCDS
    q, r = nb // XCDS, nb % XCDS
    return x * q + np.minimum(x, r) + i


def test_padded_shapes():
    for L in range(1, 1025):
        Lv = padded_labels(L)
        R, S = shape(Lv)
        assert L <= Lv <= L + 3 and S * R == Lv and (S - 1) * R < L  # no lane of padding only
        assert Lv == L or R == 4  # load_row and store_row handle a partial piece of four
        if Lv > L:
            assert Lv == (L + 3) & ~3  # the message rows' stride holds the padding labels
        assert Lv <= 8 * L // 5  # what the allocation-free inference's array allows for


def test_lane_division_by_reciprocal():
    lane = np.arange(1024, dtype=np.float32)
    for S in range(1, 1025):
        rc = np.float32(1.0) / np.float32(S)
        for c in (np.nextafter(rc, np.float32(0)), rc, np.nextafter(rc, np.float32(2))):  # one ulp off
            g = ((lane + np.float32(0.5)) * c).astype(np.int32)
            assert np.array_equal(g, np.arange(1024) // S), S


@pytest.mark.parametrize("L", [L for L in LABELS if padded_labels(L) > L])
def test_rows_with_a_partial_last_piece(L):
    Lv = padded_labels(L)
    R, S = shape(Lv)
    row = np.arange(1, L + 1)
    for lane in range(S):
        k0 = lane * R
        sh = max(k0 + R - L, 0)
        at = k0 - sh + np.arange(R)
        assert at.min() >= 0 and at.max() < L  # the access stays in the row
        x = row[at].copy()
        b = 1
        while b < R:
            if sh & b:
                x[:R - b] = x[b:]
            b <<= 1
        x = np.where(k0 + np.arange(R) < L, x, 0)
        want = np.where(k0 + np.arange(R) < L, k0 + np.arange(R) + 1, 0)
        assert np.array_equal(x, want)
        # store_row: the whole piece, or its labels but never its last slot
        stored = [k0 + r for r in range(R)] if k0 + R <= L else [k0 + r for r in range(R - 1) if k0 + r < L]
        assert stored == [k for k in range(k0, k0 + R) if k < L]


@pytest.mark.parametrize("ld", [1, 2, 3, 4, 8, 20, 21, 64, 1000, (1 << 22) - 1])
def test_narrow_row_offsets(ld):
    """narrow_rows: below its limits the 24-bit multiply and the 32-bit sum are exact."""
    rows = min(1 << 24, 0xffffffff // (4 * ld))
    for row in {0, 1, rows // 2, rows - 1}:
        for k0 in {0, ld - 1}:
            assert row < 1 << 24 and ld * 4 < 1 << 24
            off = ((row & 0xffffff) * ((ld * 4) & 0xffffff)) & 0xffffffff
            assert (off + 4 * k0) & 0xffffffff == 4 * (row * ld + k0)


def fused_launch(N, L, DS, NT, matrix_terms, nstat):
    Lv = padded_labels(L)
    R, S = shape(Lv)
    assert S <= 64
    per, waves = 64 // S, WAVE_BLOCK // 64
    grid = -(-N // (waves * per))
    t = np.arange(WAVE_BLOCK)
    lane, w = t & 63, t >> 6
    g = lane // S
    l = lane - g * S
    on = g < per
    g, l = np.where(on, g, 0), np.where(on, l, np.where(l < S, l, 0))
    k0 = l * R
    p = (xcd_block(np.arange(grid), grid)[:, None] * waves + w) * per + g
    active = on & (p < N)
    first = active & (k0 == 0)
    assert np.array_equal(np.sort(p[first]), np.arange(N))  # each pixel once
    # WavePixels: the same in every lane of a wave; at least one pixel, inside the model
    p0 = np.minimum(p - g, N - 1)
    assert np.all(p0.reshape(grid, waves, 64) == p0.reshape(grid, waves, 64)[:, :, :1])
    np_ = np.minimum(per, N - p0)
    assert np_.min() >= 1
    gp = np.minimum(g, np_ - 1)
    assert np.all(p0[active] + np.broadcast_to(gp, p.shape)[active] == p[active])
    pix = p0 + gp
    assert pix.min() >= 0 and pix.max() < N
    # rows: the caller's (load_row: clamped to the row), the padded ones whole
    assert k0.max() + R <= Lv and np.all(np.where(k0 + R > L, k0 - (k0 + R - L), k0) >= 0)
    assert (pix * Lv + k0 + R - 1).max() < N * Lv
    # slice pairs: rounds of 128, repeated past the run
    wpairs = (per * DS + 127) & ~127
    staged = np.zeros((grid, waves, wpairs), np.int64)
    n = (np_.reshape(grid, waves, 64)[:, :, 0] * DS)[..., None]
    base = (p0.reshape(grid, waves, 64)[:, :, 0] * DS)[..., None]
    for i0 in range(0, per * DS, 128):
        for off in (0, 64):
            slot = i0 + off + np.arange(64)
            src = base + np.minimum(slot, n - 1)
            assert src.min() >= 0 and src.max() < N * DS and slot.max() < wpairs
            staged[:, :, slot] = src
    for j in range(DS):  # a group reads its own pixel's pairs, staged
        at = gp * DS + j
        assert at.max() < wpairs
        got = staged[np.arange(grid)[:, None], w[None, :], at]
        assert np.array_equal(got, pix * DS + j)
    # LDS: pairs, Matrix weights, message rows, statistic
    ldm = (L + 3) & ~3
    cwf = matrix_terms * L * ldm
    stat = nstat * WAVE_BLOCK * R + nstat * waves * L
    lds = waves * wpairs * 2 + cwf + (waves * NT * per * ldm if cwf else 0) + stat
    assert lds * 4 <= 160 * 1024
    if cwf:
        msg0 = waves * wpairs * 2 + cwf
        last = msg0 + (w[on] * NT * per + (NT - 1) * per + g[on]) * ldm + k0[on] + R - 1
        assert last.max() < lds - stat and k0.max() + R <= ldm
    if nstat:  # stat_finish reads the lane and register that hold label lab
        lab = np.arange(L)
        assert (lab // R).max() < S and np.all(lab // R * R + lab % R == lab)


@pytest.mark.parametrize("L", [L for L in LABELS if shape(padded_labels(L))[1] <= 64])
@pytest.mark.parametrize("N", [1, 2, 63, 997, 24 * 20, 320 * 213])
@pytest.mark.parametrize("DS,NT", [(9, 2), (3, 1), (6, 1)])
def test_fused_kernels(N, L, DS, NT):
    fused_launch(N, L, DS, NT, 0, NT)
    if L <= 26:
        fused_launch(N, L, DS, NT, NT, 0)


def random_segments(rng, n, longest):
    """n adjoining segments (beg, end), empty ones among them."""
    length = rng.integers(0, longest + 1, n)
    end = np.cumsum(length)
    return end - length, end


@pytest.mark.parametrize("L", [9, 12, 19, 21, 64, 256])
@pytest.mark.parametrize("longest", [1, 32, 700])
def test_splat_windows(L, longest):
    """k_splat: the windows of a wave's entries, staged in rounds of 256."""
    _, S = shape(padded_labels(L))
    per = 64 // S
    beg, end = random_segments(np.random.default_rng(L + longest), 4 * per + 1, longest)
    E, n = int(end[-1]), len(beg)
    used = np.zeros(E, np.int64)
    for cw0 in range(0, n, per):
        r0, r1 = int(beg[cw0]), int(end[min(cw0 + per - 1, n - 1)])
        taken = {c: [] for c in range(cw0, min(cw0 + per, n))}
        for w0 in range(r0, r1, K_WIN):
            wn = min(K_WIN, r1 - w0)
            win = np.full(K_WIN + K_BATCH, -2, np.int64)
            for u0 in range(0, wn, 256):
                for u in range(4):
                    slot = u0 + np.arange(64) + 64 * u
                    src = w0 + np.minimum(slot, wn - 1)
                    assert src.max() < E and slot.max() < K_WIN
                    win[slot] = src
            win[wn:wn + K_BATCH] = -1  # pixel 0, weight 0
            for c in taken:
                a, b = max(int(beg[c]), w0) - w0, min(int(end[c]), w0 + wn) - w0
                for i in range(a, b, K_BATCH):
                    for u in range(K_BATCH):
                        assert i + u < wn + K_BATCH and win[i + u] >= -1  # initialised
                        if i + u < b:
                            taken[c].append(int(win[i + u]))
        for c, got in taken.items():
            assert got == list(range(int(beg[c]), int(end[c])))  # every entry, in order
            used[got] += 1
    assert np.all(used == 1)


@pytest.mark.parametrize("L", [1, 2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("longest", [1, 32, 100])
def test_splat_quads(L, longest):
    """k_splat_split: groups of S quads; a quad's lanes take every fourth entry and add all
    of them in order."""
    R, S = shape(padded_labels(L))
    assert S <= 2
    gs = S * K_SPLIT
    per = 64 // gs
    lane = np.arange(64)
    g = lane >> 2 if S == 1 else lane >> 3
    k0 = np.zeros(64, int) if S == 1 else ((lane >> 2) & 1) * R
    assert np.array_equal(g, lane // gs) and g.max() == per - 1
    assert np.array_equal(k0, (lane % gs) // K_SPLIT * R) and k0.max() + R <= padded_labels(L)
    # the next group's lane of the same position, wherever a run may continue
    nxt = (lane + gs) & 63
    inner = g + 1 < per
    assert np.all(g[nxt[inner]] == g[inner] + 1) and np.all(k0[nxt[inner]] == k0[inner])
    beg, end = random_segments(np.random.default_rng(L + longest), 3 * per + 1, longest)
    for b, e in zip(beg, end):
        order = []
        for i0 in range(int(b), int(e), K_SPLIT_BATCH * K_SPLIT):
            for u in range(K_SPLIT_BATCH):
                for kk in range(K_SPLIT):
                    i = i0 + kk + u * K_SPLIT
                    assert b <= min(i, e - 1) < e  # the clamped load
                    if i < e:
                        order.append(i)
        assert order == list(range(int(b), int(e)))


# ------------------------------------------------------------------------ segment lists
def random_terms(rng, T, NT, V, most=90):
    """Per term: runs [(tile, vertex, entries)] sorted by (tile, vertex), every tile with
    runs, some vertices without."""
    terms = []
    for k in range(T):
        runs = []
        for t in range(NT):
            for v in sorted(rng.choice(V[k], rng.integers(1, V[k]), replace=False)):
                runs.append((t, int(v), int(rng.choice([1, 2, 31, 32, 33, rng.integers(1, most)]))))
        terms.append(runs)
    return terms


def device_lists(terms, NT, V, C, per, perc, sequential, row0):
    """segments.hip, array by array."""
    T = len(terms)
    vbase = np.concatenate([[0], np.cumsum(V)])
    tile_run = [np.array([sum(r[0] < t for r in runs) for t in range(NT + 1)]) for runs in terms]
    beg = [np.concatenate([[0], np.cumsum([r[2] for r in runs])]) for runs in terms]
    tile_ptr = [beg[k][tile_run[k]] for k in range(T)]
    R = sum(len(r) for r in terms)
    E = sum(int(b[-1]) for b in beg)
    Vt, G = int(vbase[-1]), NT * T

    def group_first(tab, t, i):
        return sum(int(tab[k][t + 1 if k < i else t]) for k in range(T))

    mbase, gebase = np.full(G + 1, -1), np.full(G + 1, -1)
    rv, rb, rl, rg = (np.full(R, -1) for _ in range(4))
    for i in range(T):
        for r in range(max(len(terms[i]), NT + 1)):
            if r < NT or (r == NT and i == 0):
                mbase[r * T + i] = group_first(tile_run, r, i)
                gebase[r * T + i] = group_first(tile_ptr, r, i)
            if r >= len(terms[i]):
                continue
            t, v, n = terms[i][r]
            q = group_first(tile_run, t, i) + r - tile_run[i][t]
            assert rv[q] < 0  # written once
            rv[q], rl[q], rg[q] = vbase[i] + v, n, t * T + i
            rb[q] = group_first(tile_ptr, t, i) + beg[i][r] - tile_ptr[i][t]
    assert np.all(rv >= 0) and np.all(np.diff(mbase) >= 0) and mbase[G] == R and gebase[G] == E
    assert np.array_equal(rb, np.cumsum(rl) - rl)  # the merged runs adjoin
    S = np.concatenate([[0], np.cumsum((rl - 1) // C + 1)])
    si = np.argsort(rv, kind="stable")
    sv = rv[si]
    vrun = np.full(Vt + 1, -1)
    for i in range(R + 1):
        for v in range(sv[i - 1] + 1 if i else 0, (sv[i] if i < R else Vt) + 1):
            assert vrun[v] < 0
            vrun[v] = i
    assert np.array_equal(vrun, np.searchsorted(sv, np.arange(Vt + 1)))
    o = S[si] - S[mbase[rg[si]]]
    k = S[si + 1] - S[si]
    h = (o + k - 1) // per - o // per + 1 if per else k
    H = np.concatenate([[0], np.cumsum(h)])
    K = np.concatenate([[0], np.cumsum(k)])
    ng = S[mbase[1:]] - S[mbase[:-1]]
    gseg = np.concatenate([[0], np.cumsum(-(-ng // per) * per if per else ng)])
    n = H[vrun[1:]] - H[vrun[:-1]]
    split = 1 << 30 if sequential else SPLIT
    cnt = dict(partial=np.where(n > 1, n, 0), light=(n > 1) & (n <= split), heavy=n > split, empty=n == 0,
               pieces=np.where(n > split, -(-n // SPLIT), 0))
    vs = {a: np.concatenate([[0], np.cumsum(x)]) for a, x in cnt.items()}
    tot = {a: int(x[-1]) for a, x in vs.items()}
    tail = int(gseg[-1]) + tot["empty"]
    nch = -(-tail // per) * per if per else tail
    light_pad = -(-tot["light"] // perc) * perc if perc and tot["heavy"] else tot["light"]
    ncb = light_pad + tot["heavy"] * perc if perc else tot["light"] + tot["pieces"]
    ncb2 = 0 if perc else tot["heavy"]
    row2 = row0 + tot["partial"]
    ch, cb, cb2 = [None] * nch, [None] * ncb, [None] * ncb2

    def put(a, i, x):
        assert 0 <= i < len(a) and a[i] is None  # inside, once
        a[i] = x

    for i in range(R):
        m = si[i]
        oo, kk, first = int(o[i]), int(k[i]), H[vrun[sv[i]]]
        direct = H[vrun[sv[i] + 1]] - first == 1
        row = row0 + vs["partial"][sv[i]] + H[i] - first
        for j in range(kk):
            head = not per or j == 0 or (oo + j) % per == 0
            before = (oo + j) // per - oo // per if per else j
            b = rb[m] + j * C
            put(ch, gseg[rg[m]] + oo + j,
                (sv[i], b, b + min(C, rl[m] - j * C), (sv[i] if direct else row + before) if head else -1))
    for v in range(Vt):
        first = row0 + vs["partial"][v]
        if n[v] == 0:
            put(ch, gseg[-1] + vs["empty"][v], (v, E, E, v))
        elif 1 < n[v] <= split:
            put(cb, vs["light"][v], (v, first, n[v], 0))
        elif n[v] > split:
            pieces = min(perc, -(-n[v] // SPLIT)) if perc else -(-n[v] // SPLIT)
            off = 0
            for j in range(perc or pieces):
                q = (n[v] - off) // (pieces - j) if j < pieces else 0
                if perc:
                    put(cb, light_pad + vs["heavy"][v] * perc + j, (v, first + off, q, pieces))
                else:
                    put(cb, light_pad + vs["pieces"][v] + j, (row2 + vs["pieces"][v] + j, first + off, q, 0))
                off += q
            if not perc:
                put(cb2, vs["heavy"][v], (v, row2 + vs["pieces"][v], pieces, 0))
    for g in range(G):
        for i in range(gseg[g] + ng[g], gseg[g + 1]):
            put(ch, i, (-1, gebase[g + 1], gebase[g + 1], -1))
    for i in range(tail, nch):
        put(ch, i, (-1, E, E, -1))
    for i in range(tot["light"], light_pad):
        put(cb, i, (0, 0, 0, 0))
    assert None not in ch and None not in cb and None not in cb2
    return dict(ch=ch, cb=cb, cb2=cb2, row2=row2, E=E, rv=rv, rb=rb, rl=rl, rg=rg, si=si, S=S, K=K, vrun=vrun,
                gebase=gebase, tile_ptr=tile_ptr, R=R, V=Vt, beg=beg)


CASES = [(1, 1, [3]), (1, 5, [40]), (2, 3, [7, 30]), (3, 2, [1 + 1, 50, 4])]


@pytest.mark.parametrize("T,NT,V", CASES)
@pytest.mark.parametrize("C", [1, 32, 1 << 20])
@pytest.mark.parametrize("per,perc,sequential", [(16, 64, False), (9, 9, False), (1, 1, False), (0, 0, False), (0, 0, True),
                                                 (0, 9, False)])
def test_segment_lists(T, NT, V, C, per, perc, sequential):
    rng = np.random.default_rng(T * 100 + NT)
    terms = random_terms(rng, T, NT, V)
    row0 = sum(V) + 1
    D = device_lists(terms, NT, V, C, per, perc, sequential, row0)
    ch = D["ch"]
    # segments adjoin (the splat loads a wave's entries as one range) and cover the entries
    assert ch[0][1] == 0 and ch[-1][2] == D["E"] and all(a[2] == b[1] for a, b in zip(ch, ch[1:]))
    assert all(b - a <= C for _, a, b, _ in ch)
    # a continuation follows a segment of its vertex in its wave; fillers have no vertex
    for c, (v, _, _, out) in enumerate(ch):
        if out < 0 and v >= 0:
            assert per and c % per and ch[c - 1][0] == v
        assert v >= 0 or out == -1
    # every (tile, term) group starts a wave, so no wave holds two
    group = np.repeat(D["rg"], D["rl"])
    if per:
        for w in range(0, len(ch), per):
            a, b = ch[w][1], ch[w + per - 1][2]
            assert len(set(group[a:b].tolist())) <= 1
    # outputs: partial rows contiguous per vertex, in list order, each written once
    rows = {}
    for v, _, _, out in ch:
        if out >= 0:
            rows.setdefault(v, []).append(out)
    assert sorted(rows) == list(range(D["V"]))
    partial = []
    for v, r in rows.items():
        if len(r) == 1:
            assert r[0] == v
        else:
            assert r == list(range(r[0], r[0] + len(r)))
            partial += r
    assert sorted(partial) == list(range(row0, D["row2"]))
    # recombination: every partial row read once, whole waves for the heavy vertices
    read, second = [], []
    for i, (v, f, n, pad) in enumerate(D["cb"]):
        read += range(f, f + n)
        if n and v >= D["row2"]:
            second.append(v)
        if perc and pad:
            wave = D["cb"][i // perc * perc:(i // perc + 1) * perc]
            assert len(wave) == perc and {x[0] for x in wave} == {v} and {x[3] for x in wave} == {pad}
        if sequential and n:
            assert [f + j for j in range(n)] == rows[v]
    assert sorted(read) == list(range(row0, D["row2"]))
    assert sorted(x for _, f, n, _ in D["cb2"] for x in range(f, f + n)) == sorted(second)
    # k_ones_segments and k_ones_vertices: each entry once, a vertex's segments in list order
    seg_of = [[] for _ in range(D["V"])]
    used = [np.zeros(int(b[-1]), np.int64) for b in D["beg"]]
    assert D["K"][-1] <= D["R"] + D["E"] // C  # the partial sums' buffer
    for q in range(int(D["K"][-1])):
        lo = int(np.searchsorted(D["K"][:-1], q, side="right")) - 1
        m = D["si"][lo]
        at = (q - D["K"][lo]) * C
        g = D["rg"][m]
        i = g % T
        b = D["rb"][m] + at - D["gebase"][g] + D["tile_ptr"][i][g // T]
        n = min(C, D["rl"][m] - at)
        assert n > 0
        used[i][b:b + n] += 1
        v = int(D["rv"][m])
        assert D["K"][D["vrun"][v]] <= q < D["K"][D["vrun"][v + 1]]
        seg_of[v].append((int(D["rb"][m] + at), n))
    assert all(np.all(u == 1) for u in used)
    listed = [[(a, b - a) for v2, a, b, _ in ch if v2 == v and b > a] for v in range(D["V"])]
    assert seg_of == listed


@pytest.mark.parametrize("V,partials", [([36254, 101712], 5900), ([5], 0), ([7, 3, 11, 2], 7)])
def test_kg_relayout_to_the_paired_rows(V, partials):
    """kg_map_row: the x layout (the terms' vertices one after another, the zero row, the
    partial rows) to the paired one (forward and reverse rows per term)."""
    X = np.concatenate([[0], np.cumsum(V)])
    F, Z1, Z2 = 2 * X, int(X[-1]), 2 * int(X[-1])

    def map_row(r):
        if r < 0:
            return r
        if r > Z1:
            return Z2 + (r - Z1)
        i = max(k for k in range(len(V)) if k == 0 or r >= X[k])
        return int(F[i] + (r - X[i]))

    for i, v in enumerate(V):
        for j in (0, v // 2, v - 1):
            assert map_row(int(X[i]) + j) == F[i] + j < F[i] + v
    assert [map_row(Z1 + 1 + q) for q in range(partials)] == list(range(Z2 + 1, Z2 + 1 + partials))
    assert map_row(-1) == -1  # fillers and continuations


@pytest.mark.parametrize("D1", range(2, 8))
def test_hash_chains(D1):
    """k_hash_insert: lead is the first of a chain of equal keys D1 lanes apart."""
    rng = np.random.default_rng(D1)
    for _ in range(200):
        same = (rng.random(64) < rng.choice([0.1, 0.9, 1.0])) & (np.arange(64) >= D1)
        lead = np.where(same, np.arange(64) - D1, np.arange(64))
        n = 1
        while n <= 63 // D1:
            lead = lead[lead]
            n *= 2
        for lane in range(64):
            a = lane
            while same[a]:
                a -= D1
            assert lead[lane] == a >= 0


@pytest.mark.parametrize("per,n,D1", [(9, 1, 3), (9, 9, 6), (64, 64, 7), (64, 5, 7), (1, 1, 2)])
def test_staged_words(per, n, D1):
    """stage_words: the words of n of a wave's `per` points, the last one repeated."""
    dst = np.full(64 * D1, -1)
    for lane in range(64):
        for i in range(lane, per * D1, 64):
            assert dst[i] < 0
            dst[i] = min(i, n * D1 - 1)
    assert np.array_equal(dst[:n * D1], np.arange(n * D1)) and dst[:per * D1].min() >= 0


@pytest.mark.parametrize("n", [2 << 20, 5732160, 66060288, (8 << 20) + 3, 123456789])
def test_download_shares(n):
    """copy_to_host_window: the chunks tile the window, each thread's shares tile a chunk."""
    def off(n, T, t):
        return n if t >= T else (n // T * t) & ~4095

    C = max(n >> 23, min(n >> 21, 4), 1)
    at = 0
    for c in range(C):
        a, b = off(n, C, c), off(n, C, c + 1)
        assert a == at < b
        at = b
        for T in range(1, 9):
            x = [a + off(b - a, T, t) for t in range(T + 1)]
            assert x[0] == a and x[-1] == b and all(i <= j for i, j in zip(x, x[1:]))
    assert at == n
