// Lattice filtering and the fused mean-field update for gfx950.
//
// Replaces Permutohedral::compute (pydensecrf/densecrf/src/permutohedral.cpp:476-610),
// DenseKernel::filter (pairwise.cpp:63-80), LabelCompatibility::apply
// (labelcompatibility.cpp:46-87) and expAndNormalize (densecrf.cpp:98-106).
//
// Thread mapping: a lane group of S = L / R consecutive threads handles one item (a
// splat chunk, a lattice vertex or a pixel), lane l owning the R labels [l*R, l*R+R),
// so every vertex/pixel row of L floats is read and written as S contiguous R-float
// pieces (dcrf_device.h).  All reductions run in a fixed order: results are
// deterministic from run to run.
//   splat    each chunk (<= C contributors of one vertex, pixel ascending) is summed
//            sequentially; vertices with several chunks write partial rows that the
//            combine kernel adds in chunk order.  No atomics.
//   blur     one launch per step; step s covers the terms whose lattice has axis s
//            (a prefix of the vertex space, which is ordered by decreasing d):
//            new = old + 0.5 * (n1 + n2), the reference's update (:556-569).
//   meanfield per pixel: slice every term (sum_j w_j*alpha*norm_p * row_j), apply the
//            compatibility, subtract from -U, softmax over the lane group.
#include "dcrf_internal.h"
#include "dcrf_device.h"

#include <cmath>
#include <type_traits>

#pragma clang fp contract(off)

namespace dcrf {

// Labels per lane: the largest R in {4, 3, 2} that divides L, else 1 (so every lane's
// piece of a row is whole: no partial lanes, no conditional accesses).
int choose_labels_per_lane(int L) {
    for (int R = 4; R >= 2; R--)
        if (L % R == 0) return R;
    return 1;
}

// Rows of L floats that neither 4 nor 3 divides take one or two labels per lane: at 19
// labels 19 lanes and 3 rows per wave instruction, each with its own addresses and
// weights.  Padded to 20, five lanes of four labels and 12 rows.  10 iterations, unpadded ->
// padded, us (training forward and backward: the same ratios):
//   one label per lane    5       7       11      13      17      25      61      257
//     320x213          310/297 316/290 359/340 349/322 383/355 458/381 707/447 12357/2311
//     1024x768        1005/761 1152/767 1559/1000 1793/998 2096/1242 2962/1702 6201/3354
//   two labels per lane   10      14      22      26      34      130
//     320x213          317/344 330/323 395/367 412/374 458/402 1684/1032
//     1024x768         969/994 1173/1004 1873/1395 2259/1727 3024/2193
// 10 labels lose at every size (a fifth more bytes in every row; 64x48: 209 -> 240), the
// next, 14, gain from 320x213 on: the line for two labels per lane is there.  At 64x48,
// where launches count, the padded form is up to 12 % slower (11 labels), the same from 65
// labels on.  Three labels per lane stay: 21 labels padded to 24 (6 lanes for 7, aligned
// 16-byte pieces, but 14 % more bytes) measured 1514 against 1464 us at 1024x768.
int padded_labels(int L) {
    const int R = choose_labels_per_lane(L);
    return (R == 1 && L >= 5) || (R == 2 && L >= 14) ? (L + 3) & ~3 : L;
}

// Rows of one or two lanes (up to 8 labels) take the quad form of the splat
// (k_splat_split).  10 iterations, k_splat -> quads: 1920x1080x2 1421 -> 1127 us,
// 200x150x3 390 -> 230 us, training on 1.5 M voxels with 4 labels 2892 -> 2366 us; eight
// lanes per segment: the same within 2 %.  From three lanes on (9 labels: 21 segments a
// wave) one window holds nearly all of a wave's entries.
SplatShape splat_shape(int L) {
    const LaunchShape sh = shape_for(L);
    if (!sh.wave || sh.S > 2) return SplatShape{1, sh.per};
    return SplatShape{kSplitLanes, 64 / (sh.S * kSplitLanes)};
}

LaunchShape shape_for(int L) { return shape_for_r(L, choose_labels_per_lane(L)); }

LaunchShape shape_for_r(int L, int R) {
    const int S = (L + R - 1) / R;
    if (S <= 64) return LaunchShape{kWaveBlock, 64 / S, true, (kWaveBlock / 64) * (64 / S), R, S};
    const int block = S <= 256 ? 256 : (S <= 512 ? 512 : 1024);
    return LaunchShape{block, block / S, false, block / S, R, S};
}

namespace {

constexpr int kThreads = 256;
constexpr int kBatch = 8;  // contributors / partial rows loaded together
inline unsigned blocks_for(size_t n, int t = kThreads) { return (unsigned)((n + t - 1) / t); }

__global__ void k_fill(float* p, float v, size_t n) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// Splat: each group sums one chunk (<= C contributors of a vertex, in entry order)
// sequentially.  Entries are (pixel, weight bits) pairs.  A chunk with out < 0 continues
// the chunk before it in the same wave (same vertex): WAVE mode adds it to that chunk's
// sum instead of storing it.
//   WAVE mode: the chunks of a wave are consecutive and their entry ranges adjoin (the
//   layout guarantees chunk c+1 begins where chunk c ends), so the wave loads its whole
//   entry range cooperatively (64 consecutive pairs per load instruction) into an LDS
//   window of kWin pairs, and each group reads its pairs from there: one cache line
//   serves 16 pairs instead of one load per lane and pair.  Input rows are gathered
//   kBatch at a time.
//   block mode (a group wider than a wave): the pairs are loaded by every lane.
// The compiler must not sink a batch's loads into the masked additions that use them: it
// had moved the first entry's LDS read and row load behind all the others of its batch,
// two memory round trips per batch instead of one (loaded() keeps a value's load where
// it is written).
constexpr int kWin = 512;  // entry pairs per wave window

template <int R>
__device__ __forceinline__ void loaded(float (&x)[R]) {
#pragma unroll
    for (int r = 0; r < R; r++) asm volatile("" : "+v"(x[r]));
}

template <bool WAVE, int R, bool NARROW>
__global__ void __launch_bounds__(1024) k_splat(const Chunk* __restrict__ chunks, int n,
                                                const int2* __restrict__ ent, const float* __restrict__ in, int ldi,
                                                float* __restrict__ vals, int ldv, int L, int S, int per) {
    LaneGroup<WAVE, R> G(L, S, per, nullptr);
    const int c = G.item();
    const int k0 = G.k0;
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; r++) acc[r] = 0.0f;
    if (WAVE) {
        extern __shared__ int2 win_all[];
        int2* win = win_all + G.w * (kWin + kBatch);
        const int lane = threadIdx.x & 63;
        // the wave's first chunk: the same in every lane (scalar bounds and loop)
        const int cw0 = __builtin_amdgcn_readfirstlane(c - G.g);
        if (cw0 >= n) return;  // the whole wave is idle (no block barrier below)
        const bool mine = G.on && c < n;
        const Chunk ch = chunks[mine ? c : cw0];
        const int r0 = chunks[cw0].beg, r1 = chunks[min(cw0 + per - 1, n - 1)].end;
        for (int w0 = r0; w0 < r1; w0 += kWin) {
            const int wn = min(kWin, r1 - w0);
            const int2* __restrict__ src = ent + w0;
            __builtin_amdgcn_wave_barrier();  // the previous window's reads come first
            // four loads per lane and round (clamped, unconditional), then their stores:
            // past wn they repeat the last pair, inside the window
            for (int u0 = 0; u0 < wn; u0 += 256) {
                long long t[4];
#pragma unroll
                for (int u = 0; u < 4; u++)
                    t[u] = reinterpret_cast<const long long*>(src)[(unsigned)min(u0 + lane + 64 * u, wn - 1)];
#pragma unroll
                for (int u = 0; u < 4; u++) reinterpret_cast<long long*>(win)[u0 + lane + 64 * u] = t[u];
            }
            if (lane < kBatch) win[wn + lane] = make_int2(0, 0);  // padding: pixel 0, weight 0
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            if (mine) {
                const int a = max(ch.beg, w0) - w0, b = min(ch.end, w0 + wn) - w0;
                for (int i = a; i < b; i += kBatch) {
                    int2 e[kBatch];
                    float xx[kBatch][R];
#pragma unroll
                    for (int u = 0; u < kBatch; u++) e[u] = win[i + u];  // i + u < wn + kBatch
#pragma unroll
                    for (int u = 0; u < kBatch; u++) load_piece<R>(row_piece<NARROW>(in, e[u].x, ldi, k0), 0, L, xx[u]);
#pragma unroll
                    for (int u = 0; u < kBatch; u++) {
                        loaded<R>(xx[u]);
                        if (i + u < b) {
                            const float wu = __int_as_float(e[u].y);
#pragma unroll
                            for (int r = 0; r < R; r++) acc[r] = add_product(acc[r], wu, xx[u][r]);
                        }
                    }
                }
            }
        }
        // A run of the wave's chunks with one vertex (the layout gives the later ones
        // out = -1): their sums are folded into the run's first group, right to left, in
        // a fixed order.  Lists without such runs skip this.
        const int nv = wave_read(ch.v, lane + S);
        const int nout = wave_read(ch.out, lane + S);
        const bool cont = mine && G.g + 1 < per && c + 1 < n && nout < 0 && nv == ch.v;
        if (__any(cont)) {
            for (int j = per - 2; j >= 0; j--) {  // wave-uniform
                float y[R];
#pragma unroll
                for (int r = 0; r < R; r++) y[r] = wave_read(acc[r], lane + S);
                if (cont && G.g == j)
#pragma unroll
                    for (int r = 0; r < R; r++) acc[r] = acc[r] + y[r];
            }
        }
        if (mine && ch.out >= 0) store_piece<R>(vals + (size_t)ch.out * ldv, k0, L, acc);
        return;
    }
    if (!G.on || c >= n) return;
    const Chunk ch = chunks[c];
    for (int i = ch.beg; i < ch.end; i += kBatch) {
        int2 e[kBatch];
        float xx[kBatch][R];
#pragma unroll
        for (int u = 0; u < kBatch; u++) e[u] = ent[min(i + u, ch.end - 1)];
#pragma unroll
        for (int u = 0; u < kBatch; u++) load_piece<R>(row_piece<NARROW>(in, e[u].x, ldi, k0), 0, L, xx[u]);
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
            loaded<R>(xx[u]);
            if (i + u < ch.end) {
                const float wu = __int_as_float(e[u].y);
#pragma unroll
                for (int r = 0; r < R; r++) acc[r] = add_product(acc[r], wu, xx[u][r]);
            }
        }
    }
    store_piece<R>(vals + (size_t)ch.out * ldv, k0, L, acc);
}

// Splat for rows of few lanes (S <= 2 lanes of R labels, up to 8 labels).  With one lane
// per row piece and segment (k_splat) the wave's lanes are on up to 64 different segments:
// each LDS window of entries covers a third of them while the others wait, and every
// lane's row is a cache line of its own.  Here the K = kSplitLanes = 4 lanes of a quad
// share a segment: lane kk loads every K-th entry, straight from memory (32 consecutive
// bytes per segment and load; kSplitBatch entries per lane, so a segment of 32 in one
// round), and its row.  Neighbouring entries of a segment are mostly neighbouring pixels:
// their rows share lines.  Every lane of the quad then adds all the products in entry
// order, reading them from the other lanes as DPP operands: the rounding of a sequential
// sum, which a tree of the four shares would lose.  Same segments and in-wave runs as
// k_splat, in groups of S quads.
constexpr int kSplitBatch = 8;

template <int R, bool NARROW>
__global__ void __launch_bounds__(kWaveBlock) k_splat_split(const Chunk* __restrict__ chunks, int n,
                                                            const int2* __restrict__ ent, const float* __restrict__ in,
                                                            int ldi, float* __restrict__ vals, int ldv, int S,
                                                            int per) {
    constexpr int K = kSplitLanes;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int gs = S * K;                  // lanes of a group: 4 or 8
    const int g = S == 1 ? lane >> 2 : lane >> 3;
    const int kk = lane & 3, k0 = S == 1 ? 0 : ((lane >> 2) & 1) * R;
    const int cw0 = (xcd_block(blockIdx.x, gridDim.x) * (kWaveBlock / 64) + w) * per;
    if (cw0 >= n) return;  // the whole wave is idle (no block barrier below)
    const int c = cw0 + g;
    const bool mine = c < n;
    const Chunk ch = chunks[mine ? c : cw0];
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; r++) acc[r] = 0.0f;
    for (int i0 = ch.beg; i0 < ch.end; i0 += kSplitBatch * K) {  // the same in all lanes of a group
        int2 e[kSplitBatch];
        float x[kSplitBatch][R];
#pragma unroll
        for (int u = 0; u < kSplitBatch; u++) e[u] = ent[min(i0 + kk + u * K, ch.end - 1)];
#pragma unroll
        for (int u = 0; u < kSplitBatch; u++) load_piece<R>(row_piece<NARROW>(in, e[u].x, ldi, k0), 0, 0, x[u]);
#pragma unroll
        for (int u = 0; u < kSplitBatch; u++) {
            loaded<R>(x[u]);
            const bool on = i0 + kk + u * K < ch.end;
#pragma unroll
            for (int r = 0; r < R; r++) {
                const float prod = __int_as_float(e[u].y) * x[u][r];
                x[u][r] = on ? prod : 0.0f;
            }
        }
#pragma unroll
        for (int u = 0; u < kSplitBatch; u++)
#pragma unroll
            for (int r = 0; r < R; r++) {
                acc[r] = acc[r] + quad_value<0>(x[u][r]);
                acc[r] = acc[r] + quad_value<1>(x[u][r]);
                acc[r] = acc[r] + quad_value<2>(x[u][r]);
                acc[r] = acc[r] + quad_value<3>(x[u][r]);
            }
    }
    const int nv = wave_read(ch.v, lane + gs);
    const int nout = wave_read(ch.out, lane + gs);
    const bool cont = mine && g + 1 < per && c + 1 < n && nout < 0 && nv == ch.v;
    if (__any(cont)) {
        for (int j = per - 2; j >= 0; j--) {  // wave-uniform
            float y[R];
#pragma unroll
            for (int r = 0; r < R; r++) y[r] = wave_read(acc[r], lane + gs);
            if (cont && g == j)
#pragma unroll
                for (int r = 0; r < R; r++) acc[r] = acc[r] + y[r];
        }
    }
    if (mine && kk == 0 && ch.out >= 0) store_piece<R>(vals + (size_t)ch.out * ldv, k0, 0, acc);
}

// Tiled splat: block = one tile.  Stage 1 copies the tile's input rows, its entries
// (pixel index in the tile, weight) and its segments (beg, end, out) into LDS, every
// thread keeping kStage loads in flight; stage 2 gives the segments to the lane groups
// of the block, which sum them from LDS in the order of k_splat or k_splat_split (hence
// the same bits).
constexpr int kStage = 32;

template <int R>
__global__ void __launch_bounds__(1024) k_splat_tiled(TiledSplat ts, const int2* __restrict__ ent,
                                                            const float* __restrict__ in, float* __restrict__ vals,
                                                            int ldv, int L, int S, int per, int q_max) {
    extern __shared__ float sh[];
    const int t = xcd_block(blockIdx.x, gridDim.x);
    int p0, tw, th, stride;
    tile_rect(ts.geom, t, p0, tw, th, stride);
    const int e0 = ts.tile_e[t], ne = ts.tile_e[t + 1] - e0;
    const int c0 = ts.tile_seg[t], ns = ts.tile_seg[t + 1] - c0;
    const int rowf = tw * L;
    const int n1 = th * rowf, n3 = n1 + 2 * ne, n4 = n3 + 3 * ns;
    const float inv_rowf = 1.0f / (float)rowf;
    const long long rskip = (long long)stride * L - rowf;  // gap between two tile rows in `in`
    const unsigned* __restrict__ qsrc = reinterpret_cast<const unsigned*>(in) + (size_t)p0 * L;
    const unsigned* __restrict__ esrc = reinterpret_cast<const unsigned*>(ent + e0);
    const unsigned* __restrict__ csrc = reinterpret_cast<const unsigned*>(ts.chunks + c0);
    unsigned* shu = reinterpret_cast<unsigned*>(sh);
    // LDS: [rows: q_max floats][entries: e_max (index, weight) pairs][segments: 3 s_max]
    const int nt = blockDim.x;
    // every load is unconditional (index clamped to the last element, source chosen by
    // select), so the kStage loads of a thread are in flight together; stores follow
    for (int b = threadIdx.x; b < n4; b += kStage * nt) {
        unsigned x[kStage];
#pragma unroll
        for (int u = 0; u < kStage; u++) {
            const int i = min(b + u * nt, n4 - 1);
            int r = (int)((float)i * inv_rowf);  // row of the tile (exact within one for i < 2^24)
            r -= r * rowf > i ? 1 : 0;
            r += (r + 1) * rowf <= i ? 1 : 0;
            const int j = i - n3;
            const int c = j / 3;
            const unsigned* q = qsrc + (i + (long long)r * rskip);
            const unsigned* e = esrc + (i - n1);
            const unsigned* h = csrc + (4 * c + 1 + (j - 3 * c));  // Chunk {v, beg, end, out}
            x[u] = *(i < n1 ? q : (i < n3 ? e : h));
        }
#pragma unroll
        for (int u = 0; u < kStage; u++) {
            const int i = b + u * nt;
            if (i < n4) {
                const int off = i < n1 ? 0 : (i < n3 ? q_max - n1 : q_max + 2 * ts.e_max - n3);
                shu[i + off] = x[u];
            }
        }
    }
    __syncthreads();
    const float* tq = sh;
    const int2* te = reinterpret_cast<const int2*>(sh + q_max);
    const int* tsg = reinterpret_cast<const int*>(sh + q_max + 2 * ts.e_max);
    LaneGroup<true, R> G(L, S, per, nullptr);
    if (!G.on) return;  // no barrier below
    const int groups = (nt / 64) * per;
    const int k0 = G.k0;
    for (int c = (threadIdx.x >> 6) * per + G.g; c < ns; c += groups) {
        const int b = tsg[3 * c] - e0, e = tsg[3 * c + 1] - e0, out = tsg[3 * c + 2];
        float acc[R];
#pragma unroll
        for (int r = 0; r < R; r++) acc[r] = 0.0f;
        auto add = [&](float ww, const float (&x)[R]) {
#pragma unroll
            for (int r = 0; r < R; r++) acc[r] = add_product(acc[r], ww, x[r]);
        };
        int i = b;
        for (; i + 4 <= e; i += 4) {
            int pp[4];
            float ww[4], xx[4][R];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int2 x = te[i + u];
                pp[u] = x.x;
                ww[u] = __int_as_float(x.y);
            }
#pragma unroll
            for (int u = 0; u < 4; u++) load_piece<R>(tq + pp[u] * L, k0, L, xx[u]);
#pragma unroll
            for (int u = 0; u < 4; u++) add(ww[u], xx[u]);
        }
        for (; i < e; i++) {
            float xx[R];
            const int2 x = te[i];
            load_piece<R>(tq + x.x * L, k0, L, xx);
            add(__int_as_float(x.y), xx);
        }
        store_piece<R>(vals + (size_t)out * ldv, k0, L, acc);
    }
}

// (Sequential lists have vertices of hundreds of partial rows, added one after another:
// kLong loads in flight for those.  512x512x21: 16.1 -> 10.8 us.)
constexpr int kLong = 16;
template <bool WAVE, int R>
__global__ void __launch_bounds__(1024) k_combine(const Combine* __restrict__ cb, int n, float* __restrict__ vals,
                                                  int ldv, int L, int S, int per) {
    LaneGroup<WAVE, R> G(L, S, per, nullptr);
    const int c = G.item();
    if (!G.on || c >= n) return;
    const int k0 = G.k0;
    const Combine rc = cb[c];
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; r++) acc[r] = 0.0f;
    int i = 0;
    for (; i + kLong <= rc.count; i += kLong) {
        float xx[kLong][R];
#pragma unroll
        for (int u = 0; u < kLong; u++) load_piece<R>(vals + (size_t)(rc.first + i + u) * ldv, k0, L, xx[u]);
#pragma unroll
        for (int u = 0; u < kLong; u++)
#pragma unroll
            for (int r = 0; r < R; r++) acc[r] = acc[r] + xx[u][r];
    }
    for (; i < rc.count; i += kBatch) {  // count >= 2; loads clamped to the last row
        float xx[kBatch][R];
#pragma unroll
        for (int u = 0; u < kBatch; u++)
            load_piece<R>(vals + (size_t)(rc.first + min(i + u, rc.count - 1)) * ldv, k0, L, xx[u]);
#pragma unroll
        for (int u = 0; u < kBatch; u++)
            if (i + u < rc.count)
#pragma unroll
                for (int r = 0; r < R; r++) acc[r] = acc[r] + xx[u][r];
    }
    store_piece<R>(vals + (size_t)rc.v * ldv, k0, L, acc);
}

// One-launch recombination (wave mode).  Items are lane-group sums of cb[c].count
// partial rows from cb[c].first.  An item with pad == 0 is a whole vertex and stores
// its sum as row cb[c].v (count 0: a filler, stores nothing).  A vertex with more rows
// fills one whole wave: its items (pad = the number of pieces, the fillers after them
// count 0) sum one piece each; the pieces go to the wave's LDS rows and group 0 adds them
// in piece order and stores the vertex row.  A wave holds either light items or one
// heavy vertex, so the branch is uniform per wave.
template <int R>
__global__ void __launch_bounds__(kWaveBlock) k_combine_waves(const Combine* __restrict__ cb, int n,
                                                              float* __restrict__ vals, int ldv, int L, int S,
                                                              int per) {
    extern __shared__ float rows_lds[];  // per wave: per rows of L floats
    LaneGroup<true, R> G(L, S, per, nullptr);
    const int c = G.item();
    const int cw = c - G.g;  // the wave's first item
    if (cw >= n) return;     // whole waves only: no item of this wave exists
    const bool live = G.on && c < n;
    const Combine rc = live ? cb[c] : Combine{0, 0, 0, 0};
    const int k0 = G.k0;
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; r++) acc[r] = 0.0f;
    for (int i = 0; i < rc.count; i += kBatch) {  // loads clamped to the last row
        float xx[kBatch][R];
#pragma unroll
        for (int u = 0; u < kBatch; u++)
            load_piece<R>(vals + (size_t)(rc.first + min(i + u, rc.count - 1)) * ldv, k0, L, xx[u]);
#pragma unroll
        for (int u = 0; u < kBatch; u++)
            if (i + u < rc.count)
#pragma unroll
                for (int r = 0; r < R; r++) acc[r] = acc[r] + xx[u][r];
    }
    const Combine head = cb[cw];  // uniform over the wave
    if (head.pad == 0) {
        if (rc.count > 0) store_piece<R>(vals + (size_t)rc.v * ldv, k0, L, acc);
        return;
    }
    float* wrows = rows_lds + (size_t)G.w * per * L;
    if (G.on && G.g < head.pad) store_piece<R>(wrows + (size_t)G.g * L, k0, L, acc);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    if (G.on && G.g == 0) {
        float sum[R];
#pragma unroll
        for (int r = 0; r < R; r++) sum[r] = 0.0f;
        for (int j = 0; j < head.pad; j++) {
            float x[R];
            load_piece<R>(wrows + (size_t)j * L, k0, L, x);
#pragma unroll
            for (int r = 0; r < R; r++) sum[r] = sum[r] + x[r];
        }
        store_piece<R>(vals + (size_t)head.v * ldv, k0, L, sum);
    }
}

template <bool WAVE, int R>
__global__ void __launch_bounds__(1024) k_blur(const float* __restrict__ src, float* __restrict__ dst, int v0,
                                               int Vp, int ldv, int L, int S, int per, BlurTable bt, int step,
                                               int reverse) {
    LaneGroup<WAVE, R> G(L, S, per, nullptr);
    const int v = v0 + G.item();  // vertices [v0, Vp)
    if (!G.on || v >= Vp) return;
    const int k0 = G.k0;
    // terms are ordered by vbase; pick the last one starting at or before v
    int vb = bt.t[0].vbase, V = bt.t[0].V, d = bt.t[0].d;
    const int2* nbr = bt.t[0].nbr;
#pragma unroll
    for (int k = 1; k < DCRF_MAX_TERMS; k++) {
        if (k < bt.nterms && v >= bt.t[k].vbase) {
            vb = bt.t[k].vbase;
            V = bt.t[k].V;
            d = bt.t[k].d;
            nbr = bt.t[k].nbr;
        }
    }
    const int j = reverse ? d - step : step;
    float o[R], a[R], b[R], out[R];
    const int2 nb = nbr[(size_t)j * V + (v - vb)];
    load_piece<R>(src + (size_t)v * ldv, k0, L, o);
    load_piece<R>(src + (size_t)nb.x * ldv, k0, L, a);
    load_piece<R>(src + (size_t)nb.y * ldv, k0, L, b);
#pragma unroll
    for (int r = 0; r < R; r++) {
        const float s2 = a[r] + b[r];
        out[r] = fmaf(0.5f, s2, o[r]);
    }
    store_piece<R>(dst + (size_t)v * ldv, k0, L, out);
}

// A pass of K = 1 or 2 consecutive blur steps (axes a_1 .. a_K) of one term.  Each step
// is x' = x + 0.5 (x_n1 + x_n2) in k_blur's operation order; the pass table lists per
// vertex v the 3^K rows of the step tree: level K holds v and its two neighbours along
// a_K, each expanded along a_{K-1}, and so on, zero row for an absent vertex (whose
// value is 0 at every level, as in the intermediate buffers of single steps).  The
// kernel loads the 3^K rows together and folds them level by level: the same bits as
// K launches of k_blur, with K-1 fewer launches and no intermediate rows written.
__device__ __forceinline__ float blur_fold(float o, float a, float b) {
    const float s2 = a + b;
    return fmaf(0.5f, s2, o);
}

// zr: the zero row (absent neighbours point to it; it holds zeros in every vertex
// buffer), whose loads are skipped: a group that has it takes 0.0f instead, the value
// the load would give, and its lanes issue no memory access.  Half of the rows of a
// sparse (bilateral) lattice's pass are absent neighbours.
template <int K, int R>
__device__ __forceinline__ void blur_pass_vertex(const float* __restrict__ src, float* __restrict__ dst,
                                                 const int* __restrict__ e, int v, int ldv, int k0, int L, int zr) {
    constexpr int NR = K == 1 ? 3 : (K == 2 ? 9 : 27);
    int idx[NR];
#pragma unroll
    for (int i = 0; i < NR; i++) idx[i] = e[i];
    float x[NR][R];
#pragma unroll
    for (int i = 0; i < NR; i++) {
        if (idx[i] != zr) {
            load_piece<R>(src + (size_t)idx[i] * ldv, k0, L, x[i]);
        } else {
#pragma unroll
            for (int r = 0; r < R; r++) x[i][r] = 0.0f;
        }
    }
    float out[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        float y[NR];
#pragma unroll
        for (int i = 0; i < NR; i++) y[i] = x[i][r];
        int n = NR;
#pragma unroll
        for (int lev = 0; lev < K; lev++) {
#pragma unroll
            for (int i = 0; i < NR / 3; i++)
                if (i < n / 3) y[i] = blur_fold(y[3 * i], y[3 * i + 1], y[3 * i + 2]);
            n /= 3;
        }
        out[r] = y[0];
    }
    store_piece<R>(dst + (size_t)v * ldv, k0, L, out);
}

// A pass of three steps: the 27-row tree as its three 9-row subtrees (top-level child c
// at rows 9c .. 9c + 8), one after the other, so that at most 9 rows are held at once
// (a pass of three steps over all 27 rows would need ~80 VGPRs at three labels per
// lane and lower the occupancy of every pass of the launch).  Same folds, in the same
// order, as blur_pass_vertex<3>.
template <int R>
__device__ __forceinline__ void blur_pass_vertex3(const float* __restrict__ src, float* __restrict__ dst,
                                                  const int* __restrict__ e, int v, int ldv, int k0, int L, int zr) {
    float s[3][R];
#pragma unroll 1
    for (int c = 0; c < 3; c++) {
        int idx[9];
#pragma unroll
        for (int i = 0; i < 9; i++) idx[i] = e[9 * c + i];
        float x[9][R];
#pragma unroll
        for (int i = 0; i < 9; i++) {
            if (idx[i] != zr) {
                load_piece<R>(src + (size_t)idx[i] * ldv, k0, L, x[i]);
            } else {
#pragma unroll
                for (int r = 0; r < R; r++) x[i][r] = 0.0f;
            }
        }
#pragma unroll
        for (int r = 0; r < R; r++) {
            const float a = blur_fold(x[0][r], x[1][r], x[2][r]);
            const float b = blur_fold(x[3][r], x[4][r], x[5][r]);
            const float d = blur_fold(x[6][r], x[7][r], x[8][r]);
            const float t = blur_fold(a, b, d);
            // (a runtime index into s would put it in scratch memory)
            if (c == 0) s[0][r] = t;
            else if (c == 1) s[1][r] = t;
            else s[2][r] = t;
        }
    }
    float out[R];
#pragma unroll
    for (int r = 0; r < R; r++) out[r] = blur_fold(s[0][r], s[1][r], s[2][r]);
    store_piece<R>(dst + (size_t)v * ldv, k0, L, out);
}

template <bool WAVE, int R>
__global__ void __launch_bounds__(1024) k_blur_pass(const float* __restrict__ src, float* __restrict__ dst, int v0,
                                                    int Vp, int ldv, int L, int S, int per, PassTable pt) {
    LaneGroup<WAVE, R> G(L, S, per, nullptr);
    const int v = v0 + G.item();  // vertices [v0, Vp)
    if (!G.on || v >= Vp) return;
    const int k0 = G.k0;
    int vb = pt.t[0].vbase, steps = pt.t[0].steps;
    const int* tab = pt.t[0].tab;
#pragma unroll
    for (int k = 1; k < DCRF_MAX_TERMS; k++) {
        if (k < pt.nterms && v >= pt.t[k].vbase) {
            vb = pt.t[k].vbase;
            tab = pt.t[k].tab;
            steps = pt.t[k].steps;
        }
    }
    const size_t lv = (size_t)(v - vb);
    if (steps == 2)
        blur_pass_vertex<2, R>(src, dst, tab + lv * 9, v, ldv, k0, L, pt.zero_row);
    else if (steps == 3)
        blur_pass_vertex3<R>(src, dst, tab + lv * 27, v, ldv, k0, L, pt.zero_row);
    else
        blur_pass_vertex<1, R>(src, dst, tab + lv * 3, v, ldv, k0, L, pt.zero_row);
}

// Pass table of one term: entry (i_K, .., i_1) of vertex v at v*3^K + sum i_j 3^(j-1),
// expanding along axis ax[j-1] at level j (ax[K-1] first, the pass's last step).
__global__ void k_pass_tables(PassTableJobs J) {
    const PassTableJob& T = J.job[blockIdx.y];
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    const int V = T.V, vbase = T.vbase, zero_row = T.zero_row, K = T.K;
    if (v >= V) return;
    const int2* __restrict__ nbr = T.nbr;
    const int* ax = T.axes;
    int* __restrict__ tab = T.tab;
    int cur[27], nxt[27];
    cur[0] = vbase + v;
    int n = 1;
    for (int lev = K - 1; lev >= 0; lev--) {
        // expand every row of the current level along axis ax[lev]: (u, n1(u), n2(u))
        for (int i = 0; i < n; i++) {
            const int u = cur[i];
            const int2 nb = u == zero_row ? make_int2(zero_row, zero_row) : nbr[(size_t)ax[lev] * V + (u - vbase)];
            nxt[3 * i] = u;
            nxt[3 * i + 1] = nb.x;
            nxt[3 * i + 2] = nb.y;
        }
        n *= 3;
        for (int i = 0; i < n; i++) cur[i] = nxt[i];
    }
    for (int i = 0; i < n; i++) tab[(size_t)v * n + i] = cur[i];
}

// Mean-field update of one pixel: E = -U - sum_k C_k(w_k slice_k), Q = softmax(-E)
// (densecrf.cpp:122-129, with the per-term weight w_k = 1 unless set).
template <bool WAVE, int R, bool CWL>
__global__ void __launch_bounds__(1024) k_meanfield(const float* __restrict__ U, float* __restrict__ Q, int ldq,
                                                    int N, int L, int S, int per, SliceTable st,
                                                    float* __restrict__ tmp1, float* __restrict__ tmp2) {
    extern __shared__ float sh[];
    float* shc = sh + blockDim.x;  // compat region after the group scratch
    if (CWL) stage_compat(st, L, shc);
    LaneGroup<WAVE, R> G(L, S, per, sh);
    const int p = G.item();
    const bool active = G.on && p < N;
    const int k0 = G.k0;
    float e[R], last[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        e[r] = 0.0f;
        last[r] = 0.0f;
    }
    if (active && U) {
        load_row(U + (size_t)p * L, G, e);
#pragma unroll
        for (int r = 0; r < R; r++) e[r] = -e[r];
    }
#pragma unroll
    for (int k = 0; k < DCRF_MAX_TERMS; k++) {
        if (k < st.nterms) {
            const SliceTerm& T = st.t[k];
            float m[R], c[R];
            if (active) {
                slice_piece<R>(T, p, k0, L, m);
                if (T.mout) store_row(T.mout + (size_t)p * L, G, m);
            } else {
#pragma unroll
                for (int r = 0; r < R; r++) m[r] = 0.0f;
            }
            if (T.kw) {
                const float kw = T.kw[0];
#pragma unroll
                for (int r = 0; r < R; r++) m[r] = m[r] * kw;
            }
            compat_piece<WAVE, R>(T, m, c, G, shc);
#pragma unroll
            for (int r = 0; r < R; r++) {
                e[r] = e[r] - c[r];
                last[r] = c[r];
            }
        }
    }
    G.pad(e, -INFINITY);
    const float mx = G.all_max(e);
    float x[R];
#pragma unroll
    for (int r = 0; r < R; r++) x[r] = expf(e[r] - mx);
    const float s = G.all_sum(x);
    if (active) {
        float q[R];
        divide_all<R>(x, s, q);
        store_row(Q + (size_t)p * ldq, ldq, G, q);
        if (tmp1) store_row(tmp1 + (size_t)p * L, G, e);
        if (tmp2) store_row(tmp2 + (size_t)p * L, G, last);
    }
}

// slc[p][off + j] = (vtx[p][j], bits of sw[p][j]) for j < d1; rows of ds pairs.
__global__ void k_interleave_slice(const int* __restrict__ vtx, const float* __restrict__ sw, int N, int d1, int ds,
                                   int off, int2* __restrict__ slc) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)N * d1) return;
    const size_t p = i / d1, j = i - p * d1;
    slc[p * ds + off + j] = make_int2(vtx[i], __float_as_int(sw[i]));
}

// out = compat_which(slice_which) (ckind < 0: the plain slice).
template <bool WAVE, int R, bool CWL>
__global__ void __launch_bounds__(1024) k_slice_term(float* __restrict__ out, int N, int L, int S, int per,
                                                     SliceTable st, int which) {
    extern __shared__ float sh[];
    float* shc = sh + blockDim.x;
    if (CWL) stage_compat(st, L, shc);
    LaneGroup<WAVE, R> G(L, S, per, sh);
    const int p = G.item();
    const bool active = G.on && p < N;
    SliceTerm T = st.t[0];
#pragma unroll
    for (int k = 1; k < DCRF_MAX_TERMS; k++)
        if (k == which) T = st.t[k];
    float m[R], c[R];
    if (active) {
        slice_piece<R>(T, p, G.k0, L, m);
    } else {
#pragma unroll
        for (int r = 0; r < R; r++) m[r] = 0.0f;
    }
    if (T.kw) {
        const float kw = T.kw[0];
#pragma unroll
        for (int r = 0; r < R; r++) m[r] = m[r] * kw;
    }
    if (T.ckind >= 0) {
        compat_piece<WAVE, R>(T, m, c, G, shc);
    } else {
#pragma unroll
        for (int r = 0; r < R; r++) c[r] = m[r];
    }
    if (active) store_row(out + (size_t)p * L, G, c);
}

// KL divergence terms per pixel, reduced per block in double in a fixed order
// (densecrf.cpp:214-235: q log max(q,1e-20) + u q + sum_k q * pairwise_k(Q)).
template <bool WAVE, int R, bool CWL>
__global__ void __launch_bounds__(1024) k_kl(const float* __restrict__ Q, const float* __restrict__ U, int N, int L,
                                             int S, int per, SliceTable st, double* __restrict__ partial) {
    extern __shared__ float sh[];
    __shared__ double red[1024];
    float* shc = sh + blockDim.x;
    if (CWL) stage_compat(st, L, shc);
    LaneGroup<WAVE, R> G(L, S, per, sh);
    const int p = G.item();
    const bool active = G.on && p < N;
    const int k0 = G.k0;
    float q[R], u[R];
#pragma unroll
    for (int r = 0; r < R; r++) {
        q[r] = 0.0f;
        u[r] = 0.0f;
    }
    double acc = 0.0;
    if (active) {
        load_row(Q + (size_t)p * L, G, q);
        if (U) load_row(U + (size_t)p * L, G, u);
#pragma unroll
        for (int r = 0; r < R; r++)
            if (G.has(r)) {
                const float qc = q[r] > 1e-20f ? q[r] : 1e-20f;
                acc += (double)q[r] * log((double)qc);
                if (U) acc += (double)(u[r] * q[r]);
            }
    }
#pragma unroll
    for (int k = 0; k < DCRF_MAX_TERMS; k++) {
        if (k < st.nterms) {
            const SliceTerm& T = st.t[k];
            float m[R], c[R];
            if (active) {
                slice_piece<R>(T, p, k0, L, m);
            } else {
#pragma unroll
                for (int r = 0; r < R; r++) m[r] = 0.0f;
            }
            if (T.kw) {
                const float kw = T.kw[0];
#pragma unroll
                for (int r = 0; r < R; r++) m[r] = m[r] * kw;
            }
            compat_piece<WAVE, R>(T, m, c, G, shc);
            if (active)
#pragma unroll
                for (int r = 0; r < R; r++)
                    if (G.has(r)) acc += (double)(q[r] * c[r]);
        }
    }
    const int t = threadIdx.x;
    red[t] = acc;
    __syncthreads();
    for (int s = blockDim.x / 2; s > 0; s >>= 1) {
        if (t < s) red[t] += red[t + s];
        __syncthreads();
    }
    if (t == 0) partial[blockIdx.x] = red[0];
}

// DenseKernel::initLattice normalisers (pairwise.cpp:54-61), in double like the reference.
// The normalisers of every term (blockIdx.y) from the filtered all-ones rows: slice, then
// the normalisation (pairwise.cpp:44-61).  Bound: the gathers of single floats.  Both terms at
// 1024x768: 22 us; slice weights, slice and normalisation in launches of their own 58 us.
__global__ void k_norms(NormTerms M, int N) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= N) return;
    const NormTerm& T = M.t[blockIdx.y];
    const int* __restrict__ vt = T.vtx + (size_t)p * T.d1;
    const float* __restrict__ bary = T.bary + (size_t)p * T.d1;
    float x = 0.0f;
#pragma unroll 4
    for (int j = 0; j < T.d1; j++) x = add_product(x, bary[j] * T.alpha, T.vals[vt[j] + T.vbase]);
    const double y = (double)x + 1e-20;
    if (T.ntype == DCRF_NORMALIZE_SYMMETRIC)
        x = (float)(1.0 / sqrt(y));
    else if (T.ntype == DCRF_NORMALIZE_BEFORE || T.ntype == DCRF_NORMALIZE_AFTER)
        x = (float)(1.0 / y);
    T.norm[p] = x;
}

__global__ void k_remap_nbr(const int* __restrict__ src, int2* __restrict__ dst, int n, int vbase,
                            int zero_row) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int a = src[2 * (size_t)i], b = src[2 * (size_t)i + 1];
    dst[i] = make_int2(a >= 0 ? a + vbase : zero_row, b >= 0 ? b + vbase : zero_row);
}

// The sorted entries' (pixel, weight) pairs of term `term` in the groups' order.  Bound: the
// random reads of the weights, which stay inside a tile: each XCD takes one range of them.
// 1024x768: 33 -> 24.5 us a launch.
__global__ void k_entry_gather(const int* __restrict__ csr_e, int E, int d1, const float* __restrict__ bary,
                               const float* __restrict__ norm, int use_norm, const int* __restrict__ tile_ptr,
                               const int* __restrict__ gebase, int n_tiles, int T, int term, TileGeom g, int local,
                               int pix_off, int2* __restrict__ ent) {
    const int j = xcd_block(blockIdx.x, gridDim.x) * kThreads + (int)threadIdx.x;
    if (j >= E) return;
    const int e = csr_e[j];
    const int p = e / d1;
    int t = last_le(tile_ptr, n_tiles, __builtin_amdgcn_readfirstlane(j));  // one search a wave
    if (j >= tile_ptr[t + 1]) t = last_le(tile_ptr, n_tiles, j);
    const int pos = gebase[t * T + term] + (j - tile_ptr[t]);
    const float b = bary[e];
    const float w = use_norm ? b * norm[p] : b;
    ent[pos] = make_int2((local ? tile_local(g, p) : p) + pix_off, __float_as_int(w));
}

__global__ void k_slice_weights(const int* __restrict__ vtx, const float* __restrict__ bary,
                                const float* __restrict__ norm, int use_norm, float alpha, int N, int d1,
                                int vbase, int* __restrict__ gvtx, float* __restrict__ sw, int2* __restrict__ slc,
                                int ds, int off) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)N * d1) return;
    const size_t p = i / d1;
    const int v = vtx[i] + vbase;
    const float wa = bary[i] * alpha;
    const float w = use_norm ? wa * norm[p] : wa;
    gvtx[i] = v;
    sw[i] = w;
    if (slc) slc[p * ds + off + (i - p * d1)] = make_int2(v, __float_as_int(w));
}

// DenseCRF::currentMap (densecrf.cpp:202-211): out[p] = the first label of the largest
// Q[p][l] (a later label replaces it only when strictly larger, as Eigen's maxCoeff
// visitor does), one thread per pixel.
__global__ void k_argmax(const float* __restrict__ Q, int ldq, int N, int L, int16_t* __restrict__ out) {
    const int p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= N) return;
    const float* row = Q + (size_t)p * ldq;
    float best = row[0];
    int arg = 0;
    for (int l = 1; l < L; l++) {
        const float v = row[l];
        if (v > best) {
            best = v;
            arg = l;
        }
    }
    out[p] = (int16_t)arg;
}

// out (rows of ldo floats) = in (rows of ldi), L labels and zeros in out's padding labels;
// n floats of out.
__global__ void k_restride_rows(const float* __restrict__ in, int ldi, float* __restrict__ out, int ldo, size_t n,
                                int L) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const size_t p = i / ldo;
    const int l = (int)(i - p * ldo);
    out[i] = l < L ? in[p * ldi + l] : 0.0f;
}

// out[c][r] = in[r][c] for an rows x cols row-major input, 32x32 tiles through LDS.
__global__ void k_transpose(const float* __restrict__ in, float* __restrict__ out, int rows, int cols) {
    __shared__ float tile[32][33];
    const int bx = blockIdx.x * 32, by = blockIdx.y * 32;
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 256 threads: 32 x 8
    for (int k = 0; k < 32; k += 8) {
        const int r = by + ty + k, c = bx + tx;
        if (r < rows && c < cols) tile[ty + k][tx] = in[(size_t)r * cols + c];
    }
    __syncthreads();
    for (int k = 0; k < 32; k += 8) {
        const int c = bx + ty + k, r = by + tx;
        if (r < rows && c < cols) out[(size_t)c * rows + r] = tile[tx][ty + k];
    }
}

}  // namespace

void launch_fill(float* p, float v, size_t n, hipStream_t s) {
    if (!n) return;
    k_fill<<<blocks_for(n), kThreads, 0, s>>>(p, v, n);
    DCRF_HIP_CHECK(hipGetLastError());
}

void launch_argmax(const float* Q, int ldq, int N, int L, int16_t* out, hipStream_t s) {
    if (N <= 0) return;
    k_argmax<<<blocks_for(N), kThreads, 0, s>>>(Q, ldq, N, L, out);
    DCRF_HIP_CHECK(hipGetLastError());
}

void launch_restride_rows(const float* in, int ldi, float* out, int ldo, int N, int L, hipStream_t s) {
    const size_t n = (size_t)N * ldo;
    if (!n) return;
    k_restride_rows<<<blocks_for(n), kThreads, 0, s>>>(in, ldi, out, ldo, n, L);
    DCRF_HIP_CHECK(hipGetLastError());
}

void launch_transpose(const float* in, float* out, int rows, int cols, hipStream_t s) {
    if (!rows || !cols) return;
    dim3 grid((cols + 31) / 32, (rows + 31) / 32);
    k_transpose<<<grid, 256, 0, s>>>(in, out, rows, cols);
    DCRF_HIP_CHECK(hipGetLastError());
}

// Rows whose offsets row_piece<true> can form: 24-bit row numbers and row sizes, 32-bit
// byte offsets.
bool narrow_rows(size_t rows, int ld) {
    return rows <= ((size_t)1 << 24) && ld < (1 << 22) && rows * (size_t)ld * sizeof(float) <= 0xffffffffull;
}

void launch_splat(const Chunk* chunks, int n_chunks, const int2* ent, const float* in, size_t rows_in, int ldi,
                  float* vals, int ldv, int L, hipStream_t s) {
    if (!n_chunks) return;
    const LaunchShape sh = shape_for(L);
    const SplatShape sp = splat_shape(L);
    if (sp.K > 1) {
        const bool narrow = narrow_rows(rows_in, ldi);
        const unsigned grid = blocks_for(n_chunks, (kWaveBlock / 64) * sp.per);
#define DCRF_SPLIT(R_)                                                                              \
    case R_:                                                                                        \
        (narrow ? k_splat_split<R_, true> : k_splat_split<R_, false>)<<<grid, kWaveBlock, 0, s>>>(    \
            chunks, n_chunks, ent, in, ldi, vals, ldv, sh.S, sp.per);                                 \
        break;
        switch (sh.R) {
            DCRF_SPLIT(1) DCRF_SPLIT(2) DCRF_SPLIT(3) DCRF_SPLIT(4)
            default: throw Error{DCRF_ERR_STATE, "no split splat kernel for this shape"};
        }
#undef DCRF_SPLIT
        DCRF_HIP_CHECK(hipGetLastError());
        return;
    }
    const size_t shm = sh.wave ? (size_t)(kWaveBlock / 64) * (kWin + kBatch) * sizeof(int2) : 0;
    if (narrow_rows(rows_in, ldi))
        DCRF_DISPATCH_T(sh, k_splat, true, blocks_for(n_chunks, sh.items), shm, s, chunks, n_chunks, ent, in, ldi, vals,
                        ldv, L, sh.S, sh.per);
    else
        DCRF_DISPATCH_T(sh, k_splat, false, blocks_for(n_chunks, sh.items), shm, s, chunks, n_chunks, ent, in, ldi,
                        vals, ldv, L, sh.S, sh.per);
}

size_t tiled_splat_lds(int L, int side, int e_max, int s_max, size_t lds_cap) {
    const LaunchShape sh = shape_for(L);
    if (!sh.wave) return 0;
    const size_t words = (((size_t)side * side * L + 1) & ~(size_t)1) + 2 * (size_t)e_max + 3 * (size_t)s_max;
    const size_t bytes = words * sizeof(float);
    return bytes <= lds_cap ? bytes : 0;
}

// Workgroup size of the tiled splat: 1024 threads (16 waves of lane groups) once a tile
// takes more than a quarter of the workgroup LDS limit, else 256.
int tiled_splat_block(size_t lds, size_t lds_cap) { return lds * 4 > lds_cap ? 1024 : kWaveBlock; }

void launch_splat_tiled(const TiledSplat& ts, const int2* ent, const float* in, float* vals, int ldv, int L,
                        size_t lds_cap, hipStream_t s) {
    if (!ts.n_tiles) return;
    const LaunchShape sh = shape_for(L);
    const size_t lds = tiled_splat_lds(L, ts.geom.side, ts.e_max, ts.s_max, lds_cap);
    if (!lds) throw Error{DCRF_ERR_VALUE, "tiled splat does not fit the LDS of a block"};
    const int q_max = (ts.geom.side * ts.geom.side * L + 1) & ~1;  // the entry pairs start 8-byte aligned
    const int block = tiled_splat_block(lds, lds_cap);
    // dynamic LDS beyond the default launch limit must be granted per kernel
    static size_t granted[5] = {};
    auto grant = [&](const void* fn, int r) {
        if (lds > granted[r]) {
            DCRF_HIP_CHECK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            granted[r] = lds;
        }
    };
#define DCRF_TILED(R_)                                                                                   \
    case R_:                                                                                             \
        grant(reinterpret_cast<const void*>(&k_splat_tiled<R_>), R_);                                     \
        k_splat_tiled<R_><<<ts.n_tiles, block, lds, s>>>(ts, ent, in, vals, ldv, L, sh.S, sh.per, q_max); \
        break;
    switch (sh.R) {
        DCRF_TILED(1) DCRF_TILED(2) DCRF_TILED(3) DCRF_TILED(4)
        default: throw Error{DCRF_ERR_STATE, "no tiled splat kernel for this shape"};
    }
#undef DCRF_TILED
    DCRF_HIP_CHECK(hipGetLastError());
}

void launch_combine(const Combine* c, int n, float* vals, int ldv, int L, hipStream_t s) {
    if (!n) return;
    const LaunchShape sh = shape_for(L);
    DCRF_DISPATCH(sh, k_combine, blocks_for(n, sh.items), 0, s, c, n, vals, ldv, L, sh.S, sh.per);
}

void launch_combine_waves(const Combine* c, int n, float* vals, int ldv, int L, hipStream_t s) {
    if (!n) return;
    const LaunchShape sh = shape_for(L);
    if (!sh.wave) throw Error{DCRF_ERR_STATE, "one-launch combine: wave-mode shapes only"};
    const size_t lds = sizeof(float) * (kWaveBlock / 64) * sh.per * L;
    const unsigned grid = blocks_for(n, sh.items);
    switch (sh.R) {
        case 1: k_combine_waves<1><<<grid, kWaveBlock, lds, s>>>(c, n, vals, ldv, L, sh.S, sh.per); break;
        case 2: k_combine_waves<2><<<grid, kWaveBlock, lds, s>>>(c, n, vals, ldv, L, sh.S, sh.per); break;
        case 3: k_combine_waves<3><<<grid, kWaveBlock, lds, s>>>(c, n, vals, ldv, L, sh.S, sh.per); break;
        default: k_combine_waves<4><<<grid, kWaveBlock, lds, s>>>(c, n, vals, ldv, L, sh.S, sh.per); break;
    }
    DCRF_HIP_CHECK(hipGetLastError());
}

void launch_blur(const float* src, float* dst, int v0, int Vp, int ldv, int L, const BlurTable& bt, int step,
                 int reverse, hipStream_t s) {
    if (Vp <= v0) return;
    const LaunchShape sh = shape_for(L);
    DCRF_DISPATCH(sh, k_blur, blocks_for(Vp - v0, sh.items), 0, s, src, dst, v0, Vp, ldv, L, sh.S, sh.per, bt, step,
                  reverse);
}

void launch_blur_pass(const float* src, float* dst, int v0, int Vp, int ldv, int L, const PassTable& pt,
                      hipStream_t s, int R) {
    if (Vp <= v0) return;
    // R: labels per lane (0 = the default for L); the blur is elementwise per label, so
    // any lane split gives the same bits
    const LaunchShape sh = R > 0 && L % R == 0 ? shape_for_r(L, R) : shape_for(L);
    DCRF_DISPATCH(sh, k_blur_pass, blocks_for(Vp - v0, sh.items), 0, s, src, dst, v0, Vp, ldv, L, sh.S, sh.per, pt);
}

void launch_pass_tables(const std::vector<PassTableJob>& jobs, hipStream_t s) {
    constexpr size_t kMax = PassTableJobs::kMax;
    for (size_t i0 = 0; i0 < jobs.size(); i0 += kMax) {
        PassTableJobs J{};
        const size_t n = std::min(kMax, jobs.size() - i0);
        int V = 0;
        for (size_t i = 0; i < n; i++) {
            J.job[i] = jobs[i0 + i];
            if (J.job[i].K < 1 || J.job[i].K > 3) throw Error{DCRF_ERR_STATE, "blur pass: 1 to 3 steps"};
            V = std::max(V, J.job[i].V);
        }
        if (V <= 0) continue;
        k_pass_tables<<<dim3(blocks_for(V), (unsigned)n), kThreads, 0, s>>>(J);
        DCRF_HIP_CHECK(hipGetLastError());
    }
}

bool fused_meanfield_ok(int L, int nterms, int d1_0, int d1_1) {
    if (!shape_for(padded_labels(L)).wave) return false;
    if (nterms == 1) return d1_0 == 3 || d1_0 == 6;
    if (nterms == 2)
        return (d1_0 == 3 && d1_1 == 6) || (d1_0 == 6 && d1_1 == 3) || (d1_0 == 4 && d1_1 == 5) ||
               (d1_0 == 5 && d1_1 == 4);
    return false;
}

void launch_interleave_slice(const int* vtx, const float* sw, int N, int d1, int ds, int off, int2* slc,
                             hipStream_t s) {
    if (!N) return;
    k_interleave_slice<<<blocks_for((size_t)N * d1), kThreads, 0, s>>>(vtx, sw, N, d1, ds, off, slc);
    DCRF_HIP_CHECK(hipGetLastError());
}

namespace {
// Entry (pixel, weight) -> (its 8 x 8 block position, weight) for an image W pixels wide.
__global__ void k_entry_block(const int2* __restrict__ ent, size_t E, int W, int2* __restrict__ out) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < E) {
        const int2 e = ent[i];
        out[i] = make_int2(q_block_pos(e.x, W), e.y);
    }
}
}  // namespace

void launch_entry_block(const int2* ent, size_t E, int W, int2* out, hipStream_t s) {
    if (!E) return;
    k_entry_block<<<blocks_for(E), kThreads, 0, s>>>(ent, E, W, out);
    DCRF_HIP_CHECK(hipGetLastError());
}

int assign_compat_lds(SliceTable& st, int L, bool pad) {
    const int ldw = pad ? (L + 3) & ~3 : L;
    int total = 0;
    for (int k = 0; k < st.nterms; k++) {
        st.t[k].cw_lds = -1;
        st.t[k].ldw = ldw;
    }
    for (int k = 0; k < st.nterms; k++)
        if (st.t[k].ckind == DCRF_COMPAT_MATRIX && total + L * ldw <= kCompatLdsFloats) {
            st.t[k].cw_lds = total;
            total += L * ldw;
        }
    return total;
}

void launch_meanfield(const float* U, float* Q, int ldq, int N, int L, int Lv, const SliceTable& st_in, float* tmp1,
                      float* tmp2, hipStream_t s) {
    SliceTable st = st_in;
    const int cwf = assign_compat_lds(st, L);
    const LaunchShape sh = shape_for(Lv);
    DCRF_DISPATCH_CWL(sh, cwf, k_meanfield, blocks_for(N, sh.items), sizeof(float) * (sh.block + cwf), s, U, Q, ldq,
                      N, L, sh.S, sh.per, st, tmp1, tmp2);
}

void launch_softmax_neg(const float* U, float* Q, int ldq, int N, int L, int Lv, hipStream_t s) {
    SliceTable st{};
    st.nterms = 0;
    launch_meanfield(U, Q, ldq, N, L, Lv, st, nullptr, nullptr, s);
}

void launch_slice_term(float* out, int N, int L, int Lv, const SliceTable& st_in, int which, hipStream_t s) {
    SliceTable st = st_in;
    const int cwf = assign_compat_lds(st, L);
    const LaunchShape sh = shape_for(Lv);
    DCRF_DISPATCH_CWL(sh, cwf, k_slice_term, blocks_for(N, sh.items), sizeof(float) * (sh.block + cwf), s, out, N,
                      L, sh.S, sh.per, st, which);
}

int kl_blocks(int N, int Lv) { return (int)blocks_for(N, shape_for(Lv).items); }

void launch_kl(const float* Q, const float* U, int N, int L, int Lv, const SliceTable& st_in, double* partials,
               hipStream_t s) {
    SliceTable st = st_in;
    const int cwf = assign_compat_lds(st, L);
    const LaunchShape sh = shape_for(Lv);
    DCRF_DISPATCH_CWL(sh, cwf, k_kl, kl_blocks(N, Lv), sizeof(float) * (sh.block + cwf), s, Q, U, N, L, sh.S, sh.per, st,
                      partials);
}

void launch_norms(const NormTerms& terms, int N, hipStream_t s) {
    if (!N || !terms.T) return;
    k_norms<<<dim3(blocks_for(N), terms.T), kThreads, 0, s>>>(terms, N);
    DCRF_HIP_CHECK(hipGetLastError());
}

void launch_remap_nbr(const int* src, int2* dst, int n, int vbase, int zero_row, hipStream_t s) {
    if (!n) return;
    k_remap_nbr<<<blocks_for(n), kThreads, 0, s>>>(src, dst, n, vbase, zero_row);
    DCRF_HIP_CHECK(hipGetLastError());
}

void launch_entry_gather(const int* csr_e, int E, int d1, const float* bary, const float* norm, int use_norm,
                         const int* tile_ptr, const int* gebase, int n_tiles, int T, int i, const TileGeom* local,
                         int2* ent_out, hipStream_t s, int pix_off) {
    if (!E) return;
    const TileGeom g = local ? *local : TileGeom{};
    k_entry_gather<<<blocks_for(E), kThreads, 0, s>>>(csr_e, E, d1, bary, norm, use_norm, tile_ptr, gebase, n_tiles,
                                                      T, i, g, local ? 1 : 0, pix_off, ent_out);
    DCRF_HIP_CHECK(hipGetLastError());
}

void launch_slice_weights(const int* vtx, const float* bary, const float* norm, int use_norm, float alpha, int N,
                          int d1, int vbase, int* gvtx, float* sw, int2* slc, int ds, int off, hipStream_t s) {
    if (!N) return;
    k_slice_weights<<<blocks_for((size_t)N * d1), kThreads, 0, s>>>(vtx, bary, norm, use_norm, alpha, N, d1, vbase,
                                                                    gvtx, sw, slc, ds, off);
    DCRF_HIP_CHECK(hipGetLastError());
}

}  // namespace dcrf
