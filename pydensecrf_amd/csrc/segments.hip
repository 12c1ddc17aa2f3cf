// Splat segment and recombination lists, built on the device.
//
// A term's entries are sorted by (tile of the pixel, vertex, pixel); a run is a maximal
// range of one (tile, vertex).  RunSet merges the runs of several terms, tile by tile and
// inside a tile term by term (a group); a run is cut into segments of at most C entries.
// A SegLists lays the segments out for one row shape:
//   - every group starts a wave: empty fillers (v = out = -1) pad the group before, and the
//     vertices without entries (touched by padding lanes only) get empty segments in waves
//     of their own at the end;
//   - a run's segments inside one wave are added there (k_splat): the first one of them
//     (a head) carries the output row, the others out = -1;
//   - a vertex with one head over all tiles is written directly, the others get partial
//     rows, contiguous per vertex in list order, and an item in the recombination list.
// (Without in-wave runs, for the LDS-tiled splat, lane groups wider than a wave and
// sequential lists, every segment is a head and there are no fillers.)
//
// The host built these lists from downloaded runs before: at 1024x768 3.3 ms of a new
// model's 14 ms went into its loops, and the lists into the uploads.  Here each stage is a
// scan or one thread per run, vertex or group, the stages that do not wait for each other
// in one launch; the host reads one set of counts to size the lists.  The order of a
// vertex's partial rows is that of the stable sort by vertex, i.e. list order, so the sums
// do not depend on anything but the runs.
#include <cstring>
#include <limits>

#include <rocprim/rocprim.hpp>

#include "dcrf_internal.h"
#include "dcrf_device.h"

namespace dcrf {
namespace {

constexpr int kThreads = 256;
constexpr int kCombineSplit = 16;  // longest serial chain of partial rows in one item
inline unsigned blocks_for(size_t n) { return (unsigned)((n + kThreads - 1) / kThreads); }

// The terms of a run set, in its order.
struct MergeTerm {
    const int *run_v, *run_t, *run_beg, *tile_run, *tile_ptr;
    int n, vbase;
};
struct MergeTerms {
    int T;
    MergeTerm t[DCRF_MAX_TERMS];
};

// First element of group t * T + i, from the terms' first ones of each tile (tab: tile_run
// or tile_ptr): the terms' elements of the tiles before t, and of tile t those of the terms
// before i.
template <const int* MergeTerm::*tab>
__device__ __forceinline__ int group_first(const MergeTerms& M, int t, int i) {
    int n = 0;
    for (int k = 0; k < M.T; k++) n += (M.t[k].*tab)[k < i ? t + 1 : t];
    return n;
}

// The runs of every term (blockIdx.y) into the merged order: vertex (from vbase), first entry,
// entries, group, segments; and the first run and entry of every group.
__global__ void k_merge_runs(MergeTerms M, int NT, int C, int* __restrict__ mbase, int* __restrict__ gebase,
                             int* __restrict__ rv, int* __restrict__ rb, int* __restrict__ rl, int* __restrict__ rg,
                             int* __restrict__ ns, int* __restrict__ id) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y;
    const MergeTerm& m = M.t[i];
    if (r < NT || (r == NT && i == 0)) {
        mbase[r * M.T + i] = group_first<&MergeTerm::tile_run>(M, r, i);
        gebase[r * M.T + i] = group_first<&MergeTerm::tile_ptr>(M, r, i);
    }
    if (r >= m.n) return;
    const int t = m.run_t[r];
    const int q = group_first<&MergeTerm::tile_run>(M, t, i) + (r - m.tile_run[t]);
    const int b = m.run_beg[r], len = m.run_beg[r + 1] - b;
    rv[q] = m.vbase + m.run_v[r];
    rb[q] = group_first<&MergeTerm::tile_ptr>(M, t, i) + (b - m.tile_ptr[t]);
    rl[q] = len;
    rg[q] = t * M.T + i;
    ns[q] = (len - 1) / C + 1;
    id[q] = q;
}

// Heads of a run of k segments from position o of its group (per segments a wave; 0: each
// segment is one).
__device__ __forceinline__ int run_heads(int o, int k, int per) {
    return per ? (o + k - 1) / per - o / per + 1 : k;
}

// Thread i < R: heads and segments of the i-th run in vertex order; thread R + g: padded
// segments of group g.
__global__ void k_run_counts(const int* __restrict__ si, int R, const int* __restrict__ rg,
                             const int* __restrict__ mbase, const int* __restrict__ S, int G, int per,
                             int2* __restrict__ h, int* __restrict__ n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < R) {
        const int m = si[i], k = S[m + 1] - S[m];
        h[i] = make_int2(run_heads(S[m] - S[mbase[rg[m]]], k, per), k);
    } else if (i - R < G) {
        const int g = i - R, k = S[mbase[g + 1]] - S[mbase[g]];
        n[g] = per ? (k + per - 1) / per * per : k;
    }
}

// First run in vertex order of every vertex: the first run of a vertex fills it in for its
// vertex and for the ones without runs before it, thread R for those behind the last
// run's and for V.
__global__ void k_vertex_runs(const int* __restrict__ sv, int R, int V, int* __restrict__ vrun) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i > R) return;
    const int last = i < R ? sv[i] : V;
    for (int v = i ? sv[i - 1] + 1 : 0; v <= last; v++) vrun[v] = i;
}

struct PlusInt2 {
    __host__ __device__ int2 operator()(const int2& a, const int2& b) const { return make_int2(a.x + b.x, a.y + b.y); }
};

// What a vertex contributes to the lists.
struct PlusCounts {
    __host__ __device__ SegCounts operator()(const SegCounts& a, const SegCounts& b) const {
        return SegCounts{a.partial + b.partial, a.light + b.light, a.heavy + b.heavy, a.empty + b.empty,
                         a.pieces + b.pieces};
    }
};
__global__ void k_vertex_counts(const int* __restrict__ vrun, const int2* __restrict__ H, int V, int split,
                                SegCounts* __restrict__ vc) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v > V) return;
    const int n = v < V ? H[vrun[v + 1]].x - H[vrun[v]].x : 1;  // (one past the last: adds nothing)
    SegCounts c{0, 0, 0, 0, 0};
    c.partial = n > 1 ? n : 0;
    c.light = n > 1 && n <= split;
    c.heavy = n > split;
    c.empty = n == 0;
    c.pieces = c.heavy ? (n + kCombineSplit - 1) / kCombineSplit : 0;
    vc[v] = c;
}

// out[0] = the totals, out[1].partial = the segments of all groups.
__global__ void k_totals(const SegCounts* __restrict__ vs, int V, const int* __restrict__ gseg, int G,
                         SegCounts* __restrict__ out) {
    out[0] = vs[V];
    out[1] = SegCounts{gseg[G], 0, 0, 0, 0};
}

// What the emission reads and writes.
struct Emit {
    const int *sv, *si, *rb, *rl, *rg, *mbase, *S, *gseg, *gebase, *vrun;
    const int2* H;
    const SegCounts* vs;
    int R, V, G, E, C, per, perc, split, row0, row2, n_group, tail, nch, light, light_pad;
    Chunk* ch;
    Combine *cb, *cb2;
};

// kRunLanes threads per run: its segments.  (One thread per run waited for the runs of
// hundreds of segments that flat image regions have: 25 us at 512x512, now 5.6.)
constexpr int kRunLanes = 8;
__device__ __forceinline__ void emit_run(const Emit& A, size_t t) {
    const int i = (int)(t / kRunLanes);
    const int v = A.sv[i], m = A.si[i], g = A.rg[m];
    const int o = A.S[m] - A.S[A.mbase[g]], k = A.S[m + 1] - A.S[m];
    const int beg = A.rb[m], len = A.rl[m];
    const int h0 = A.H[A.vrun[v]].x, per = A.per;
    const bool direct = A.H[A.vrun[v + 1]].x - h0 == 1;
    const int row = A.row0 + A.vs[v].partial + (A.H[i].x - h0);
    Chunk* out = A.ch + A.gseg[g] + o;
    for (int j = (int)(t % kRunLanes); j < k; j += kRunLanes) {
        const bool head = !per || j == 0 || (o + j) % per == 0;
        const int before = per ? (o + j) / per - o / per : j;  // heads before a head
        const int b = beg + j * A.C;
        out[j] = Chunk{v, b, b + min(A.C, len - j * A.C), head ? (direct ? v : row + before) : -1};
    }
}

// One thread per vertex: its empty segment, or its recombination item(s).  perc: lane
// groups a wave of the recombination (0: two levels, row2 the first second-level row).
__device__ __forceinline__ void emit_vertex(const Emit& A, int v) {
    const int n = A.H[A.vrun[v + 1]].x - A.H[A.vrun[v]].x;
    const SegCounts c = A.vs[v];
    const int first = A.row0 + c.partial;
    if (n == 0) {
        A.ch[A.n_group + c.empty] = Chunk{v, A.E, A.E, v};
    } else if (n > 1 && n <= A.split) {
        A.cb[c.light] = Combine{v, first, n, 0};
    } else if (n > A.split && A.perc) {  // a whole wave: up to perc pieces side by side
        const int pieces = min(A.perc, (n + kCombineSplit - 1) / kCombineSplit);
        for (int j = 0, off = 0; j < A.perc; j++) {
            const int q = j < pieces ? (n - off) / (pieces - j) : 0;
            A.cb[A.light_pad + c.heavy * A.perc + j] = Combine{v, first + off, q, pieces};
            off += q;
        }
    } else if (n > A.split) {
        const int pieces = (n + kCombineSplit - 1) / kCombineSplit;
        for (int j = 0, off = 0; j < pieces; j++) {
            const int q = (n - off) / (pieces - j);
            A.cb[A.light_pad + c.pieces + j] = Combine{A.row2 + c.pieces + j, first + off, q, 0};
            off += q;
        }
        A.cb2[c.heavy] = Combine{v, A.row2 + c.pieces, pieces, 0};
    }
}

// Fillers: g < G those of group g; G the segments after the empty ones and the light
// items' padding.
__device__ __forceinline__ void emit_fillers(const Emit& A, int g) {
    if (g == A.G) {
        for (int i = A.tail; i < A.nch; i++) A.ch[i] = Chunk{-1, A.E, A.E, -1};
        for (int i = A.light; i < A.light_pad; i++) A.cb[i] = Combine{0, 0, 0, 0};
        return;
    }
    const int e = A.gebase[g + 1];
    for (int i = A.gseg[g] + A.S[A.mbase[g + 1]] - A.S[A.mbase[g]]; i < A.gseg[g + 1]; i++)
        A.ch[i] = Chunk{-1, e, e, -1};
}

// All of it in one launch: threads for the runs, then the vertices, then the groups.
__global__ void k_emit(Emit A) {
    size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t runs = (size_t)A.R * kRunLanes;
    if (t < runs) return emit_run(A, t);
    t -= runs;
    if (t < (size_t)A.V) return emit_vertex(A, (int)t);
    t -= A.V;
    if (t <= (size_t)A.G) emit_fillers(A, (int)t);
}

// The all-ones input splatted to rows of one float, each vertex's segments one after another:
// the sums of a sequential list, without its lists and entries.  Segments in vertex order
// (H[].y), a quad per segment: its lanes load every fourth weight and add all of them in
// entry order (quad_value), like the splat of few labels.
// Bound: the random reads of the weights, in vertex order (52 us at 1024x768, 8 at 512x512;
// the entries in tile order and a list splat: 2 x 24 + 19 us).  One range of segments per XCD
// took 62 us: the terms' vertices differ in entries, so the ranges differ in work.
struct OnesTerms {
    int T;
    struct {
        const int *csr_e, *tile_ptr;
        const float* bary;
    } t[DCRF_MAX_TERMS];
};
__global__ void k_ones_segments(OnesTerms O, const int* __restrict__ si, const int* __restrict__ rb,
                                const int* __restrict__ rl, const int* __restrict__ rg,
                                const int* __restrict__ gebase, const int2* __restrict__ H, int R, int C,
                                float* __restrict__ part) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int kk = (int)(t & 3);
    const bool on = t / 4 < (size_t)H[R].y;  // the same in the quad's lanes
    const int q = on ? (int)(t / 4) : 0;
    int lo = 0, hi = R - 1;  // the run of segment q
    while (lo < hi) {
        const int mid = (int)(((unsigned)lo + hi + 1) >> 1);
        if (H[mid].y <= q)
            lo = mid;
        else
            hi = mid - 1;
    }
    const int m = si[lo], g = rg[m], at = (q - H[lo].y) * C;
    const int i = g % O.T;
    const int beg = rb[m] + at - gebase[g] + O.t[i].tile_ptr[g / O.T];  // in the term's order
    const int len = on ? min(C, rl[m] - at) : 0;
    const int* __restrict__ csr = O.t[i].csr_e + beg;
    const float* __restrict__ bary = O.t[i].bary;
    float acc = 0.0f;
    constexpr int kBatch = 8;
    for (int o = 0; o < len; o += 4 * kBatch) {
        float w[kBatch];
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
            const int j = o + kk + 4 * u;
            const float b = bary[csr[min(j, len - 1)]];
            w[u] = j < len ? b : 0.0f;
        }
#pragma unroll
        for (int u = 0; u < kBatch; u++) {
            acc = acc + quad_value<0>(w[u]);
            acc = acc + quad_value<1>(w[u]);
            acc = acc + quad_value<2>(w[u]);
            acc = acc + quad_value<3>(w[u]);
        }
    }
    if (on && kk == 0) part[q] = acc;
}

// The vertices' rows from their segments' (v0), and the zero row V of both buffers.
__global__ void k_ones_vertices(const float* __restrict__ part, const int* __restrict__ vrun,
                                const int2* __restrict__ H, int V, float* __restrict__ v0, float* __restrict__ v1) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v > V) return;
    float acc = 0.0f;
    if (v < V) {
        int i = H[vrun[v]].y;
        const int e = H[vrun[v + 1]].y;
        constexpr int kBatch = 16;  // loads in flight for vertices of hundreds of segments
        for (; i + kBatch <= e; i += kBatch) {
            float x[kBatch];
#pragma unroll
            for (int u = 0; u < kBatch; u++) x[u] = part[i + u];
#pragma unroll
            for (int u = 0; u < kBatch; u++) acc = acc + x[u];
        }
        for (; i < e; i++) acc = acc + part[i];
    } else {
        v1[v] = 0.0f;
    }
    v0[v] = acc;
}

// out[0 .. n] = exclusive scan of in[0 .. n) and the total (in has n + 1 readable entries,
// in[n] = anything).
template <typename T, typename Op>
void scan(const T* in, T* out, T zero, size_t n, Op op, hipStream_t s) {
    size_t tb = 0;
    DCRF_HIP_CHECK(rocprim::exclusive_scan(nullptr, tb, in, out, zero, n + 1, op, s));
    DevBuf<char> tmp;
    tmp.reserve(tb);
    DCRF_HIP_CHECK(rocprim::exclusive_scan(tmp.get(), tb, in, out, zero, n + 1, op, s));
}

}  // namespace

void build_run_set(const std::vector<const TermLattice*>& lats, const std::vector<int>& vbase, int n_tiles, int C,
                   RunSet& rs, hipStream_t s) {
    const int T = (int)lats.size();
    rs.T = T;
    rs.NT = n_tiles;
    rs.C = C;
    const int G = rs.G = n_tiles * T;
    long long R = 0, E = 0, V = 0;
    int most = n_tiles + 1;
    MergeTerms M{};
    M.T = T;
    for (int i = 0; i < T; i++) {
        const TermLattice& l = *lats[i];
        R += l.n_runs;
        E += l.n_entries;
        V += l.V;
        most = std::max(most, l.n_runs);
        M.t[i] = MergeTerm{l.run_v.get(), l.run_t.get(), l.run_beg.get(), l.tile_run.get(), l.tile_ptr.get(),
                           l.n_runs, vbase[i]};
    }
    if (E > 0x7ffffff0ll || R > 0x7ffffff0ll || V > 0x7ffffff0ll)
        throw Error{DCRF_ERR_VALUE, "splat layout too large"};
    rs.R = (int)R;
    rs.E = (int)E;
    rs.V = (int)V;
    if (!T) return;
    DevBuf<int> ns, id;
    rs.mbase.reserve(G + 1);
    rs.gebase.reserve(G + 1);
    for (DevBuf<int>* b : {&rs.rv, &rs.rb, &rs.rl, &rs.rg, &rs.sv, &rs.si, &id}) b->reserve(R);
    ns.reserve(R + 1);
    rs.S.reserve(R + 1);
    rs.vrun.reserve(V + 1);
    k_merge_runs<<<dim3(blocks_for(most), T), kThreads, 0, s>>>(M, n_tiles, C, rs.mbase.get(), rs.gebase.get(),
                                                                rs.rv.get(), rs.rb.get(), rs.rl.get(), rs.rg.get(),
                                                                ns.get(), id.get());
    DCRF_HIP_CHECK(hipGetLastError());
    scan(ns.get(), rs.S.get(), 0, R, rocprim::plus<int>(), s);
    int vbits = 1;
    while (vbits < 31 && (1ll << vbits) <= V) vbits++;
    if (R) {
        size_t tb = 0;
        DCRF_HIP_CHECK(rocprim::radix_sort_pairs(nullptr, tb, reinterpret_cast<unsigned*>(rs.rv.get()),
                                                 reinterpret_cast<unsigned*>(rs.sv.get()), id.get(), rs.si.get(),
                                                 (size_t)R, 0, vbits, s));
        DevBuf<char> tmp;
        tmp.reserve(tb);
        DCRF_HIP_CHECK(rocprim::radix_sort_pairs(tmp.get(), tb, reinterpret_cast<unsigned*>(rs.rv.get()),
                                                 reinterpret_cast<unsigned*>(rs.sv.get()), id.get(), rs.si.get(),
                                                 (size_t)R, 0, vbits, s));
    }
    k_vertex_runs<<<blocks_for((size_t)R + 1), kThreads, 0, s>>>(rs.sv.get(), rs.R, rs.V, rs.vrun.get());
    DCRF_HIP_CHECK(hipGetLastError());
}

void count_segments(const RunSet& rs, int per, int perc, bool sequential, SegPlan& P, hipStream_t s) {
    P.per = per;
    P.perc = perc;
    P.split = sequential ? std::numeric_limits<int>::max() : kCombineSplit;
    DevBuf<int> n;
    DevBuf<int2> h;
    DevBuf<SegCounts> vc, tot;
    n.reserve(rs.G + 1);
    P.gseg.reserve(rs.G + 1);
    h.reserve(rs.R + 1);
    P.H.reserve(rs.R + 1);
    if ((size_t)rs.R + rs.G) {
        k_run_counts<<<blocks_for((size_t)rs.R + rs.G), kThreads, 0, s>>>(rs.si.get(), rs.R, rs.rg.get(),
                                                                          rs.mbase.get(), rs.S.get(), rs.G, per,
                                                                          h.get(), n.get());
        DCRF_HIP_CHECK(hipGetLastError());
    }
    scan(n.get(), P.gseg.get(), 0, rs.G, rocprim::plus<int>(), s);
    scan(h.get(), P.H.get(), make_int2(0, 0), rs.R, PlusInt2(), s);
    vc.reserve(rs.V + 1);
    P.vs.reserve(rs.V + 1);
    k_vertex_counts<<<blocks_for((size_t)rs.V + 1), kThreads, 0, s>>>(rs.vrun.get(), P.H.get(), rs.V, P.split,
                                                                      vc.get());
    DCRF_HIP_CHECK(hipGetLastError());
    scan(vc.get(), P.vs.get(), SegCounts{0, 0, 0, 0, 0}, rs.V, PlusCounts(), s);
    tot.reserve(2);
    k_totals<<<1, 1, 0, s>>>(P.vs.get(), rs.V, P.gseg.get(), rs.G, tot.get());
    DCRF_HIP_CHECK(hipGetLastError());
    DCRF_HIP_CHECK(hipMemcpyAsync(P.host, tot.get(), sizeof(P.host), hipMemcpyDeviceToHost, s));
}

void emit_segments(const RunSet& rs, const SegPlan& P, int row0, SegLists& L, hipStream_t s) {
    const SegCounts& c = P.host[0];
    const int n_group = P.host[1].partial, tail = n_group + c.empty;
    L.waves = P.perc > 0;
    L.nch = P.per ? (tail + P.per - 1) / P.per * P.per : tail;
    const int light_pad = L.waves && c.heavy ? (c.light + P.perc - 1) / P.perc * P.perc : c.light;
    L.ncb = L.waves ? light_pad + c.heavy * P.perc : c.light + c.pieces;
    L.ncb2 = L.waves ? 0 : c.heavy;
    const int row2 = row0 + c.partial;
    L.rows = row2 + (L.waves ? 0 : c.pieces);
    L.ch.reserve(L.nch);
    L.cb.reserve(L.ncb);
    L.cb2.reserve(L.ncb2);
    const Emit A{rs.sv.get(), rs.si.get(), rs.rb.get(), rs.rl.get(), rs.rg.get(), rs.mbase.get(), rs.S.get(),
                 P.gseg.get(), rs.gebase.get(), rs.vrun.get(), P.H.get(), P.vs.get(), rs.R, rs.V, rs.G, rs.E, rs.C,
                 P.per, P.perc, P.split, row0, row2, n_group, tail, L.nch, c.light, light_pad, L.ch.get(),
                 L.cb.get(), L.cb2.get()};
    k_emit<<<blocks_for((size_t)rs.R * kRunLanes + rs.V + rs.G + 1), kThreads, 0, s>>>(A);
    DCRF_HIP_CHECK(hipGetLastError());
}

void splat_ones(const std::vector<const TermLattice*>& lats, const RunSet& rs, const SegPlan& P, float* v0, float* v1,
                hipStream_t s) {
    OnesTerms O{};
    O.T = rs.T;
    for (int i = 0; i < rs.T; i++) {
        O.t[i].csr_e = lats[i]->csr_e.get();
        O.t[i].tile_ptr = lats[i]->tile_ptr.get();
        O.t[i].bary = lats[i]->bary.get();
    }
    DevBuf<float> part;
    const size_t segs = (size_t)rs.R + rs.E / rs.C;  // a run's last segment may be short
    part.reserve(segs);
    if (rs.R) {
        k_ones_segments<<<blocks_for(4 * segs), kThreads, 0, s>>>(O, rs.si.get(), rs.rb.get(), rs.rl.get(),
                                                                  rs.rg.get(), rs.gebase.get(), P.H.get(), rs.R, rs.C,
                                                                  part.get());
        DCRF_HIP_CHECK(hipGetLastError());
    }
    k_ones_vertices<<<blocks_for((size_t)rs.V + 1), kThreads, 0, s>>>(part.get(), rs.vrun.get(), P.H.get(), rs.V, v0,
                                                                      v1);
    DCRF_HIP_CHECK(hipGetLastError());
}

}  // namespace dcrf
