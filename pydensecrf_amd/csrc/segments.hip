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
// scan or one thread per run, vertex or group; the host reads one set of counts to size
// the lists.  The order of a vertex's partial rows is that of the stable sort by vertex,
// i.e. list order, so the sums do not depend on anything but the runs.
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

// Group sizes of term i (of T): runs and entries per tile.
__global__ void k_group_counts(const int* __restrict__ tile_run, const int* __restrict__ tile_ptr, int NT, int T, int i,
                               int* __restrict__ runs, int* __restrict__ entries) {
    const int t = blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= NT) return;
    runs[t * T + i] = tile_run[t + 1] - tile_run[t];
    entries[t * T + i] = tile_ptr[t + 1] - tile_ptr[t];
}

// The runs of term i into the merged order: vertex (from vbase), first entry, entries, group.
__global__ void k_merge_runs(const int* __restrict__ run_v, const int* __restrict__ run_t,
                             const int* __restrict__ run_beg, int n, const int* __restrict__ tile_run,
                             const int* __restrict__ tile_ptr, int T, int i, int vbase, const int* __restrict__ mbase,
                             const int* __restrict__ gebase, int C, int* __restrict__ rv, int* __restrict__ rb,
                             int* __restrict__ rl, int* __restrict__ rg, int* __restrict__ ns, int* __restrict__ id) {
    const int r = blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= n) return;
    const int t = run_t[r], g = t * T + i;
    const int m = mbase[g] + (r - tile_run[t]);
    const int b = run_beg[r], len = run_beg[r + 1] - b;
    rv[m] = vbase + run_v[r];
    rb[m] = gebase[g] + (b - tile_ptr[t]);
    rl[m] = len;
    rg[m] = g;
    ns[m] = (len - 1) / C + 1;
    id[m] = m;
}

// Heads of a run of k segments from position o of its group (per segments a wave; 0: each
// segment is one).
__device__ __forceinline__ int run_heads(int o, int k, int per) {
    return per ? (o + k - 1) / per - o / per + 1 : k;
}

// Padded segment count of every group.
__global__ void k_group_segments(const int* __restrict__ mbase, const int* __restrict__ S, int G, int per,
                                 int* __restrict__ n) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= G) return;
    const int k = S[mbase[g + 1]] - S[mbase[g]];
    n[g] = per ? (k + per - 1) / per * per : k;
}

// Heads of every run in vertex order.
__global__ void k_heads(const int* __restrict__ si, int R, const int* __restrict__ rg, const int* __restrict__ mbase,
                        const int* __restrict__ S, int per, int* __restrict__ h) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= R) return;
    const int m = si[i];
    h[i] = run_heads(S[m] - S[mbase[rg[m]]], S[m + 1] - S[m], per);
}

// Heads before every vertex: the first run of a vertex fills it in for its vertex and for
// the ones without runs before it, thread R for those behind the last run's and for V.
__global__ void k_vertex_first(const int* __restrict__ sv, const int* __restrict__ H, int R, int V,
                               int* __restrict__ vfirst) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i > R) return;
    const int last = i < R ? sv[i] : V, h = R ? H[i] : 0;
    for (int v = i ? sv[i - 1] + 1 : 0; v <= last; v++) vfirst[v] = h;
}

// What a vertex contributes to the lists.
struct PlusCounts {
    __host__ __device__ SegCounts operator()(const SegCounts& a, const SegCounts& b) const {
        return SegCounts{a.partial + b.partial, a.light + b.light, a.heavy + b.heavy, a.empty + b.empty,
                         a.pieces + b.pieces};
    }
};
__global__ void k_vertex_counts(const int* __restrict__ vfirst, int V, int split, SegCounts* __restrict__ vc) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v > V) return;
    const int n = v < V ? vfirst[v + 1] - vfirst[v] : 1;  // (one past the last: adds nothing)
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

// kRunLanes threads per run: its segments.  (One thread per run waited for the runs of
// hundreds of segments that flat image regions have: 25 us at 512x512, now 5.6.)
constexpr int kRunLanes = 8;
__global__ void k_emit_runs(const int* __restrict__ sv, const int* __restrict__ si, int R, const int* __restrict__ rb,
                            const int* __restrict__ rl, const int* __restrict__ rg, const int* __restrict__ mbase,
                            const int* __restrict__ S, const int* __restrict__ gseg, const int* __restrict__ H,
                            const int* __restrict__ vfirst, const SegCounts* __restrict__ vs, int C, int per, int row0,
                            Chunk* __restrict__ ch) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const int i = (int)(t / kRunLanes);
    if (i >= R) return;
    const int v = sv[i], m = si[i], g = rg[m];
    const int o = S[m] - S[mbase[g]], k = S[m + 1] - S[m];
    const int beg = rb[m], end = beg + rl[m];
    const bool direct = vfirst[v + 1] - vfirst[v] == 1;
    const int row = row0 + vs[v].partial + (H[i] - vfirst[v]);
    Chunk* out = ch + gseg[g] + o;
    for (int j = (int)(t % kRunLanes); j < k; j += kRunLanes) {
        const bool head = !per || j == 0 || (o + j) % per == 0;
        const int before = per ? (o + j) / per - o / per : j;  // heads before a head
        out[j] = Chunk{v, beg + j * C, min(end, beg + (j + 1) * C), head ? (direct ? v : row + before) : -1};
    }
}

// One thread per vertex: its empty segment, or its recombination item(s).  perc: lane
// groups a wave of the recombination (0: two levels, row2 the first second-level row).
__global__ void k_emit_vertices(const int* __restrict__ vfirst, const SegCounts* __restrict__ vs, int V, int E,
                                int n_group_segs, int row0, int perc, int split, int light_pad,
                                int row2,
                                Chunk* __restrict__ ch, Combine* __restrict__ cb, Combine* __restrict__ cb2) {
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v >= V) return;
    const int n = vfirst[v + 1] - vfirst[v];
    const SegCounts c = vs[v];
    const int first = row0 + c.partial;
    if (n == 0) {
        ch[n_group_segs + c.empty] = Chunk{v, E, E, v};
    } else if (n > 1 && n <= split) {
        cb[c.light] = Combine{v, first, n, 0};
    } else if (n > split && perc) {  // a whole wave: up to perc pieces side by side
        const int pieces = min(perc, (n + kCombineSplit - 1) / kCombineSplit);
        for (int j = 0, off = 0; j < perc; j++) {
            const int q = j < pieces ? (n - off) / (pieces - j) : 0;
            cb[light_pad + c.heavy * perc + j] = Combine{v, first + off, q, pieces};
            off += q;
        }
    } else if (n > split) {
        const int pieces = (n + kCombineSplit - 1) / kCombineSplit;
        for (int j = 0, off = 0; j < pieces; j++) {
            const int q = (n - off) / (pieces - j);
            cb[light_pad + c.pieces + j] = Combine{row2 + c.pieces + j, first + off, q, 0};
            off += q;
        }
        cb2[c.heavy] = Combine{v, row2 + c.pieces, pieces, 0};
    }
}

// Fillers: thread g < G those of group g; thread G the segments after the empty ones and
// the light items' padding.
__global__ void k_emit_fillers(const int* __restrict__ mbase, const int* __restrict__ S, const int* __restrict__ gseg,
                               const int* __restrict__ gebase, int G, int E, int tail, int n_chunks, int light,
                               int light_pad, Chunk* __restrict__ ch, Combine* __restrict__ cb) {
    const int g = blockIdx.x * blockDim.x + threadIdx.x;
    if (g > G) return;
    if (g == G) {
        for (int i = tail; i < n_chunks; i++) ch[i] = Chunk{-1, E, E, -1};
        for (int i = light; i < light_pad; i++) cb[i] = Combine{0, 0, 0, 0};
        return;
    }
    const int e = gebase[g + 1];
    for (int i = gseg[g] + S[mbase[g + 1]] - S[mbase[g]]; i < gseg[g + 1]; i++) ch[i] = Chunk{-1, e, e, -1};
}

// out[0 .. n] = exclusive scan of in[0 .. n) and the total (in has n + 1 readable entries,
// in[n] = anything).
void scan_int(const int* in, int* out, size_t n, hipStream_t s) {
    size_t tb = 0;
    DCRF_HIP_CHECK(rocprim::exclusive_scan(nullptr, tb, in, out, 0, n + 1, rocprim::plus<int>(), s));
    DevBuf<char> tmp;
    tmp.reserve(tb);
    DCRF_HIP_CHECK(rocprim::exclusive_scan(tmp.get(), tb, in, out, 0, n + 1, rocprim::plus<int>(), s));
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
    for (const TermLattice* l : lats) {
        R += l->n_runs;
        E += l->n_entries;
        V += l->V;
    }
    if (E > 0x7ffffff0ll || R > 0x7ffffff0ll || V > 0x7ffffff0ll)
        throw Error{DCRF_ERR_VALUE, "splat layout too large"};
    rs.R = (int)R;
    rs.E = (int)E;
    rs.V = (int)V;
    DevBuf<int> gr, ge, ns, id;
    gr.reserve(G + 1);
    ge.reserve(G + 1);
    rs.mbase.reserve(G + 1);
    rs.gebase.reserve(G + 1);
    for (int i = 0; i < T; i++) {
        k_group_counts<<<blocks_for(n_tiles), kThreads, 0, s>>>(lats[i]->tile_run.get(), lats[i]->tile_ptr.get(),
                                                                n_tiles, T, i, gr.get(), ge.get());
        DCRF_HIP_CHECK(hipGetLastError());
    }
    scan_int(gr.get(), rs.mbase.get(), G, s);
    scan_int(ge.get(), rs.gebase.get(), G, s);
    for (DevBuf<int>* b : {&rs.rv, &rs.rb, &rs.rl, &rs.rg, &rs.sv, &rs.si, &id}) b->reserve(R);
    ns.reserve(R + 1);
    rs.S.reserve(R + 1);
    for (int i = 0; i < T; i++) {
        const TermLattice& l = *lats[i];
        if (!l.n_runs) continue;
        k_merge_runs<<<blocks_for(l.n_runs), kThreads, 0, s>>>(
            l.run_v.get(), l.run_t.get(), l.run_beg.get(), l.n_runs, l.tile_run.get(), l.tile_ptr.get(), T, i, vbase[i],
            rs.mbase.get(), rs.gebase.get(), C, rs.rv.get(), rs.rb.get(), rs.rl.get(), rs.rg.get(), ns.get(), id.get());
        DCRF_HIP_CHECK(hipGetLastError());
    }
    scan_int(ns.get(), rs.S.get(), R, s);
    if (!R) return;
    int vbits = 1;
    while (vbits < 31 && (1ll << vbits) <= V) vbits++;
    size_t tb = 0;
    DCRF_HIP_CHECK(rocprim::radix_sort_pairs(nullptr, tb, reinterpret_cast<unsigned*>(rs.rv.get()),
                                             reinterpret_cast<unsigned*>(rs.sv.get()), id.get(), rs.si.get(), (size_t)R,
                                             0, vbits, s));
    DevBuf<char> tmp;
    tmp.reserve(tb);
    DCRF_HIP_CHECK(rocprim::radix_sort_pairs(tmp.get(), tb, reinterpret_cast<unsigned*>(rs.rv.get()),
                                             reinterpret_cast<unsigned*>(rs.sv.get()), id.get(), rs.si.get(), (size_t)R,
                                             0, vbits, s));
}

void count_segments(const RunSet& rs, int per, int perc, bool sequential, SegPlan& P, hipStream_t s) {
    P.per = per;
    P.perc = perc;
    P.split = sequential ? std::numeric_limits<int>::max() : kCombineSplit;
    DevBuf<int> n, h;
    DevBuf<SegCounts> vc, tot;
    n.reserve(rs.G + 1);
    P.gseg.reserve(rs.G + 1);
    if (rs.G) {
        k_group_segments<<<blocks_for(rs.G), kThreads, 0, s>>>(rs.mbase.get(), rs.S.get(), rs.G, per, n.get());
        DCRF_HIP_CHECK(hipGetLastError());
    }
    scan_int(n.get(), P.gseg.get(), rs.G, s);
    P.vfirst.reserve(rs.V + 1);
    h.reserve(rs.R + 1);
    P.H.reserve(rs.R + 1);
    if (rs.R) {
        k_heads<<<blocks_for(rs.R), kThreads, 0, s>>>(rs.si.get(), rs.R, rs.rg.get(), rs.mbase.get(), rs.S.get(),
                                                      per, h.get());
        DCRF_HIP_CHECK(hipGetLastError());
    }
    scan_int(h.get(), P.H.get(), rs.R, s);
    k_vertex_first<<<blocks_for((size_t)rs.R + 1), kThreads, 0, s>>>(rs.sv.get(), P.H.get(), rs.R, rs.V,
                                                                     P.vfirst.get());
    DCRF_HIP_CHECK(hipGetLastError());
    vc.reserve(rs.V + 1);
    P.vs.reserve(rs.V + 1);
    k_vertex_counts<<<blocks_for((size_t)rs.V + 1), kThreads, 0, s>>>(P.vfirst.get(), rs.V, P.split, vc.get());
    DCRF_HIP_CHECK(hipGetLastError());
    const SegCounts zero{0, 0, 0, 0, 0};
    size_t tb = 0;
    DCRF_HIP_CHECK(rocprim::exclusive_scan(nullptr, tb, vc.get(), P.vs.get(), zero, (size_t)rs.V + 1, PlusCounts(), s));
    DevBuf<char> tmp;
    tmp.reserve(tb);
    DCRF_HIP_CHECK(rocprim::exclusive_scan(tmp.get(), tb, vc.get(), P.vs.get(), zero, (size_t)rs.V + 1, PlusCounts(), s));
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
    if (rs.R) {
        k_emit_runs<<<blocks_for((size_t)rs.R * kRunLanes), kThreads, 0, s>>>(rs.sv.get(), rs.si.get(), rs.R, rs.rb.get(), rs.rl.get(),
                                                          rs.rg.get(), rs.mbase.get(), rs.S.get(), P.gseg.get(),
                                                          P.H.get(), P.vfirst.get(), P.vs.get(), rs.C,
                                                          P.per, row0, L.ch.get());
        DCRF_HIP_CHECK(hipGetLastError());
    }
    if (rs.V) {
        k_emit_vertices<<<blocks_for(rs.V), kThreads, 0, s>>>(P.vfirst.get(), P.vs.get(), rs.V, rs.E, n_group, row0,
                                                              P.perc, P.split, light_pad, row2, L.ch.get(), L.cb.get(),
                                                              L.cb2.get());
        DCRF_HIP_CHECK(hipGetLastError());
    }
    k_emit_fillers<<<blocks_for((size_t)rs.G + 1), kThreads, 0, s>>>(rs.mbase.get(), rs.S.get(), P.gseg.get(),
                                                                     rs.gebase.get(), rs.G, rs.E, tail, L.nch, c.light,
                                                                     light_pad, L.ch.get(), L.cb.get());
    DCRF_HIP_CHECK(hipGetLastError());
}

}  // namespace dcrf
