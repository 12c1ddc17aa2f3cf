// The fused adjoint step over interleaved slice pairs (see adjoint.hip for the recursion).
#include "dcrf_fused.h"

#pragma clang fp contract(off)

namespace dcrf {
namespace {

inline unsigned blocks_for(size_t n, int t) { return (unsigned)((n + t - 1) / t); }

// The adjoint step of k_adjoint (adjoint.hip) over the same interleaved slice pairs:
// g = sum_k C_k(w_k slice_k(filtered b)), b = sumAndNormalize(Q .* g, Q), dU (UnarySum) and
// the terms' statistic rows (SliceTerm::gstat).  The pairs carry the transposed filter's
// slice weights.  Same arithmetic, in the same order, as k_adjoint.
template <int R, int D0, int D1, bool CWL, bool NARROW>
__global__ void __launch_bounds__(kWaveBlock) __attribute__((amdgpu_waves_per_eu(R <= 3 ? 8 : 7)))
k_adjoint_fused(const float* __restrict__ Q, float* __restrict__ b, float* __restrict__ dU, UnarySum us, int N, int L, int Lv,
                int S, int per, SliceTable st, const int2* __restrict__ slc, int cwf) {
    constexpr int DS = D0 + D1;
    LaneGroup<true, R> G(L, S, per, nullptr);
    const int p = G.item();
    const bool active = G.on && p < N;
    const int k0 = G.k0;
    const WavePixels W(G, p, N);
    const int gp = min(G.g, W.np - 1);
    extern __shared__ __align__(16) int2 pairs_all[];
    const int wpairs = wave_pairs(per, DS);
    int2* wp = pairs_all + G.w * wpairs;
    float* shc = reinterpret_cast<float*>(pairs_all + (kWaveBlock / 64) * wpairs);
    const size_t wrow = (size_t)W.p0 * Lv;           // the wave's rows of Q and b
    const unsigned grow = (unsigned)(gp * Lv + k0);  // the lane's piece of them
    float q[R];
    load_piece<R>(Q + wrow + grow, 0, L, q);  // in flight while the pairs are staged
    if (CWL) stage_compat(st, L, shc);
    stage_wave_pairs<R, DS>(W, per, slc, wp);
    int2 e[DS];
#pragma unroll
    for (int j = 0; j < DS; j++) e[j] = wp[gp * DS + j];
    float x[DS][R];
#pragma unroll
    for (int j = 0; j < DS; j++) {
        const SliceTerm& T = j < D0 ? st.t[0] : st.t[1];
        load_piece<R>(row_piece<NARROW>(T.vals, e[j].x, T.ldv, k0), 0, L, x[j]);
    }
    constexpr int NT = D1 ? 2 : 1;
    float raw[NT][R], mk[NT][R], c[NT][R];  // (the adjoint stores no raw messages)
#pragma unroll
    for (int k = 0; k < NT; k++) term_message<R, D0, D1>(st.t[k], k, e, x, raw[k], mk[k]);
    // statistic region after the message rows (present with a compat region)
    float* sst = shc + cwf + (cwf ? (kWaveBlock / 64) * NT * per * ((L + 3) & ~3) : 0);
#pragma unroll
    for (int k = 0; k < NT; k++)
        if (st.t[k].gslot >= 0) {
            float v[R];
#pragma unroll
            for (int r = 0; r < R; r++) v[r] = active ? raw[k][r] * q[r] : 0.0f;
            stat_put<R>(sst, st.t[k].gslot, v);
        }
    float* msg = shc + cwf + (size_t)G.w * NT * per * ((L + 3) & ~3);
    compat_terms<R, NT, CWL>(G, st, mk, c, shc, msg);
    float gsum[R];
#pragma unroll
    for (int r = 0; r < R; r++) gsum[r] = 0.0f;
#pragma unroll
    for (int k = 0; k < NT; k++)
#pragma unroll
        for (int r = 0; r < R; r++) gsum[r] = gsum[r] + c[k][r];
    float bn[R];
    sum_normalize<true, R>(q, gsum, bn, G);
    if (active) {
        store_piece<R>(b + wrow + grow, 0, L, bn);
        add_unary(us, wrow + grow, dU + (size_t)W.p0 * L + (unsigned)(gp * L), G, bn);
    }
    if (st.nstat) stat_finish<true, R, NT>(st, G, sst);  // uniform condition
}

}  // namespace

#define DCRF_ADJ_FUSED(R_, D0_, D1_)                                                                      \
    DCRF_FUSED_FORM(k_adjoint_fused, R_, D0_, D1_)<<<                                                       \
        blocks_for(N, sh.items), kWaveBlock, fused_lds_bytes(sh, D0_ + D1_, D1_ ? 2 : 1, L, cwf, st.nstat),  \
        s>>>(Q, b, dU, us, N, L, Lv, sh.S, sh.per, st, slc, cwf)

template <int R>
void launch_adj_fused_r(const LaunchShape& sh, const float* Q, float* b, float* dU, const UnarySum& us, int N, int L, int Lv,
                        const SliceTable& st, const int2* slc, int cwf, hipStream_t s) {
    const int a = st.t[0].d1, c = st.nterms > 1 ? st.t[1].d1 : 0;
    const bool narrow = narrow_rows(st.rows, st.t[0].ldv);
    if (a == 3 && c == 0) DCRF_ADJ_FUSED(R, 3, 0);
    else if (a == 6 && c == 0) DCRF_ADJ_FUSED(R, 6, 0);
    else if (a == 3 && c == 6) DCRF_ADJ_FUSED(R, 3, 6);
    else if (a == 6 && c == 3) DCRF_ADJ_FUSED(R, 6, 3);
    else if (a == 4 && c == 5) DCRF_ADJ_FUSED(R, 4, 5);
    else if (a == 5 && c == 4) DCRF_ADJ_FUSED(R, 5, 4);
    else throw Error{DCRF_ERR_VALUE, "no fused adjoint kernel for these terms"};
    DCRF_HIP_CHECK(hipGetLastError());
}
#undef DCRF_ADJ_FUSED
void launch_adjoint_fused(const float* Q, float* b, float* dU, const UnarySum& us, int N, int L, int Lv, const SliceTable& st_in,
                          const int2* slc, hipStream_t s) {
    SliceTable st = st_in;
    const int cwf = assign_compat_lds(st, L, true);  // 16-byte rows for matrix_piece_rows
    const LaunchShape sh = shape_for(Lv);
    if (!fused_meanfield_ok(L, st.nterms, st.t[0].d1, st.nterms > 1 ? st.t[1].d1 : 0))
        throw Error{DCRF_ERR_VALUE, "no fused adjoint kernel for these terms"};
    switch (sh.R) {
        case 1: launch_adj_fused_r<1>(sh, Q, b, dU, us, N, L, Lv, st, slc, cwf, s); break;
        case 2: launch_adj_fused_r<2>(sh, Q, b, dU, us, N, L, Lv, st, slc, cwf, s); break;
        case 3: launch_adj_fused_r<3>(sh, Q, b, dU, us, N, L, Lv, st, slc, cwf, s); break;
        default: launch_adj_fused_r<4>(sh, Q, b, dU, us, N, L, Lv, st, slc, cwf, s); break;
    }
}

}  // namespace dcrf
