// The fused mean-field update (slice of every term, compatibility, softmax) over
// interleaved slice pairs, and its form over LDS-staged pixel runs.  Replaces the second
// half of the reference's iteration (densecrf.cpp:122-129, permutohedral.cpp:571-609).
#include <cmath>
#include <type_traits>

#include "dcrf_fused.h"

#pragma clang fp contract(off)

namespace dcrf {
namespace {

// blocks of t items
inline unsigned blocks_for(size_t n, int t) { return (unsigned)((n + t - 1) / t); }

// Mean-field update for models of one or two terms with d+1 = D0 (and D1) lattice
// entries per pixel: slc holds every pixel's (vertex, weight bits) pairs of both terms
// side by side, so all D0 + D1 vertex rows are gathered after one dependent load.  Same
// arithmetic, in the same order, as k_meanfield.
//   3 and 6 entries are images; 4 and 5 volumes with intensity, where the generic kernels
// took 45 us (mean-field) and 62 us (adjoint) per launch on 1.5 M voxels with 4 labels,
// and these 32 and 48.
template <int R, int D0, int D1, bool CWL, bool NARROW>
__global__ void __launch_bounds__(kWaveBlock) __attribute__((amdgpu_waves_per_eu(R <= 3 ? 8 : 7)))  // <= 64 (72) VGPRs
k_meanfield_fused(const float* __restrict__ U, float* __restrict__ Q, int ldq, int N, int L, int S, int per,
                  SliceTable st, const int2* __restrict__ slc, int cwf, int bw) {
    constexpr int DS = D0 + D1;
    LaneGroup<true, R> G(L, S, per, nullptr);
    const int p = G.item();
    const bool active = G.on && p < N;
    const int k0 = G.k0;
    const WavePixels W(G, p, N);
    const int gp = min(G.g, W.np - 1);  // groups without a pixel repeat the wave's last one
    extern __shared__ __align__(16) int2 pairs_all[];
    const int wpairs = wave_pairs(per, DS);
    int2* wp = pairs_all + G.w * wpairs;
    // CWL: some Matrix term has an LDS copy of its weights (staging costs a barrier, so
    // it is compiled in only then)
    float* shc = reinterpret_cast<float*>(pairs_all + (kWaveBlock / 64) * wpairs);
    // the unary row does not depend on the slice pairs: its load is in flight while they
    // are staged (not at four labels per lane, where the longer-lived row would spill)
    constexpr bool kEarlyU = R <= 3;
    float u[R];
    auto load_u = [&]() {
        if (U) {
            load_row(U + (size_t)W.p0 * L + (unsigned)(gp * L), G, u);
        } else {
#pragma unroll
            for (int r = 0; r < R; r++) u[r] = 0.0f;
        }
    };
    if (kEarlyU) load_u();
    if (CWL) stage_compat(st, L, shc);
    stage_wave_pairs<R, DS>(W, per, slc, wp);
    int2 e[DS];
#pragma unroll
    for (int j = 0; j < DS; j++) e[j] = wp[gp * DS + j];
    if (!kEarlyU) load_u();
    float x[DS][R];
#pragma unroll
    for (int j = 0; j < DS; j++) {
        const SliceTerm& T = j < D0 ? st.t[0] : st.t[1];
        load_piece<R>(row_piece<NARROW>(T.vals, e[j].x, T.ldv, k0), 0, L, x[j]);
    }
    // CWL: the wave's message rows follow the compat region
    float* msg = shc + cwf + (size_t)G.w * (D1 ? 2 : 1) * per * ((L + 3) & ~3);
    // bw > 0: Q is written in 8 x 8 pixel blocks of an image bw pixels wide (q_block_pos)
    float* qrow = bw > 0 ? Q + (size_t)q_block_pos(W.p0 + gp, bw) * ldq : Q + (size_t)W.p0 * ldq + (unsigned)(gp * ldq);
    finish_pixel<R, D0, D1, CWL>(G, st, e, x, u, active, qrow, ldq, shc, p, msg);
}

// The same update over pixel runs (2-D rectangles whose rows hold whole waves of
// pixels), one workgroup per run: the run's distinct vertex rows (a few hundred, against
// P*(D0+D1) gathers) are staged in LDS once, then every pixel's slice reads them from
// there (rs.loc holds the pairs with the vertex replaced by its index in the run's
// list, in run-major pixel order).
template <int R, int D0, int D1>
__global__ void __launch_bounds__(kWaveBlock) k_meanfield_runs(const float* __restrict__ U, float* __restrict__ Q,
                                                               int ldq, int N, int L, int Lv, int S, int per,
                                                               SliceTable st, RunSliceDev rs) {
    (void)N;  // the runs cover the pixels exactly (rs.pix_base)
    constexpr int DS = D0 + D1;
    extern __shared__ float lds[];
    float* tq = lds;  // rs.rows_lds floats: the run's rows
    int2* tp = reinterpret_cast<int2*>(lds + rs.rows_lds);  // rs.P * DS pairs: the run's slice pairs
    float* shc = reinterpret_cast<float*>(tp + (size_t)rs.P * DS);
    stage_compat(st, L, shc);
    LaneGroup<true, R> G(L, S, per, nullptr);
    const int k0 = G.k0;
    const int run = xcd_block(blockIdx.x, gridDim.x);
    const int k0r = rs.pix_base[run], np = rs.pix_base[run + 1] - k0r;  // run-major positions
    const int u0 = rs.base[run], nu = rs.base[run + 1] - u0;
    const int items = (blockDim.x >> 6) * per;
    const int gi = (threadIdx.x >> 6) * per + G.g;
    // stage the rows (group gi takes rows gi, gi + items, ...) and the pairs (all threads,
    // consecutive words): loads first, then stores
    for (int q0 = 0; q0 < nu; q0 += 4 * items) {
        float xs[4][R];
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const int q = min(q0 + b * items + gi, nu - 1);
            const int tag = rs.rows[u0 + q];
            load_piece<R>(((tag & 1) ? rs.v1 : rs.v0) + (size_t)(tag >> 1) * st.t[0].ldv, k0, L, xs[b]);
        }
#pragma unroll
        for (int b = 0; b < 4; b++) {
            const int q = q0 + b * items + gi;
            if (G.on && q < nu) store_piece<R>(tq + (size_t)q * Lv, k0, L, xs[b]);
        }
    }
    {
        const int npairs = np * DS;
        const int2* src = rs.loc + (size_t)k0r * DS;
        for (int i0 = 0; i0 < npairs; i0 += 4 * (int)blockDim.x) {
            int2 t[4];
#pragma unroll
            for (int b = 0; b < 4; b++) t[b] = src[min(i0 + b * (int)blockDim.x + (int)threadIdx.x, npairs - 1)];
#pragma unroll
            for (int b = 0; b < 4; b++) {
                const int i = i0 + b * (int)blockDim.x + (int)threadIdx.x;
                if (i < npairs) tp[i] = t[b];
            }
        }
    }
    __syncthreads();
    // pixel passes: each pass's unary rows are loaded one pass ahead
    auto pixel = [&](int b0) { return rs.rpix[b0 + gi < np && G.on ? k0r + b0 + gi : k0r]; };
    float un[R];
    int pn = pixel(0);
    if (U) {
        load_row(U + (size_t)pn * L, G, un);
    } else {
#pragma unroll
        for (int r = 0; r < R; r++) un[r] = 0.0f;
    }
    for (int b0 = 0; b0 < np; b0 += items) {
        const bool active = G.on && b0 + gi < np;
        const int p = pn;
        float u[R];
#pragma unroll
        for (int r = 0; r < R; r++) u[r] = un[r];
        if (b0 + items < np) {
            pn = pixel(b0 + items);
            if (U) load_row(U + (size_t)pn * L, G, un);
        }
        int2 e[DS];
#pragma unroll
        for (int j = 0; j < DS; j++) e[j] = active ? tp[(b0 + gi) * DS + j] : make_int2(0, 0);
        float x[DS][R];
#pragma unroll
        for (int j = 0; j < DS; j++) load_piece<R>(tq + (size_t)e[j].x * Lv, k0, L, x[j]);
        finish_pixel<R, D0, D1, false>(G, st, e, x, u, active, Q + (size_t)p * ldq, ldq, shc, p, nullptr);
    }
}

}  // namespace

#define DCRF_FUSED(R_, D0_, D1_)                                                                          \
    DCRF_FUSED_FORM(k_meanfield_fused, R_, D0_, D1_)<<<                                                     \
        blocks_for(N, sh.items), kWaveBlock, fused_lds_bytes(sh, D0_ + D1_, D1_ ? 2 : 1, L, cwf), s>>>(       \
        U, Q, ldq, N, L, sh.S, sh.per, st, slc, cwf, bw)

template <int R>
void launch_fused_r(const LaunchShape& sh, const float* U, float* Q, int ldq, int N, int L, const SliceTable& st,
                    const int2* slc, int cwf, int bw, hipStream_t s) {
    const int a = st.t[0].d1, b = st.nterms > 1 ? st.t[1].d1 : 0;
    const bool narrow = narrow_rows(st.rows, st.t[0].ldv);
    if (a == 3 && b == 0) DCRF_FUSED(R, 3, 0);
    else if (a == 6 && b == 0) DCRF_FUSED(R, 6, 0);
    else if (a == 3 && b == 6) DCRF_FUSED(R, 3, 6);
    else if (a == 6 && b == 3) DCRF_FUSED(R, 6, 3);
    else if (a == 4 && b == 5) DCRF_FUSED(R, 4, 5);
    else if (a == 5 && b == 4) DCRF_FUSED(R, 5, 4);
    else throw Error{DCRF_ERR_VALUE, "no fused mean-field kernel for these terms"};
    DCRF_HIP_CHECK(hipGetLastError());
}
#undef DCRF_FUSED

#define DCRF_RUNS(R_, D0_, D1_)                                                                           \
    k_meanfield_runs<R_, D0_, D1_><<<rs.n_runs, kWaveBlock, lds, s>>>(U, Q, ldq, N, L, Lv, sh.S, sh.per, st, rs)

template <int R>
void launch_runs_r(const LaunchShape& sh, const float* U, float* Q, int ldq, int N, int L, int Lv,
                   const SliceTable& st, const RunSliceDev& rs, size_t lds, hipStream_t s) {
    const int a = st.t[0].d1, b = st.nterms > 1 ? st.t[1].d1 : 0;
    if (a == 3 && b == 0) DCRF_RUNS(R, 3, 0);
    else if (a == 6 && b == 0) DCRF_RUNS(R, 6, 0);
    else if (a == 3 && b == 6) DCRF_RUNS(R, 3, 6);
    else if (a == 6 && b == 3) DCRF_RUNS(R, 6, 3);
    else if (a == 4 && b == 5) DCRF_RUNS(R, 4, 5);
    else if (a == 5 && b == 4) DCRF_RUNS(R, 5, 4);
    else throw Error{DCRF_ERR_VALUE, "no run mean-field kernel for these terms"};
    DCRF_HIP_CHECK(hipGetLastError());
}
#undef DCRF_RUNS

size_t meanfield_runs_lds(int L, int ds, int P, int rows_lds, int cwf) {
    (void)L;
    return (size_t)rows_lds * sizeof(float) + (size_t)P * ds * sizeof(int2) + (size_t)cwf * sizeof(float);
}

void launch_meanfield_runs(const float* U, float* Q, int ldq, int N, int L, int Lv, const SliceTable& st_in,
                           const RunSliceDev& rs, hipStream_t s) {
    SliceTable st = st_in;
    const int cwf = assign_compat_lds(st, L);
    const LaunchShape sh = shape_for(Lv);
    if (!fused_meanfield_ok(L, st.nterms, st.t[0].d1, st.nterms > 1 ? st.t[1].d1 : 0))
        throw Error{DCRF_ERR_VALUE, "no run mean-field kernel for these terms"};
    const int ds = st.t[0].d1 + (st.nterms > 1 ? st.t[1].d1 : 0);
    const size_t lds = meanfield_runs_lds(L, ds, rs.P, rs.rows_lds, cwf);
    static size_t granted[5] = {};
    auto grant = [&](const void* fn, int r) {
        if (lds > granted[r]) {
            DCRF_HIP_CHECK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            granted[r] = lds;
        }
    };
    const int a = st.t[0].d1, b = st.nterms > 1 ? st.t[1].d1 : 0;
    auto fn_for = [&](auto rtag) -> const void* {
        constexpr int R_ = decltype(rtag)::value;
        if (a == 3 && b == 0) return reinterpret_cast<const void*>(&k_meanfield_runs<R_, 3, 0>);
        if (a == 6 && b == 0) return reinterpret_cast<const void*>(&k_meanfield_runs<R_, 6, 0>);
        if (a == 3 && b == 6) return reinterpret_cast<const void*>(&k_meanfield_runs<R_, 3, 6>);
        if (a == 4 && b == 5) return reinterpret_cast<const void*>(&k_meanfield_runs<R_, 4, 5>);
        if (a == 5 && b == 4) return reinterpret_cast<const void*>(&k_meanfield_runs<R_, 5, 4>);
        return reinterpret_cast<const void*>(&k_meanfield_runs<R_, 6, 3>);
    };
    switch (sh.R) {
        case 1: grant(fn_for(std::integral_constant<int, 1>{}), 1); launch_runs_r<1>(sh, U, Q, ldq, N, L, Lv, st, rs, lds, s); break;
        case 2: grant(fn_for(std::integral_constant<int, 2>{}), 2); launch_runs_r<2>(sh, U, Q, ldq, N, L, Lv, st, rs, lds, s); break;
        case 3: grant(fn_for(std::integral_constant<int, 3>{}), 3); launch_runs_r<3>(sh, U, Q, ldq, N, L, Lv, st, rs, lds, s); break;
        default: grant(fn_for(std::integral_constant<int, 4>{}), 4); launch_runs_r<4>(sh, U, Q, ldq, N, L, Lv, st, rs, lds, s); break;
    }
}

void launch_meanfield_fused(const float* U, float* Q, int ldq, int N, int L, int Lv, const SliceTable& st_in,
                            const int2* slc, hipStream_t s, int bw) {
    SliceTable st = st_in;
    const int cwf = assign_compat_lds(st, L, true);  // 16-byte rows for matrix_piece_rows
    const LaunchShape sh = shape_for(Lv);
    if (!fused_meanfield_ok(L, st.nterms, st.t[0].d1, st.nterms > 1 ? st.t[1].d1 : 0))
        throw Error{DCRF_ERR_VALUE, "no fused mean-field kernel for these terms"};
    switch (sh.R) {
        case 1: launch_fused_r<1>(sh, U, Q, ldq, N, L, st, slc, cwf, bw, s); break;
        case 2: launch_fused_r<2>(sh, U, Q, ldq, N, L, st, slc, cwf, bw, s); break;
        case 3: launch_fused_r<3>(sh, U, Q, ldq, N, L, st, slc, cwf, bw, s); break;
        default: launch_fused_r<4>(sh, U, Q, ldq, N, L, st, slc, cwf, bw, s); break;
    }
}

}  // namespace dcrf
