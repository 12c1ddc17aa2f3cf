// What the fused per-pixel kernels (meanfield.hip, adjoint_fused.hip) share: the pixel's
// gathered rows summed per term, the compatibilities, the wave's staged slice pairs.
#pragma once

#include "dcrf_internal.h"
#include "dcrf_device.h"

#pragma clang fp contract(off)

namespace dcrf {

// Term k's message in a fused pixel update: the weighted sum of its gathered rows (entry
// order, as slice_piece) into raw, and raw times the term weight into m.  The caller
// stores raw to the term's `mout` (as k_meanfield does) only after its last read of
// the terms' weights: once a kernel may have stored to global memory, the compiler
// reads those weights through the vector memory path and waits for every load in
// flight (the row gathers among them).
template <int R, int D0, int D1>
__device__ __forceinline__ void term_message(const SliceTerm& T, int k, const int2 (&e)[D0 + D1],
                                             const float (&x)[D0 + D1][R], float (&raw)[R], float (&m)[R]) {
    constexpr int DS = D0 + D1;
    const int jb = k ? D0 : 0, je = k ? DS : D0;
#pragma unroll
    for (int r = 0; r < R; r++) raw[r] = 0.0f;
#pragma unroll
    for (int j = jb; j < je; j++) {
        const float w = __int_as_float(e[j].y);
#pragma unroll
        for (int r = 0; r < R; r++) raw[r] = add_product(raw[r], w, x[j][r]);
    }
#pragma unroll
    for (int r = 0; r < R; r++) m[r] = raw[r];
    if (T.kw) {
        const float kw = T.kw[0];
#pragma unroll
        for (int r = 0; r < R; r++) m[r] = m[r] * kw;
    }
}

// The compatibility transforms c[k] of the pixel's NT term messages.  ROWS: the Matrix
// terms whose weights have an LDS copy (16-byte aligned rows) first write the group's
// message vector into the wave's message region `msg` (NT rows of (L + 3) & ~3 floats
// per group), then read it back whole with matrix_piece_rows: no cross-lane shuffles.
// The other terms go through compat_piece.  Same results either way.
template <int R, int NT, bool ROWS>
__device__ __forceinline__ void compat_terms(LaneGroup<true, R>& G, const SliceTable& st, const float (&mk)[NT][R],
                                             float (&c)[NT][R], const float* shc, float* msg) {
    const int ldm = (G.L + 3) & ~3;
    if (ROWS) {
        bool any = false;
#pragma unroll
        for (int k = 0; k < NT; k++)
            if (st.t[k].ckind == DCRF_COMPAT_MATRIX && st.t[k].cw_lds >= 0) {
                any = true;
                if (G.on) {  // idle lanes shadow group 0: they must not write its row
                    float* row = msg + ((size_t)k * G.per + G.g) * ldm + G.k0;
#pragma unroll
                    for (int r = 0; r < R; r++) row[r] = mk[k][r];
                }
            }
        if (any) {
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        }
    }
#pragma unroll
    for (int k = 0; k < NT; k++) {
        const SliceTerm& T = st.t[k];
        if (ROWS && T.ckind == DCRF_COMPAT_MATRIX && T.cw_lds >= 0)
            matrix_piece_rows<R>(shc + T.cw_lds, T.ldw, msg + ((size_t)k * G.per + G.g) * ldm, G, c[k]);
        else
            compat_piece<true, R>(T, mk[k], c[k], G, shc);
    }
}

// The per-pixel tail of the fused mean-field kernels: the terms' compatibility
// messages subtracted from -U, then the softmax over the lane group, stored when
// `active`.
template <int R, int D0, int D1, bool ROWS>
__device__ __forceinline__ void finish_pixel(LaneGroup<true, R>& G, const SliceTable& st, const int2 (&e)[D0 + D1],
                                             const float (&x)[D0 + D1][R], const float (&u)[R], bool active,
                                             float* __restrict__ qrow, int ldq, const float* shc, int p, float* msg) {
    constexpr int NT = D1 ? 2 : 1;
    float raw[NT][R], mk[NT][R], c[NT][R];
#pragma unroll
    for (int k = 0; k < NT; k++) term_message<R, D0, D1>(st.t[k], k, e, x, raw[k], mk[k]);
    compat_terms<R, NT, ROWS>(G, st, mk, c, shc, msg);
    float en[R];
#pragma unroll
    for (int r = 0; r < R; r++) en[r] = -u[r];
#pragma unroll
    for (int k = 0; k < NT; k++)
#pragma unroll
        for (int r = 0; r < R; r++) en[r] = en[r] - c[k][r];
    G.pad(en, -INFINITY);
    const float mx = G.all_max(en);
    float y[R];
#pragma unroll
    for (int r = 0; r < R; r++) y[r] = expf(en[r] - mx);
    const float sum = G.all_sum(y);
    if (active) {
        float q[R];
        divide_all<R>(y, sum, q);
        store_row(qrow, ldq, G, q);
#pragma unroll
        for (int k = 0; k < NT; k++)
            if (st.t[k].mout) store_row(st.t[k].mout + (size_t)p * G.L, G, raw[k]);
    }
}

// The pixels of a wave of the fused kernels: np >= 1 consecutive ones from p0 (a wave past
// the last pixel repeats it; its results are not stored).  Both are the same in every
// lane, so the wave's rows of the unary, Q and the slice pairs start at scalar addresses.
struct WavePixels {
    int p0, np;
    template <int R>
    __device__ __forceinline__ WavePixels(const LaneGroup<true, R>& G, int p, int N) {
        p0 = __builtin_amdgcn_readfirstlane(min(p - G.g, N - 1));
        np = min(G.per, N - p0);
    }
};

// LDS pairs of one wave's staged slice pairs: its per * ds pairs rounded up to whole rounds
// of 128 (stage_wave_pairs stores whole rounds).
__host__ __device__ inline int wave_pairs(int per, int ds) { return (per * ds + 127) & ~127; }

// Stage the slice pairs of the wave's pixels (one contiguous run of np * DS pairs, 64 pairs
// per load instruction) into the wave's LDS slice wp; the wave's groups then read their
// own.  Past the run the last pair is repeated, so a group without a pixel reads valid
// rows and needs no mask (a masked LDS read per entry, each waited for on its own, had
// made nine round trips of one).
template <int R, int DS>
__device__ __forceinline__ void stage_wave_pairs(const WavePixels& W, int per, const int2* __restrict__ slc,
                                                 int2* wp) {
    const int np = W.np * DS;
    const int lane = threadIdx.x & 63;
    // two loads per lane per round (clamped, unconditional), then the stores.  The pairs
    // are read once per iteration: nontemporal loads keep them from displacing the Q rows
    // this kernel writes, which the next splat gathers (at 1024x768x21 the splat went from
    // 72.5 to 58.3 us; nontemporal loads of the splat's own entries or of the unary row
    // measured slower)
    const long long* __restrict__ src = reinterpret_cast<const long long*>(slc + (size_t)W.p0 * DS);
    long long* dst = reinterpret_cast<long long*>(wp);
    for (int i0 = 0; i0 < per * DS; i0 += 128) {
        const long long t0 = __builtin_nontemporal_load(src + (unsigned)min(i0 + lane, np - 1));
        const long long t1 = __builtin_nontemporal_load(src + (unsigned)min(i0 + 64 + lane, np - 1));
        dst[i0 + lane] = t0;
        dst[i0 + 64 + lane] = t1;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// dynamic LDS of the fused kernels: the wave's slice pairs, the compat region (cwf
// floats), with a compat region the message rows (NT per group, (L + 3) & ~3 floats),
// and the adjoint's statistic region (stat_lds_floats)
inline size_t fused_lds_bytes(const LaunchShape& sh, int ds, int nt, int L, int cwf, int nstat = 0) {
    const size_t waves = kWaveBlock / 64;
    return waves * wave_pairs(sh.per, ds) * sizeof(int2) + (size_t)cwf * sizeof(float) +
           (cwf ? waves * nt * sh.per * (size_t)((L + 3) & ~3) * sizeof(float) : 0) +
           stat_lds_floats(true, nstat, L, kWaveBlock, sh.R) * sizeof(float);
}

// One of a fused kernel's four forms: with or without the LDS copy of Matrix weights, with
// 24-bit or 64-bit row offsets.
#define DCRF_FUSED_FORM(kernel, R_, D0_, D1_)                                              \
    (cwf ? (narrow ? kernel<R_, D0_, D1_, true, true> : kernel<R_, D0_, D1_, true, false>) \
         : (narrow ? kernel<R_, D0_, D1_, false, true> : kernel<R_, D0_, D1_, false, false>))

}  // namespace dcrf
