// Sweep of T targets over sources that are spread over the 256 threads of a
// workgroup: the inner part of the per-target T matvec (tmv_rows.hip).
//
// A pair is compared with the target's cutoff rc2 (beyond it no pair of the target is
// damped, whatever the source), one compare per pair; damping acts within a few
// Angstrom of a target.  T < kRowListT: the argument and the exponential are formed
// where a lane of the wave is inside.  With many sources a target's few dozen such
// pairs are spread over half of the steps of a wave, each of which would compute them
// for a few lanes.  So from kRowListT targets on (many sources) pairs inside are left
// out of the sweep, listed in LDS by target and wave, and done at its end with full
// waves, where the exact argument decides.  A list that is full (a dense cluster, an
// outlying polarizability) damps in place.  The order of a list is that of the sweep:
// sums are reproducible.  Instructions per undamped pair (FP64, one column): 80 -> 36;
// 9,001 sites FP64 one column 160 -> 121 us per matvec, 5,003: 58 -> 42; with one or
// two targets (below 3,000 sites) the list's end costs 1 us of 3-6.
#pragma once

#include <hip/hip_runtime.h>

#include "device.h"
#include "pair_math.h"

namespace ommp {

constexpr int kRowListT = 4;              // targets per workgroup from which pairs are listed
constexpr int kRowCap = 64;              // listed pairs per target and wave
constexpr int kRowWaves = kBlock / 64;

// v[NT * C] per lane -> every lane of the k-th 64 / NT lanes holds the wave's sum
// of v[k * C .. k * C + C): at each step the two halves of a lane group exchange
// the half they do not keep.  Fixed order.
template <typename R, int NT, int C>
__device__ __forceinline__ void wave_rows(R (&v)[NT * C]) {
    const int lane = threadIdx.x & 63;
    int mask = 32;
#pragma unroll
    for (int cnt = NT; cnt > 1; cnt >>= 1, mask >>= 1) {
        const bool hi = lane & mask;
        const int h = cnt / 2 * C;
#pragma unroll
        for (int k = 0; k < NT * C / 2; k++)
            if (k < h) {
                const R keep = hi ? v[k + h] : v[k], send = hi ? v[k] : v[k + h];
                v[k] = keep + __shfl_xor(send, mask, 64);
            }
    }
#pragma unroll
    for (; mask > 0; mask >>= 1)
#pragma unroll
        for (int k = 0; k < C; k++) v[k] += __shfl_xor(v[k], mask, 64);
}

template <typename R, int M, int T> struct RowLds {
    int near[T][kRowWaves][kRowCap], nnear[T][kRowWaves];
    R row[kRowWaves][T][3 * M];
    double corr[T][3 * M], dot[T][3 * M];
};

template <typename R, int M, int T> struct RowAcc {
    R x[T], y[T], z[T], rc2[T];  // targets (uniform over the workgroup)
    R w[T], a[T];
    int n[T];                    // pairs listed by this wave
    R f[T][M][3];
};

template <typename R, int M, int T>
__device__ __forceinline__ void row_target(RowAcc<R, M, T> &acc, int t, const typename V4<R>::t &p, R a, R rc2) {
    acc.x[t] = p.x;
    acc.y[t] = p.y;
    acc.z[t] = p.z;
    acc.w[t] = p.w;
    acc.a[t] = a;
    acc.rc2[t] = rc2;
    acc.n[t] = 0;
#pragma unroll
    for (int m = 0; m < M; m++) acc.f[t][m][0] = acc.f[t][m][1] = acc.f[t][m][2] = R(0);
}

// Source i at p (damping pa) with dipoles v: sites site / adamp are indexed by i and,
// for target t, by tgt(t).
template <bool AMOEBA, typename R, int M, int T, typename Tgt>
__device__ __forceinline__ void row_source(RowAcc<R, M, T> &a, RowLds<R, M, T> &lds, int w, int i,
                                           const typename V4<R>::t &p, R pa, const typename V4<R>::t (&v)[M],
                                           const typename V4<R>::t *__restrict__ site, const R *__restrict__ adamp,
                                           Tgt &&tgt) {
#pragma unroll
    for (int t = 0; t < T; t++) {
        typename V4<R>::t pt;
        pt.x = a.x[t];
        pt.y = a.y[t];
        pt.z = a.z[t];
        pt.w = a.w[t];
        R dx, dy, dz, k2, k3, arg;
        bool near;
        const bool in = pair_bare<R>(pt, p, dx, dy, dz, k2, k3) < a.rc2[t];  // the target itself among them
        const unsigned long long mask = __ballot(in);
        if (T < kRowListT) {
            if (mask) {
                pair_geom<R, AMOEBA>(pt, a.a[t], p, pa, dx, dy, dz, k2, k3, arg, near);
                if (__ballot(near)) pair_damp<R, AMOEBA>(arg, near, k2, k3);
            }
        } else if (mask) {
            const int c = __popcll(mask);
            if (a.n[t] + c <= kRowCap) {
                const int before = __builtin_amdgcn_mbcnt_hi((unsigned)(mask >> 32),
                                                             __builtin_amdgcn_mbcnt_lo((unsigned)mask, 0));
                if (in) lds.near[t][w][a.n[t] + before] = i;
                a.n[t] += c;
                k2 = in ? R(0) : k2;
                k3 = in ? R(0) : k3;
            } else {
                pair_geom<R, AMOEBA>(site[tgt(t)], adamp[tgt(t)], site[i], adamp[i], dx, dy, dz, k2, k3, arg, near);
                if (__ballot(near)) pair_damp<R, AMOEBA>(arg, near, k2, k3);
            }
        }
        pair_accum<R, M>(a.f[t], v, dx, dy, dz, k2, k3);
    }
}

// End of the sweep: the lanes' sums to lds.row, the listed pairs and the screened
// pairs (pp lists, FP64) of every target to lds.corr.  x is indexed by site: id(i)
// of source i and of target t, id(tgt(t)).
template <bool AMOEBA, typename R, int M, int T, typename Tgt, typename Id>
__device__ __forceinline__ void row_finish(RowAcc<R, M, T> &a, RowLds<R, M, T> &lds, int w,
                                           const typename V4<R>::t *__restrict__ site, const R *__restrict__ adamp,
                                           const double *__restrict__ x, long xstride,
                                           const double4 *__restrict__ ps, const double *__restrict__ pa,
                                           const int *__restrict__ pp_ri, const int *__restrict__ pp_ci,
                                           const double *__restrict__ pp_f, Tgt &&tgt, Id &&id) {
    constexpr int C = 3 * M, W = kRowWaves, G = 64 / T;
    const int lane = threadIdx.x & 63;
    R flat[T * C];
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int c = 0; c < C; c++) flat[t * C + c] = a.f[t][c / 3][c % 3];
    wave_rows<R, T, C>(flat);
    if (lane % G == 0) {
#pragma unroll
        for (int c = 0; c < C; c++) lds.row[w][lane / G][c] = flat[c];
    }
    if (lane == 0) {
#pragma unroll
        for (int t = 0; t < T; t++) lds.nnear[t][w] = a.n[t];
    }
    __syncthreads();
    // target t by wave t % W, pairs over its lanes
    for (int t = w; t < T; t += W) {
        const int ti = tgt(t), j = id(ti);
        double corr[C];
#pragma unroll
        for (int c = 0; c < C; c++) corr[c] = 0.0;
        int end[W];  // of the target's four lists, one after the other
#pragma unroll
        for (int u = 0; u < W; u++) end[u] = lds.nnear[t][u] + (u > 0 ? end[u - 1] : 0);
        if (T >= kRowListT && end[W - 1] > 0) {
            const typename V4<R>::t pt = site[ti];
            const R at = adamp[ti];
            for (int e = lane; e < end[W - 1]; e += 64) {
                int u = 0, first = 0;
#pragma unroll
                for (int k = 0; k < W - 1; k++)
                    if (e >= end[k]) {
                        u = k + 1;
                        first = end[k];
                    }
                const int i = lds.near[t][u][e - first];
                const long xi = 3L * id(i);
                typename V4<R>::t v[M];
#pragma unroll
                for (int m = 0; m < M; m++) {
                    v[m].x = (R)x[m * xstride + xi];
                    v[m].y = (R)x[m * xstride + xi + 1];
                    v[m].z = (R)x[m * xstride + xi + 2];
                }
                R dx, dy, dz, k2, k3, arg, f[M][3];
                bool near;
#pragma unroll
                for (int m = 0; m < M; m++) f[m][0] = f[m][1] = f[m][2] = R(0);
                pair_geom<R, AMOEBA>(pt, at, site[i], adamp[i], dx, dy, dz, k2, k3, arg, near);  // 0 for itself
                pair_damp<R, AMOEBA>(arg, near, k2, k3);
                pair_accum<R, M>(f, v, dx, dy, dz, k2, k3);
#pragma unroll
                for (int c = 0; c < C; c++) corr[c] -= (double)f[c / 3][c % 3];
            }
        }
        screened_pairs<AMOEBA, M>(j, lane, 64, ps, pa, pp_ri, pp_ci, pp_f, x, xstride, corr);
        wave_rows<double, 1, C>(corr);
        if (lane == 0) {
#pragma unroll
            for (int c = 0; c < C; c++) lds.corr[t][c] = corr[c];
        }
    }
    __syncthreads();
}

// y of target t < nt (site id(tgt(t))) from lds.row and lds.corr, and the
// workgroup's y.x sum of column m to dot[m * dstride] by thread m.
template <typename R, int M, int T, typename Tgt, typename Id>
__device__ __forceinline__ void row_store(RowLds<R, M, T> &lds, int nt, const double *__restrict__ alpha,
                                          const double *__restrict__ x, long xstride, double *__restrict__ y,
                                          long ystride, bool dodiag, double *__restrict__ dot, long dstride, Tgt &&tgt,
                                          Id &&id) {
    constexpr int C = 3 * M;
    const int tid = threadIdx.x;
    if (tid < T * C) {
        const int t = tid / C, c = tid % C;
        double out = 0.0;
        if (t < nt) {
            const int j = id(tgt(t));
            R s = lds.row[0][t][c];
#pragma unroll
            for (int q = 1; q < kRowWaves; q++) s += lds.row[q][t][c];
            const double xj = x[c / 3 * xstride + 3L * j + c % 3];
            double v = lds.corr[t][c] - (double)s;
            if (dodiag) v += xj * (1.0 / alpha[j]);
            y[c / 3 * ystride + 3L * j + c % 3] = v;
            out = v * xj;
        }
        lds.dot[t][c] = out;
    }
    if (!dot) return;
    __syncthreads();
    if (tid < M) {
        double d = 0.0;
#pragma unroll
        for (int t = 0; t < T; t++)
            d += (lds.dot[t][3 * tid] + lds.dot[t][3 * tid + 1]) + lds.dot[t][3 * tid + 2];
        dot[tid * dstride] = d;
    }
}

}  // namespace ommp
