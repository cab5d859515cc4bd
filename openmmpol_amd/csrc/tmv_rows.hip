// T matvec on the fly, per target: one workgroup per T target sites, its 256
// threads on the sources (thread t takes sources t, t + 256, ...), for the sizes
// where the pair-once sweep (tmv_sym.hip) does not pay.  The targets' data is
// uniform over the workgroup (scalar registers), every source is loaded once per
// workgroup and met by T targets, and the sum over the sources ends in the same
// workgroup: lane exchanges that hand each half of a wave half of the targets,
// then the four waves' rows through LDS.  The sparse (1 - s) corrections, the
// diagonal x / alpha and the y.x partial follow there, so a matvec is one launch
// and writes no partial sums.
//
// What bounds it: below ~2,000 sites the latency of one launch and of the few
// loads a thread makes; above, the vector ALUs.  Measured against the sweep it
// replaces (one target per thread, the sources split over workgroups, partial
// sums added by a second kernel; chain systems, us per matvec, FP64 one column /
// FP32 two columns): 99 sites 21.5 -> 2.9 / 15.7 -> 3.2, 648 43 -> 4.8 / 31 ->
// 4.7, 2,001 51 -> 12.7 / 37 -> 10.2, 5,003 76 -> 59 / 47 -> 38.
//
// T (rows_targets), us at T = 1 / 2 / 4 / 8: with few sites one target per
// workgroup keeps the most workgroups (99 sites, FP64: 2.9 / 3.2 / 4.7 / 5.2); then
// one source load has to serve several pairs (3,000 sites, FP64: 41 / 24.0 / 25.1 /
// 27; 5,003: 108 / 60 / 59 / 60); FP32 with two columns does the least per
// source and wants eight (5,003: 74 / 43.6 / 46.0 / 38.5).
#include <hip/hip_runtime.h>

#include <type_traits>

#include "device.h"
#include "pair_math.h"

namespace ommp {

namespace {

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

template <typename R, int M, bool AMOEBA, int T>
__global__ __launch_bounds__(kBlock) void k_tmv_rows(
    int npol, const typename V4<R>::t *__restrict__ site, const R *__restrict__ adamp,
    const double4 *__restrict__ ps, const double *__restrict__ pa, const double *__restrict__ alpha,
    const int *__restrict__ pp_ri, const int *__restrict__ pp_ci, const double *__restrict__ pp_f,
    const double *__restrict__ x, long xstride, double *__restrict__ y, long ystride, int dodiag,
    double *__restrict__ dotpart, const CgState *__restrict__ skip, int skipM) {
    using R4 = typename V4<R>::t;
    constexpr int C = 3 * M, W = kBlock / 64;
    if (skip) {
        bool all = true;
        for (int m = 0; m < skipM; m++) all = all && skip[m].done;
        if (all) return;
    }
    __shared__ R s_row[W][T][C];
    __shared__ double s_corr[T][C];
    __shared__ double s_dot[T][C];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j0 = blockIdx.x * T;
    // targets past the end repeat the last site; their results are not written
    R4 pj[T];
    R aj[T];
#pragma unroll
    for (int t = 0; t < T; t++) {
        const int j = min(j0 + t, npol - 1);
        pj[t] = site[j];
        aj[t] = adamp[j];
    }
    R acc[T][M][3];
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
        for (int m = 0; m < M; m++) acc[t][m][0] = acc[t][m][1] = acc[t][m][2] = R(0);
    auto load = [&](int i, R4 &p, R &a, R4 (&v)[M]) {
        p = site[i];
        a = adamp[i];
#pragma unroll
        for (int m = 0; m < M; m++) {
            v[m].x = (R)x[m * xstride + 3L * i + 0];
            v[m].y = (R)x[m * xstride + 3L * i + 1];
            v[m].z = (R)x[m * xstride + 3L * i + 2];
        }
    };
    R4 pn, vn[M];
    R an;
    if (tid < npol) load(tid, pn, an, vn);
    for (int i = tid; i < npol; i += kBlock) {
        const R4 pi = pn;
        const R ai = an;
        R4 v[M];
#pragma unroll
        for (int m = 0; m < M; m++) v[m] = vn[m];
        if (i + kBlock < npol) load(i + kBlock, pn, an, vn);  // the next source while this one is used
#pragma unroll
        for (int t = 0; t < T; t++) {
            R dx, dy, dz, k2, k3, arg;
            bool near;
            pair_geom<R, AMOEBA>(pj[t], aj[t], pi, ai, dx, dy, dz, k2, k3, arg, near);
            if (__ballot(near)) pair_damp<R, AMOEBA>(arg, near, k2, k3);
            pair_accum<R, M>(acc[t], v, dx, dy, dz, k2, k3);
        }
    }
    {
        R flat[T * C];
#pragma unroll
        for (int t = 0; t < T; t++)
#pragma unroll
            for (int m = 0; m < M; m++)
#pragma unroll
                for (int c = 0; c < 3; c++) flat[t * C + 3 * m + c] = acc[t][m][c];
        wave_rows<R, T, C>(flat);
        constexpr int G = 64 / T;
        if (lane % G == 0) {
#pragma unroll
            for (int c = 0; c < C; c++) s_row[w][lane / G][c] = flat[c];
        }
    }
    // corrections of target t by wave t % W: the listed pairs over its lanes
    for (int t = w; t < T; t += W) {
        const int j = min(j0 + t, npol - 1);
        const int k0 = pp_ri[j], k1 = pp_ri[j + 1];
        double corr[C];
#pragma unroll
        for (int c = 0; c < C; c++) corr[c] = 0.0;
        if (k0 < k1) {
            const double4 qj = ps[j];
            const double bj = pa[j];
            for (int k = k0 + lane; k < k1; k += 64) {
                const int i = pp_ci[k];
                const double f = pp_f[k];
                const double4 pi = ps[i];
                const double dx = qj.x - pi.x, dy = qj.y - pi.y, dz = qj.z - pi.z;
                const double r2 = dx * dx + dy * dy + dz * dz;
                double k2, k3;
                dip_kernel<double, AMOEBA>(r2, rsqrt(r2), pi.w, qj.w, pa[i], bj, k2, k3);
#pragma unroll
                for (int m = 0; m < M; m++) {
                    const double *xi = x + m * xstride + 3L * i;
                    const double c = k3 * (xi[0] * dx + xi[1] * dy + xi[2] * dz);
                    corr[3 * m + 0] += f * (c * dx - k2 * xi[0]);
                    corr[3 * m + 1] += f * (c * dy - k2 * xi[1]);
                    corr[3 * m + 2] += f * (c * dz - k2 * xi[2]);
                }
            }
            wave_rows<double, 1, C>(corr);
        }
        if (lane == 0) {
#pragma unroll
            for (int c = 0; c < C; c++) s_corr[t][c] = corr[c];
        }
    }
    __syncthreads();
    if (tid < T * C) {
        const int t = tid / C, c = tid % C, j = j0 + t;
        double out = 0.0;
        if (j < npol) {
            R s = s_row[0][t][c];
#pragma unroll
            for (int q = 1; q < W; q++) s += s_row[q][t][c];
            const double xj = x[c / 3 * xstride + 3L * j + c % 3];
            double v = s_corr[t][c] - (double)s;
            if (dodiag) v += xj * (1.0 / alpha[j]);
            y[c / 3 * ystride + 3L * j + c % 3] = v;
            out = v * xj;
        }
        s_dot[t][c] = out;
    }
    if (!dotpart) return;
    __syncthreads();
    if (tid < M) {
        double d = 0.0;
#pragma unroll
        for (int t = 0; t < T; t++) d += (s_dot[t][3 * tid] + s_dot[t][3 * tid + 1]) + s_dot[t][3 * tid + 2];
        dotpart[tid * gridDim.x + blockIdx.x] = d;
    }
}

int rows_targets(int npol, int prec, int ncols) {
    if (npol <= 512) return 1;
    if (npol <= 3000) return 2;
    return prec == 32 && ncols == 2 ? 8 : 4;
}

template <typename R, int M, bool AMOEBA>
void rows_launch(hipStream_t st, int npol, const typename V4<R>::t *site, const R *ad, const double4 *ps64,
                 const double *pa64, const double *alpha, const CsrDev &pp, const double *x, long xs, double *y,
                 long ys, bool dodiag, double *dotpart, const CgState *skip) {
    constexpr int prec = 8 * sizeof(R), TL = prec == 32 && M == 2 ? 8 : 4;
    const dim3 grid(tmv_rows_dot_parts(npol, prec, M)), block(kBlock);
    switch (rows_targets(npol, prec, M)) {
        case 1:
            hipLaunchKernelGGL((k_tmv_rows<R, M, AMOEBA, 1>), grid, block, 0, st, npol, site, ad, ps64, pa64, alpha,
                               pp.ri, pp.ci, pp.f, x, xs, y, ys, (int)dodiag, dotpart, skip, M);
            break;
        case 2:
            hipLaunchKernelGGL((k_tmv_rows<R, M, AMOEBA, 2>), grid, block, 0, st, npol, site, ad, ps64, pa64, alpha,
                               pp.ri, pp.ci, pp.f, x, xs, y, ys, (int)dodiag, dotpart, skip, M);
            break;
        default:
            hipLaunchKernelGGL((k_tmv_rows<R, M, AMOEBA, TL>), grid, block, 0, st, npol, site, ad, ps64, pa64, alpha,
                               pp.ri, pp.ci, pp.f, x, xs, y, ys, (int)dodiag, dotpart, skip, M);
    }
    HIP_CHECK(hipGetLastError());
}

}  // namespace

int tmv_rows_dot_parts(int npol, int prec, int ncols) {
    const int t = rows_targets(npol, prec, ncols);
    return (npol + t - 1) / t;
}

void launch_tmv_rows(hipStream_t st, int prec, bool amoeba, int npol, int M, const double4 *ps64, const double *pa64,
                     const float4 *ps32, const float *pa32, const double *alpha, const CsrDev &pp, const double *x,
                     long xstride, double *y, long ystride, bool dodiag, double *dotpart, const int *skip_flag,
                     hipEvent_t evb, hipEvent_t eve) {
    if (npol == 0) return;
    const CgState *skip = reinterpret_cast<const CgState *>(skip_flag);
    if (evb) HIP_CHECK(hipEventRecord(evb, st));
    auto go = [&](auto am) {
        constexpr bool A = decltype(am)::value;
        if (prec == 32 && M == 1)
            rows_launch<float, 1, A>(st, npol, ps32, pa32, ps64, pa64, alpha, pp, x, xstride, y, ystride, dodiag,
                                     dotpart, skip);
        else if (prec == 32)
            rows_launch<float, 2, A>(st, npol, ps32, pa32, ps64, pa64, alpha, pp, x, xstride, y, ystride, dodiag,
                                     dotpart, skip);
        else if (M == 1)
            rows_launch<double, 1, A>(st, npol, ps64, pa64, ps64, pa64, alpha, pp, x, xstride, y, ystride, dodiag,
                                      dotpart, skip);
        else
            rows_launch<double, 2, A>(st, npol, ps64, pa64, ps64, pa64, alpha, pp, x, xstride, y, ystride, dodiag,
                                      dotpart, skip);
    };
    if (amoeba) go(std::true_type{});
    else go(std::false_type{});
    if (eve) HIP_CHECK(hipEventRecord(eve, st));
}

}  // namespace ommp
