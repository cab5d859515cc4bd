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
// FP32 two columns): 99 sites 21.5 -> 3.2 / 15.7 -> 4.1, 648 43 -> 5.1 / 31 ->
// 5.4, 2,001 51 -> 11.9 / 37 -> 11.3, 5,003 75 -> 42 / 48 -> 38.
//
// T (rows_targets), us at T = 1 / 2 / 4: with few sites one target per workgroup
// keeps the most workgroups (FP64 one column: 99 sites 3.2 / 3.5 / 5.0, 512 4.3 / 4.2 /
// 5.9); then one source load has to serve several pairs (1,300 sites 9.1 / 8.1 / 9.4,
// 2,400 20.5 / 15.5 / 16.1, 2,700 24.6 / 19.2 / 17.6, 4,000 49 / 33 / 29), and from 4
// targets on damped pairs are listed.  FP32 with two columns does the least per source
// and wants eight instead of four (1 / 2 / 8: 2,400 sites 21 / 14.4 / 19.3, 3,300 35 /
// 23.0 / 23.0, 3,600 42 / 26.4 / 24.7, 5,003 71 / 43.5 / 38).  The line at 3,000 lies
// between those of the two precisions.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "device.h"
#include "pair_math.h"
#include "row_sweep.h"

namespace ommp {

namespace {

template <typename R, int M, bool AMOEBA, int T>
__global__ __launch_bounds__(kBlock) void k_tmv_rows(
    int npol, const typename V4<R>::t *__restrict__ site, const R *__restrict__ adamp, const R *__restrict__ rc2,
    const double4 *__restrict__ ps, const double *__restrict__ pa, const double *__restrict__ alpha,
    const int *__restrict__ pp_ri, const int *__restrict__ pp_ci, const double *__restrict__ pp_f,
    const double *__restrict__ x, long xstride, double *__restrict__ y, long ystride, int dodiag,
    double *__restrict__ dotpart, const CgState *__restrict__ skip, int skipM) {
    using R4 = typename V4<R>::t;
    if (skip) {
        bool all = true;
        for (int m = 0; m < skipM; m++) all = all && skip[m].done;
        if (all) return;
    }
    __shared__ RowLds<R, M, T> lds;
    const int tid = threadIdx.x;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j0 = blockIdx.x * T;
    // targets past the end repeat the last site; their results are not written
    auto tgt = [&](int t) { return min(j0 + t, npol - 1); };
    auto id = [](int i) { return i; };
    RowAcc<R, M, T> acc;
#pragma unroll
    for (int t = 0; t < T; t++) row_target(acc, t, site[tgt(t)], adamp[tgt(t)], rc2[tgt(t)]);
    R4 pn, vn[M];
    R an = R(0);
    auto load = [&](int i) {
        pn = site[i];
        an = adamp[i];
#pragma unroll
        for (int m = 0; m < M; m++) {
            vn[m].x = (R)x[m * xstride + 3L * i + 0];
            vn[m].y = (R)x[m * xstride + 3L * i + 1];
            vn[m].z = (R)x[m * xstride + 3L * i + 2];
        }
    };
    if (tid < npol) load(tid);
    for (int i = tid; i < npol; i += kBlock) {
        const R4 p = pn;
        const R a = an;
        R4 v[M];
#pragma unroll
        for (int m = 0; m < M; m++) v[m] = vn[m];
        if (i + kBlock < npol) load(i + kBlock);  // the next source while this one is used
        row_source<AMOEBA>(acc, lds, w, i, p, a, v, site, adamp, tgt);
    }
    row_finish<AMOEBA>(acc, lds, w, site, adamp, x, xstride, ps, pa, pp_ri, pp_ci, pp_f, tgt, id);
    row_store(lds, npol - j0, alpha, x, xstride, y, ystride, dodiag != 0, dotpart ? dotpart + blockIdx.x : nullptr,
              (long)gridDim.x, tgt, id);
}

int rows_targets(int npol, int prec, int ncols) {
    if (npol <= 512) return 1;
    if (npol <= 3000) return 2;
    return prec == 32 && ncols == 2 ? 8 : 4;
}

template <typename R, int M, bool AMOEBA>
void rows_launch(hipStream_t st, int npol, const typename V4<R>::t *site, const R *ad, const R *rc2, const double4 *ps64,
                 const double *pa64, const double *alpha, const CsrDev &pp, const double *x, long xs, double *y,
                 long ys, bool dodiag, double *dotpart, const CgState *skip) {
    constexpr int prec = 8 * sizeof(R), TL = prec == 32 && M == 2 ? 8 : 4;
    const dim3 grid(tmv_rows_dot_parts(npol, prec, M)), block(kBlock);
    switch (rows_targets(npol, prec, M)) {
        case 1:
            hipLaunchKernelGGL((k_tmv_rows<R, M, AMOEBA, 1>), grid, block, 0, st, npol, site, ad, rc2, ps64, pa64, alpha,
                               pp.ri, pp.ci, pp.f, x, xs, y, ys, (int)dodiag, dotpart, skip, M);
            break;
        case 2:
            hipLaunchKernelGGL((k_tmv_rows<R, M, AMOEBA, 2>), grid, block, 0, st, npol, site, ad, rc2, ps64, pa64, alpha,
                               pp.ri, pp.ci, pp.f, x, xs, y, ys, (int)dodiag, dotpart, skip, M);
            break;
        default:
            hipLaunchKernelGGL((k_tmv_rows<R, M, AMOEBA, TL>), grid, block, 0, st, npol, site, ad, rc2, ps64, pa64, alpha,
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
                     const float4 *ps32, const float *pa32, const double *rc64, const float *rc32, const double *alpha,
                     const CsrDev &pp, const double *x, long xstride, double *y, long ystride, bool dodiag,
                     double *dotpart, const int *skip_flag, hipEvent_t evb, hipEvent_t eve) {
    if (npol == 0) return;
    const CgState *skip = reinterpret_cast<const CgState *>(skip_flag);
    if (evb) HIP_CHECK(hipEventRecord(evb, st));
    auto go = [&](auto am) {
        constexpr bool A = decltype(am)::value;
        if (prec == 32 && M == 1)
            rows_launch<float, 1, A>(st, npol, ps32, pa32, rc32, ps64, pa64, alpha, pp, x, xstride, y, ystride, dodiag,
                                     dotpart, skip);
        else if (prec == 32)
            rows_launch<float, 2, A>(st, npol, ps32, pa32, rc32, ps64, pa64, alpha, pp, x, xstride, y, ystride, dodiag,
                                     dotpart, skip);
        else if (M == 1)
            rows_launch<double, 1, A>(st, npol, ps64, pa64, rc64, ps64, pa64, alpha, pp, x, xstride, y, ystride, dodiag,
                                      dotpart, skip);
        else
            rows_launch<double, 2, A>(st, npol, ps64, pa64, rc64, ps64, pa64, alpha, pp, x, xstride, y, ystride, dodiag,
                                      dotpart, skip);
    };
    if (amoeba) go(std::true_type{});
    else go(std::false_type{});
    if (eve) HIP_CHECK(hipEventRecord(eve, st));
}

}  // namespace ommp
