// Potential and field of the static multipoles and of the induced dipoles at
// arbitrary external points (potential_M2E / potential_D2E / field_M2E /
// field_D2E, mod_electrostatics.F90:3067-3336): undamped, unscreened, FP64.
// One thread per 1, 2 or 4 external points, sources staged through LDS in tiles of 256,
// the source range split over gridDim.y (down to 16 sources a split where there
// are few points: 30 points and 2,001 sources 34 -> 6 us); the per-split partial
// results are added in a fixed order by the finalize kernel.  The sweeps are
// bound by the FP64 vector ALUs and form the potential, the field or both as the
// entry point asks (20,000 points, 24,000 multipoles, potential alone: 1,238 -> 564 us with
// four points per thread and the quadrupole as a quadratic form, 38 instructions a pair).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <mutex>
#include <string>
#include <type_traits>

#include "device.h"
#include "pair_math.h"

namespace ommp {

constexpr double kEps2 = kEpsRpDev * kEpsRpDev;

// d and 1/r of one source and a thread's P points.  1/r is the refined hardware
// estimate; where some lane's r2 is not clearly between kEps2 and 1e300 (one test
// of the high word for all P, a branch that is never taken in earnest) the
// general routine is used instead, and 0 with *hit set for a point on the source.
template <int P>
__device__ __forceinline__ void x2e_geom(const double (&px)[P], const double (&py)[P], const double (&pz)[P],
                                         const double4 &s, double (&dx)[P], double (&dy)[P], double (&dz)[P],
                                         double (&k1)[P], int &hit) {
    constexpr unsigned lo = 0x3A500000u, span = 0x7E370000u - lo;  // high words above kEps2 = 4.93e-28 and below 1e300
    static_assert(kEps2 < 5e-28, "lo is the high word of 8.1e-28");
    unsigned odd = 0;
#pragma unroll
    for (int h = 0; h < P; h++) {
        dx[h] = px[h] - s.x;
        dy[h] = py[h] - s.y;
        dz[h] = pz[h] - s.z;
        const double r2 = fma(dz[h], dz[h], fma(dy[h], dy[h], dx[h] * dx[h]));
        odd = max(odd, (unsigned)__double2hiint(r2) - lo);
        k1[h] = fast_rsqrt(r2);
    }
    if (__ballot(odd >= span)) {
#pragma unroll
        for (int h = 0; h < P; h++) {
            double r2 = fma(dz[h], dz[h], fma(dy[h], dy[h], dx[h] * dx[h]));
            asm volatile("" : "+v"(r2));  // keeps the general routine's work inside the branch
            if (r2 < kEps2) hit = 1;
            k1[h] = r2 < kEps2 ? 0.0 : rsqrt(r2);
        }
    }
}

// P points per thread (x2e_points): every source read from LDS then meets P
// points; with one point per thread the sweep waits on the LDS (14 broadcast
// doubles per multipole).
//
// Multipole sources: ms[i] = (x, y, z, .), mq[i][LD] = q, mu, quadrupole / 3
// (xx, xy, yy, xz, yz, zz).  V = q k1 + (mu.d) k2 + 3 (d.Q d) k3;
// E = q k2 d + 3 (mu.d) k3 d - k2 mu + 15 (d.Q d) k4 d - 6 k3 Q d, d = r_ext - r_i.
template <int LD, bool V, bool E, int P>
__global__ __launch_bounds__(kBlock) void k_m2e(int n, const double *__restrict__ cext, int nsrc, int chunk,
                                                const double4 *__restrict__ ms, const double *__restrict__ mq,
                                                double4 *__restrict__ part, int *__restrict__ bad) {
    __shared__ double4 s_pos[kBlock];
    __shared__ double s_q[kBlock][LD];
    const int tid = threadIdx.x;
    const int j0 = blockIdx.x * kBlock * P + tid;  // points j0, j0 + kBlock, ...
    double px[P], py[P], pz[P], v[P], ex[P], ey[P], ez[P];
#pragma unroll
    for (int h = 0; h < P; h++) {
        const int j = min(j0 + h * kBlock, n - 1);  // past the end: the last point again, not written
        px[h] = cext[3L * j];
        py[h] = cext[3L * j + 1];
        pz[h] = cext[3L * j + 2];
        v[h] = ex[h] = ey[h] = ez[h] = 0.0;
    }
    int hit = 0;
    const int i0 = blockIdx.y * chunk;
    const int i1 = min(nsrc, i0 + chunk);
    for (int base = i0; base < i1; base += kBlock) {
        const int cnt = min(kBlock, i1 - base);
        __syncthreads();
        if (tid < cnt) {
            s_pos[tid] = ms[base + tid];
#pragma unroll
            for (int c = 0; c < LD; c++) {
                const double v = mq[(long)LD * (base + tid) + c];
                // the potential alone takes 3 d.Q d as a quadratic form: its factors
                // are put into the coefficients here
                s_q[tid][c] = E || c < 4 ? v : (c == 4 || c == 6 || c == 9 ? 3.0 * v : 6.0 * v);
            }
        }
        __syncthreads();
        for (int k = 0; k < cnt; k++) {
            const double4 ps = s_pos[k];
            double m[LD];
#pragma unroll
            for (int c = 0; c < LD; c++) m[c] = s_q[k][c];
            double ax[P], ay[P], az[P], ak[P];
            x2e_geom<P>(px, py, pz, ps, ax, ay, az, ak, hit);
#pragma unroll
            for (int h = 0; h < P; h++) {
                const double dx = ax[h], dy = ay[h], dz = az[h], k1 = ak[h], ir2 = k1 * k1;
                if (LD == 1) {
                    if (V) v[h] += m[0] * k1;
                    if (E) {
                        const double c = m[0] * (k1 * ir2);
                        ex[h] += c * dx;
                        ey[h] += c * dy;
                        ez[h] += c * dz;
                    }
                } else {
                    const double md = m[1] * dx + m[2] * dy + m[3] * dz;
                    if (!E) {
                        const double q3 = (m[4] * dx + m[5] * dy + m[7] * dz) * dx + (m[6] * dy + m[8] * dz) * dy +
                                          m[9] * dz * dz;
                        v[h] += k1 * (m[0] + ir2 * (md + ir2 * q3));
                        continue;
                    }
                    const double qx = m[4] * dx + m[5] * dy + m[7] * dz;
                    const double qy = m[5] * dx + m[6] * dy + m[8] * dz;
                    const double qz = m[7] * dx + m[8] * dy + m[9] * dz;
                    const double q3 = 3.0 * (qx * dx + qy * dy + qz * dz);
                    if (V) v[h] += k1 * (m[0] + ir2 * (md + ir2 * q3));
                    const double k2 = k1 * ir2, k3 = k2 * ir2;
                    const double cd = k2 * (m[0] + ir2 * (3.0 * md + ir2 * (5.0 * q3)));
                    ex[h] += cd * dx - m[1] * k2 - 6.0 * qx * k3;
                    ey[h] += cd * dy - m[2] * k2 - 6.0 * qy * k3;
                    ez[h] += cd * dz - m[3] * k2 - 6.0 * qz * k3;
                }
            }
        }
    }
#pragma unroll
    for (int h = 0; h < P; h++) {
        const int j = j0 + h * kBlock;
        if (j < n) part[(long)blockIdx.y * n + j] = make_double4(v[h], ex[h], ey[h], ez[h]);
    }
    if (hit) *bad = 1;
}

// Induced-dipole sources: ps[i] = position, potential from muV (the D set for
// AMOEBA), field from muE (1/2 (mu_D + mu_P) for AMOEBA, mod_electrostatics.F90:3250).
template <bool V, bool E, int P>
__global__ __launch_bounds__(kBlock) void k_d2e(int n, const double *__restrict__ cext, int nsrc, int chunk,
                                                const double4 *__restrict__ ps, const double *__restrict__ ipd,
                                                int amoeba, double4 *__restrict__ part, int *__restrict__ bad) {
    __shared__ double4 s_pos[kBlock];
    __shared__ double s_mv[3][kBlock], s_me[3][kBlock];
    const int tid = threadIdx.x;
    const int j0 = blockIdx.x * kBlock * P + tid;
    double px[P], py[P], pz[P], v[P], ex[P], ey[P], ez[P];
#pragma unroll
    for (int h = 0; h < P; h++) {
        const int j = min(j0 + h * kBlock, n - 1);
        px[h] = cext[3L * j];
        py[h] = cext[3L * j + 1];
        pz[h] = cext[3L * j + 2];
        v[h] = ex[h] = ey[h] = ez[h] = 0.0;
    }
    int hit = 0;
    const int i0 = blockIdx.y * chunk;
    const int i1 = min(nsrc, i0 + chunk);
    const long np3 = 3L * nsrc;
    for (int base = i0; base < i1; base += kBlock) {
        const int cnt = min(kBlock, i1 - base);
        __syncthreads();
        if (tid < cnt) {
            const long i = base + tid;
            s_pos[tid] = ps[i];
#pragma unroll
            for (int c = 0; c < 3; c++) {
                const double d = ipd[3 * i + c];
                s_mv[c][tid] = d;
                if (E) s_me[c][tid] = amoeba ? 0.5 * (ipd[np3 + 3 * i + c] + d) : d;
            }
        }
        __syncthreads();
        for (int k = 0; k < cnt; k++) {
            const double4 q = s_pos[k];
            const double vx = s_mv[0][k], vy = s_mv[1][k], vz = s_mv[2][k];
            const double mx = E ? s_me[0][k] : 0.0, my = E ? s_me[1][k] : 0.0, mz = E ? s_me[2][k] : 0.0;
            double ax[P], ay[P], az[P], ak[P];
            x2e_geom<P>(px, py, pz, q, ax, ay, az, ak, hit);
#pragma unroll
            for (int h = 0; h < P; h++) {
                const double dx = ax[h], dy = ay[h], dz = az[h], k1 = ak[h], ir2 = k1 * k1, k2 = k1 * ir2;
                if (V) v[h] += (vx * dx + vy * dy + vz * dz) * k2;
                if (E) {
                    const double c3 = 3.0 * (mx * dx + my * dy + mz * dz) * (k2 * ir2);
                    ex[h] += c3 * dx - mx * k2;
                    ey[h] += c3 * dy - my * k2;
                    ez[h] += c3 * dz - mz * k2;
                }
            }
        }
    }
#pragma unroll
    for (int h = 0; h < P; h++) {
        const int j = j0 + h * kBlock;
        if (j < n) part[(long)blockIdx.y * n + j] = make_double4(v[h], ex[h], ey[h], ez[h]);
    }
    if (hit) *bad = 1;
}

// kXfQ groups of kXfPts threads per workgroup of kXfPts points: group q adds
// every kXfQ-th partial, group 0 the group results in a fixed order.
constexpr int kXfQ = 16, kXfPts = kBlock / kXfQ;
__global__ __launch_bounds__(kBlock) void k_x2e_finalize(int n, int nparts, const double4 *__restrict__ part,
                                                         double4 *__restrict__ out) {
    __shared__ double4 sh[kXfQ - 1][kXfPts];
    const int q = threadIdx.x / kXfPts, li = threadIdx.x % kXfPts;
    const int j = blockIdx.x * kXfPts + li;
    double4 a = make_double4(0.0, 0.0, 0.0, 0.0);
    auto add = [&](const double4 &p) {
        a.x += p.x;
        a.y += p.y;
        a.z += p.z;
        a.w += p.w;
    };
    if (j < n)
        for (int s = q; s < nparts; s += kXfQ) add(part[(long)s * n + j]);
    if (q > 0) sh[q - 1][li] = a;
    __syncthreads();
    if (q != 0 || j >= n) return;
    for (int g = 0; g < kXfQ - 1; g++) add(sh[g][li]);
    out[j] = a;
}

// Points per thread: two from 2,048 points, four from 16,384, where the source
// splits still give several workgroups per CU.  Up to kX2eNoAllocMaxPoints the
// splits are those of one point per thread, which bounds the partial sums of the
// no-allocation entry.
constexpr int kX2eNoAllocMaxPoints = 8192;
static int x2e_points(int n) { return n >= 16384 ? 4 : (n >= 2048 ? 2 : 1); }
static int x2e_point_blocks(int n) { return (n + kBlock * x2e_points(n) - 1) / (kBlock * x2e_points(n)); }

int x2e_splits(int n, int nsrc) {
    const int pb = x2e_point_blocks(n), pf = n > kX2eNoAllocMaxPoints ? pb : (n + kBlock - 1) / kBlock;
    // two workgroups per CU and not a few more: a third on some CUs sets the time (20,000
    // points, 5,004 charges, field: 520 workgroups 118 us, 500 95)
    const int thin = std::min((nsrc + 15) / 16, std::max(1, 512 / pb));
    const int full = std::min((nsrc + kBlock - 1) / kBlock, (2048 + pf - 1) / pf);
    return std::max(1, std::max(thin, full));
}

// f with the compile-time choice of potential, field or both and of the points per thread.
template <typename F>
static void x2e_dispatch(int n, bool v, bool e, F &&f) {
    auto points = [&](auto wv, auto we) {
        const int p = x2e_points(n);
        if (p == 4) f(wv, we, std::integral_constant<int, 4>{});
        else if (p == 2) f(wv, we, std::integral_constant<int, 2>{});
        else f(wv, we, std::integral_constant<int, 1>{});
    };
    if (v && e) points(std::true_type{}, std::true_type{});
    else if (v) points(std::true_type{}, std::false_type{});
    else points(std::false_type{}, std::true_type{});
    HIP_CHECK(hipGetLastError());
}

void launch_x2e(hipStream_t st, int n, const double *cext, bool mm, bool pol, bool amoeba, int ld, int nmm,
                const double4 *ms, const double *mq, int npol, const double4 *ps, const double *ipd, bool want_v,
                bool want_e, double4 *part, int smm, int spol, double4 *out, int *bad) {
    if (n == 0) return;
    const int pb = x2e_point_blocks(n);
    int off = 0;
    if (mm && nmm > 0) {
        const int chunk = (nmm + smm - 1) / smm;
        x2e_dispatch(n, want_v, want_e, [&](auto v, auto e, auto p) {
            constexpr bool V = decltype(v)::value, E = decltype(e)::value;
            constexpr int P = decltype(p)::value;
            if (ld == 10)
                hipLaunchKernelGGL((k_m2e<10, V, E, P>), dim3(pb, smm), dim3(kBlock), 0, st, n, cext, nmm, chunk, ms,
                                   mq, part, bad);
            else
                hipLaunchKernelGGL((k_m2e<1, V, E, P>), dim3(pb, smm), dim3(kBlock), 0, st, n, cext, nmm, chunk, ms,
                                   mq, part, bad);
        });
        off = smm;
    }
    if (pol && npol > 0) {
        const int chunk = (npol + spol - 1) / spol;
        x2e_dispatch(n, want_v, want_e, [&](auto v, auto e, auto p) {
            constexpr bool V = decltype(v)::value, E = decltype(e)::value;
            constexpr int P = decltype(p)::value;
            hipLaunchKernelGGL((k_d2e<V, E, P>), dim3(pb, spol), dim3(kBlock), 0, st, n, cext, npol, chunk, ps, ipd,
                               amoeba ? 1 : 0, part + (long)off * n, bad);
        });
        off += spol;
    }
    hipLaunchKernelGGL(k_x2e_finalize, dim3((n + kXfPts - 1) / kXfPts), dim3(kBlock), 0, st, n, off, part, out);
    HIP_CHECK(hipGetLastError());
}

// ------------------------------------------------ no-allocation variant
// ommp_amd_field_mmpol2ext_noalloc keeps everything beyond its inputs and
// outputs in one file-scope device array per GPU, `scratch`: the external
// points and the caller's field (copied in), the per-split partial sums, the
// summed result and the coincident-point flag.  Split counts are those of the
// allocating entry (x2e_splits), so both give the same bits.  For n points
// each source kind takes at most ceil(2048 / ceil(n / 256)) splits, or
// 512 / ceil(n / 512) or 512 / ceil(n / 256), which is fewer, so the
// partial sums need at most 2 (2048 + ceil(n / 256) - 1) 256 double4.
// Every call on a GPU uses that GPU's array: calls that overlap on one GPU
// (other host threads, other streams) race; each call waits for its own work.
constexpr long kX2eNoAllocMaxParts = 2L * (2048 + (kX2eNoAllocMaxPoints + kBlock - 1) / kBlock - 1) * kBlock;
constexpr size_t kScrPart = 0;
constexpr size_t kScrOut = kScrPart + sizeof(double4) * kX2eNoAllocMaxParts;
constexpr size_t kScrC = kScrOut + sizeof(double4) * kX2eNoAllocMaxPoints;
constexpr size_t kScrE = kScrC + sizeof(double) * 3 * kX2eNoAllocMaxPoints;
constexpr size_t kScrBad = kScrE + sizeof(double) * 3 * kX2eNoAllocMaxPoints;
constexpr size_t kScrBytes = kScrBad + 256;
static_assert(kScrOut % 256 == 0 && kScrC % 256 == 0 && kScrE % 256 == 0 && kScrBad % 256 == 0,
              "scratch sub-buffers stay 256-byte aligned");

static __device__ __align__(256) unsigned char scratch[kScrBytes];

int x2e_noalloc_max_points() { return kX2eNoAllocMaxPoints; }
size_t x2e_noalloc_scratch_bytes() { return kScrBytes; }

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
unsigned char *g_scratch_ptr[kMaxDevices] = {};

// Device address of `scratch` on `device` (each GPU holds its own copy),
// looked up once per device with that device current.
unsigned char *scratch_on(int device) {
    if (device < 0 || device >= kMaxDevices) fatal("Device index out of range for the no-allocation entry point");
    std::lock_guard<std::mutex> g(g_scratch_mu);
    if (!g_scratch_ptr[device]) {
        int cur = 0;
        HIP_CHECK(hipGetDevice(&cur));
        if (cur != device) HIP_CHECK(hipSetDevice(device));
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (cur != device) HIP_CHECK(hipSetDevice(cur));
        HIP_CHECK(e);
        if (!p) fatal("No device address for the scratch array of the no-allocation entry point");
        g_scratch_ptr[device] = static_cast<unsigned char *>(p);
    }
    return g_scratch_ptr[device];
}

__global__ void k_zero_flag(int *__restrict__ flag) {
    if (threadIdx.x == 0) *flag = 0;
}

// e[j] += field part of out[j] (out = V, Ex, Ey, Ez)
__global__ __launch_bounds__(kBlock) void k_add_x2e_field(int n, const double4 *__restrict__ out,
                                                          double *__restrict__ e) {
    const int j = blockIdx.x * kBlock + threadIdx.x;
    if (j >= n) return;
    const double4 o = out[j];
    e[3L * j] += o.y;
    e[3L * j + 1] += o.z;
    e[3L * j + 2] += o.w;
}

}  // namespace

int x2e_field_noalloc(hipStream_t st, int device, int n, const double *cext, bool mm, bool pol, bool amoeba, int ld,
                      int nmm, const double4 *ms, const double *mq, int npol, const double4 *ps, const double *ipd,
                      double *e) {
    if (n <= 0) return 0;
    if (n > kX2eNoAllocMaxPoints)
        fatal("ommp_amd_field_mmpol2ext_noalloc takes at most " + std::to_string(kX2eNoAllocMaxPoints) +
              " external points per call (" + std::to_string(n) + " requested)");
    const int smm = mm ? x2e_splits(n, nmm) : 0, spol = pol ? x2e_splits(n, npol) : 0;
    if ((long)(smm + spol) * n > kX2eNoAllocMaxParts) fatal("Scratch of the no-allocation entry point too small");
    unsigned char *base = scratch_on(device);
    double4 *part = reinterpret_cast<double4 *>(base + kScrPart);
    double4 *out = reinterpret_cast<double4 *>(base + kScrOut);
    double *c = reinterpret_cast<double *>(base + kScrC);
    double *es = reinterpret_cast<double *>(base + kScrE);
    int *bad = reinterpret_cast<int *>(base + kScrBad);
    HIP_CHECK(hipMemcpyAsync(c, cext, sizeof(double) * 3L * n, hipMemcpyHostToDevice, st));
    HIP_CHECK(hipMemcpyAsync(es, e, sizeof(double) * 3L * n, hipMemcpyHostToDevice, st));
    hipLaunchKernelGGL(k_zero_flag, dim3(1), dim3(64), 0, st, bad);
    HIP_CHECK(hipGetLastError());
    launch_x2e(st, n, c, mm, pol, amoeba, ld, nmm, ms, mq, npol, ps, ipd, false, true, part, smm, spol, out, bad);
    hipLaunchKernelGGL(k_add_x2e_field, dim3((n + kBlock - 1) / kBlock), dim3(kBlock), 0, st, n, out, es);
    HIP_CHECK(hipGetLastError());
    int bad_h = 0;
    HIP_CHECK(hipMemcpyAsync(e, es, sizeof(double) * 3L * n, hipMemcpyDeviceToHost, st));
    HIP_CHECK(hipMemcpyAsync(&bad_h, bad, sizeof(int), hipMemcpyDeviceToHost, st));
    HIP_CHECK(hipStreamSynchronize(st));
    return bad_h;
}

}  // namespace ommp
