// Far field on the matrix cores (far.h).  A T matvec is six launches:
//   k_far_sort    the dipoles in the order of the sorted sites;
//   k_far_p2m     moments of every occupied cell of every level straight from its
//                 sites (no translation upwards: a level is one more pass over the
//                 stored basis functions, 16 KB per 64 sites);
//   k_far_m2l     the transfer: a group of cells with the same interaction list
//                 takes one offset at a time, the source cells at that offset being
//                 the columns of K(offset) M on v_mfma_{f64,f32}_16x16x4 tiles, two
//                 sets of 16 columns per loaded matrix; the four waves of a
//                 workgroup and nsplit workgroups take different offsets;
//   k_far_field   the sums of the splits, as the expansion of the field (its
//                 gradient form) of every cell;
//   k_far_near    per T sites of a leaf: the 27 leaves around it pair by pair, the
//                 field expansions of all levels, the screened-pair corrections, the
//                 diagonal and the y.x partial;
//   k_far_dots    the workgroups' y.x partials as kFarDots sums.
// Every sum has a fixed order.
//
// The FP64 form replaces, for orders up to 8, a chain of complex kernels (one
// thread per coefficient, both factors of every product from LDS, a launch per
// level up and down, the near field as 27 partial fields): 3.1 -> 0.56 ms per
// matvec of one dipole set at 120,000 sites, order 8 (near field 0.27, transfer
// 0.20, moments 0.06).
// What bounds it: the near field's vector ALUs and the transfer's matrix rate.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "far.h"
#include "pair_math.h"

namespace ommp {

namespace {

template <typename R> struct Mat;
template <> struct Mat<double> {
    typedef double acc __attribute__((ext_vector_type(4)));
    typedef double vec __attribute__((ext_vector_type(2)));
    static __device__ __forceinline__ acc fma(double a, double b, acc c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int q, int e) { return q + 4 * e; }
};
template <> struct Mat<float> {
    typedef float acc __attribute__((ext_vector_type(4)));
    typedef float vec __attribute__((ext_vector_type(4)));
    static __device__ __forceinline__ acc fma(float a, float b, acc c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int q, int e) { return 4 * q + e; }
};

__device__ __forceinline__ void degree_of(int i, int &n, int &m, bool &im) {
    n = 1;
    while ((n + 1) * (n + 1) - 1 <= i) n++;
    const int r = i - (n * n - 1);
    m = (r + 1) / 2;
    im = r > 0 && (r & 1) == 0;
}

// i^e z
__device__ __forceinline__ double2 turn(int e, double2 z) {
    switch (e & 3) {
        case 0: return z;
        case 1: return make_double2(-z.y, z.x);
        case 2: return make_double2(-z.x, -z.y);
        default: return make_double2(z.y, -z.x);
    }
}

__device__ __forceinline__ int level_of(const FarLevels &lv, long c) {
    int l = 2;
    while (l < lv.levels && c >= lv.off[l + 1] - lv.off[2]) l++;
    return l;
}

__device__ __forceinline__ bool all_done(const CgState *skip, int M) {
    if (!skip) return false;
    bool all = true;
    for (int m = 0; m < M; m++) all = all && skip[m].done;
    return all;
}

// ------------------------------------------------------------- transfer
// Real moments in units of the cell side, from the complex ones.
__global__ __launch_bounds__(kBlock) void k_far_moments(FarLevels lv, int p, int nc, long cells,
                                                        const double2 *__restrict__ mexp, double *__restrict__ mom,
                                                        double *__restrict__ mom0) {
    const long t = (long)blockIdx.x * kBlock + threadIdx.x;
    const long c = t / nc;
    const int i = (int)(t - c * nc);
    if (c >= cells) return;
    const int ncoef = (p + 1) * (p + 1);
    double v = 0.0;
    if (i < ncoef - 1) {
        int n, m;
        bool im;
        degree_of(i, n, m, im);
        const double ih = (double)(1 << level_of(lv, c)) / lv.side;
        double f = ih;
        for (int k = 1; k < n; k++) f *= ih;
        // i^m O_n^m = C - i S
        const double2 z = turn(m, mexp[(lv.off[2] + c) * ncoef + n * n + n + m]);
        v = f * (im ? -z.y : z.x);
    }
    mom[t] = v;
    if (i == 0) mom0[c] = mexp[(lv.off[2] + c) * ncoef].x;
}

template <typename R, int M, int RT, bool MONO>
__global__ __launch_bounds__(kBlock) void k_far_m2l(FarLevels lv, int nsplit, const R *__restrict__ zero,
                                                    const int *__restrict__ gcell, const int *__restrict__ glevel,
                                                    const int *__restrict__ cnt_src, const R *__restrict__ K,
                                                    const R *__restrict__ K0, const R *__restrict__ mom,
                                                    const R *__restrict__ mom0, R *__restrict__ part,
                                                    const CgState *__restrict__ skip) {
    using V = typename Mat<R>::vec;
    constexpr int NC = 16 * RT, PER = NC / 4, VE = 16 / sizeof(R), NV = PER / VE, TW = 16 / M;
    if (all_done(skip, M)) return;
    __shared__ R s_sum[32][NC + 1];
    const int tid = threadIdx.x, lane = tid & 63, col = lane & 15, q = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l = glevel[blockIdx.x];
    if (l == 0) return;
    const int ns = 1 << l;
    const long base = lv.off[l] - lv.off[2];
    // columns of the two sets: cell col / M, dipole column col % M
    int tx[2], ty[2], tz[2];
    bool tgt[2];
#pragma unroll
    for (int s = 0; s < 2; s++) {
        const int c = gcell[blockIdx.x * 2 * TW + s * TW + col / M];
        tgt[s] = c >= 0;
        tx[s] = c & (ns - 1);
        ty[s] = c >> l & (ns - 1);
        tz[s] = c >> 2 * l;
    }
    const int first = gcell[blockIdx.x * 2 * TW];  // never -1; all cells share its place in the parent
    const int lox = -2 - (first & 1), loy = -2 - (first >> l & 1), loz = -2 - (first >> 2 * l & 1);
    typename Mat<R>::acc acc[2][RT];
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
        for (int r = 0; r < RT; r++) acc[s][r] = R(0);
    for (int o = blockIdx.y * 4 + w; o < 216; o += 4 * nsplit) {
        const int dx = lox + o % 6, dy = loy + o / 6 % 6, dz = loz + o / 36;
        if (abs(dx) <= 1 && abs(dy) <= 1 && abs(dz) <= 1) continue;
        long src[2];
        const V *xv[2];
        bool any = false;
#pragma unroll
        for (int s = 0; s < 2; s++) {
            const int x = tx[s] + dx, y = ty[s] + dy, z = tz[s] + dz;
            bool ok = tgt[s] && x >= 0 && y >= 0 && z >= 0 && x < ns && y < ns && z < ns;
            const int c = ok ? (z * ns + y) * ns + x : 0;
            ok = ok && cnt_src[lv.off[l] + c] != 0;
            src[s] = ok ? base + c : -1;
            xv[s] = reinterpret_cast<const V *>((ok ? mom + ((base + c) * M + col % M) * NC : zero) + q * PER);
            any = any || ok;
        }
        if (!__ballot(any)) continue;
        const int ko = (dz + 3) * 49 + (dy + 3) * 7 + dx + 3;
        const V *a = reinterpret_cast<const V *>(K) + (long)ko * RT * NV * 64 + lane;
#pragma unroll 2
        for (int v = 0; v < NV; v++) {
            const V x0 = xv[0][v], x1 = xv[1][v];
            V k[RT];
#pragma unroll
            for (int r = 0; r < RT; r++) k[r] = a[(r * NV + v) * 64];
#pragma unroll
            for (int e = 0; e < VE; e++)
#pragma unroll
                for (int r = 0; r < RT; r++) {
                    acc[0][r] = Mat<R>::fma(k[r][e], x0[e], acc[0][r]);
                    acc[1][r] = Mat<R>::fma(k[r][e], x1[e], acc[1][r]);
                }
        }
        if (MONO) {
            const R x0 = q == 0 && src[0] >= 0 ? mom0[src[0]] : R(0), x1 = q == 0 && src[1] >= 0 ? mom0[src[1]] : R(0);
#pragma unroll
            for (int r = 0; r < RT; r++) {
                const R k = K0[((long)ko * RT + r) * 64 + lane];
                acc[0][r] = Mat<R>::fma(k, x0, acc[0][r]);
                acc[1][r] = Mat<R>::fma(k, x1, acc[1][r]);
            }
        }
    }
    // the waves' sums in wave order
    for (int t = 0; t < 4; t++) {
        if (w == t)
#pragma unroll
            for (int s = 0; s < 2; s++)
#pragma unroll
                for (int r = 0; r < RT; r++)
#pragma unroll
                    for (int e = 0; e < 4; e++) {
                        const int row = 16 * r + Mat<R>::row(q, e);
                        const R v = acc[s][r][e];
                        s_sum[16 * s + col][row] = t == 0 ? v : s_sum[16 * s + col][row] + v;
                    }
        __syncthreads();
    }
    R *o = part + ((long)blockIdx.y * gridDim.x + blockIdx.x) * 32 * NC;
    for (int e = tid; e < 32 * NC; e += kBlock) o[e] = s_sum[e / NC][e % NC];
}

__global__ __launch_bounds__(kBlock) void k_far_zero(long n, double2 *__restrict__ v) {
    const long k = (long)blockIdx.x * kBlock + threadIdx.x;
    if (k < n) v[k] = make_double2(0.0, 0.0);
}

// Complex local expansions of a group's cells from the splits' sums, in the tree's
// units: L_j^0 = (-1)^j a, L_j^k = i^k (-1)^j (a - i b) / 2 and L_j^-k = (-1)^k
// conj(L_j^k) for the coefficients a of Re and b of Im Phi_j^k.
__global__ __launch_bounds__(kBlock) void k_far_locals(FarLevels lv, int p, int nc, int nsplit, int ngroups,
                                                       const int *__restrict__ gcell, const int *__restrict__ glevel,
                                                       const double *__restrict__ part, double2 *__restrict__ loc) {
    const int npair = (p + 1) * (p + 2) / 2, slot = blockIdx.x, g = slot / 32, col = slot % 32;
    const int cell = gcell[slot];
    if (cell < 0) return;
    const int l = glevel[g], ncoef = (p + 1) * (p + 1);
    for (int r = threadIdx.x; r < npair; r += kBlock) {
        int j = 0;
        while ((j + 1) * (j + 2) / 2 <= r) j++;
        const int k = r - j * (j + 1) / 2;
        double a = 0.0, b = 0.0;
        if (j > 0) {
            const double *s = part + ((long)g * 32 + col) * nc + j * j - 1 + (k == 0 ? 0 : 2 * k - 1);
            for (int q = 0; q < nsplit; q++) {
                a += s[(long)q * ngroups * 32 * nc];
                if (k > 0) b += s[(long)q * ngroups * 32 * nc + 1];
            }
            const double ih = (double)(1 << l) / lv.side;
            double f = (j & 1) ? -ih : ih;
            for (int m = 0; m < j; m++) f *= ih;
            if (k > 0) f *= 0.5;
            a *= f;
            b *= f;
        }
        double2 *out = loc + (lv.off[l] + cell) * ncoef + j * j + j;
        const double2 v = turn(k, make_double2(a, -b));
        out[k] = v;
        if (k > 0) out[-k] = (k & 1) ? make_double2(-v.x, v.y) : make_double2(v.x, -v.y);
    }
}

// ------------------------------------------------------------ T matvec
// B_i(v / h) of degree < p of every sorted site at every level, one thread per
// (site, level, m).
template <typename R>
__global__ __launch_bounds__(kBlock) void k_far_basis(FarLevels lv, int p, int npol, const int *__restrict__ order,
                                                      const int *__restrict__ leaf,
                                                      const double4 *__restrict__ ps, R *__restrict__ basis) {
    const long t = (long)blockIdx.x * kBlock + threadIdx.x;
    const int site = (int)(t % npol), m = (int)(t / npol % p), l = 2 + (int)(t / npol / p);
    if (l > lv.levels) return;
    const double4 s = ps[order[site]];
    const int ns = 1 << l;
    const double ih = ns / lv.side;
    const int lf = leaf[site], mask = (1 << lv.levels) - 1, up = lv.levels - l;
    double v[3] = {s.x, s.y, s.z};
    for (int c = 0; c < 3; c++)
        v[c] = (v[c] - lv.origin[c]) * ih - (((lf >> c * lv.levels & mask) >> up) + 0.5);
    const double r2 = v[0] * v[0] + v[1] * v[1] + v[2] * v[2];
    double2 cur = make_double2(1.0, 0.0);
    for (int k = 1; k <= m; k++) {
        const double f = 1.0 / (2.0 * k);
        cur = make_double2(f * (cur.x * v[0] - cur.y * v[1]), f * (cur.x * v[1] + cur.y * v[0]));
    }
    R *out = basis + ((long)(l - 2) * npol + site) * kFarBasis;
    double2 before = make_double2(0.0, 0.0);
    for (int n = m; n < p; n++) {
        if (m == 0) out[n * n] = (R)cur.x;
        else {
            out[n * n + 2 * m - 1] = (R)cur.x;
            out[n * n + 2 * m] = (R)cur.y;
        }
        // Phi_{n+1}^m = ((2n + 1) z Phi_n^m - r^2 Phi_{n-1}^m) / ((n + 1)^2 - m^2), z Phi_m^m for n = m
        const double a = n == m ? v[2] : (2.0 * n + 1.0) * v[2] / ((n + 1.0) * (n + 1.0) - (double)m * m);
        const double b = n == m ? 0.0 : r2 / ((n + 1.0) * (n + 1.0) - (double)m * m);
        const double2 next = make_double2(a * cur.x - b * before.x, a * cur.y - b * before.y);
        before = cur;
        cur = next;
    }
    if (m == 0)
        for (int i = p * p; i < kFarBasis; i++) out[i] = R(0);
}

// The dipoles in the order of the sorted sites (order given) or already in it: both
// the moments and the near field then read neighbours as neighbours (gathered there, 64
// lanes of 24 bytes each, they made the moments of 60,000 sites, two columns in FP32, 74
// instead of 32 us and the near field 397 instead of 353; this pass takes 5).
template <typename R>
__global__ __launch_bounds__(kBlock) void k_far_sort(int npol, const int *__restrict__ order,
                                                     const R *__restrict__ adamp, const double *__restrict__ x,
                                                     long xstride, typename V4<R>::t *__restrict__ xs,
                                                     const CgState *__restrict__ skip, int M) {
    if (all_done(skip, M)) return;
    const int t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= npol) return;
    const double *v = x + blockIdx.y * xstride + 3L * (order ? order[t] : t);
    typename V4<R>::t o;
    o.x = (R)v[0];
    o.y = (R)v[1];
    o.z = (R)v[2];
    o.w = adamp[t];
    xs[(long)blockIdx.y * npol + t] = o;
}

// Moments of one cell (blockIdx.x: a place in the groups), added to init where
// given: sums A_c,i = sum mu_c B_i
// over its sites, one basis function per lane, then
//   M_n^m (Re) = (1 / h) [(Ax,c^{m-1} - Ax,c^{m+1}) / 2 - (Ay,s^{m-1} + Ay,s^{m+1}) / 2 + Az,c^m]_{n-1}
//   M_n^m (Im) = (1 / h) [(Ax,s^{m-1} - Ax,s^{m+1}) / 2 + (Ay,c^{m-1} + Ay,c^{m+1}) / 2 + Az,s^m]_{n-1}
//   M_n^0      = (1 / h) [-Ax,c^1 - Ay,s^1 + Az,c^0]_{n-1}
// from the derivatives of Phi.
constexpr int kP2mThreads = 512, kP2mWaves = kP2mThreads / 64;
template <typename R, int M>
__global__ __launch_bounds__(kP2mThreads) void k_far_p2m(FarLevels lv, int p, int nc, int npol, int width,
                                                    const int *__restrict__ gcell, const int *__restrict__ glevel,
                                                    const int *__restrict__ leaf_start,
                                                    const R *__restrict__ basis,
                                                    const typename V4<R>::t *__restrict__ xs,
                                                    const R *__restrict__ init,
                                                    R *__restrict__ mom,
                                                    const CgState *__restrict__ skip) {
    if (all_done(skip, M)) return;
    const int cell = gcell[blockIdx.x];
    if (cell < 0) return;
    __shared__ R s_a[kP2mWaves][M][3][kFarBasis];
    const int l = glevel[blockIdx.x / width], k = lv.levels - l, ns = 1 << l, nl = 1 << lv.levels;
    const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int cx = cell & (ns - 1), cy = cell >> l & (ns - 1), cz = cell >> 2 * l;
    const R *bas = basis + (long)(l - 2) * npol * kFarBasis + lane;
    R a[M][3];
#pragma unroll
    for (int m = 0; m < M; m++) a[m][0] = a[m][1] = a[m][2] = R(0);
    // the runs of leaves of this cell; the waves share the sites of each
    for (int run = 0; run < 1 << 2 * k; run++) {
        const int row = (((cz << k) + (run >> k)) * nl + (cy << k) + (run & ((1 << k) - 1))) * nl + (cx << k);
        const int t1 = leaf_start[row + (1 << k)];
#pragma unroll 8
        for (int t = leaf_start[row] + w; t < t1; t += kP2mWaves) {
            const R b = bas[(long)t * kFarBasis];
#pragma unroll
            for (int m = 0; m < M; m++) {
                const typename V4<R>::t v = xs[(long)m * npol + t];
                a[m][0] += v.x * b;
                a[m][1] += v.y * b;
                a[m][2] += v.z * b;
            }
        }
    }
#pragma unroll
    for (int m = 0; m < M; m++)
#pragma unroll
        for (int c = 0; c < 3; c++) s_a[w][m][c][lane] = a[m][c];
    __syncthreads();
    constexpr int st = M * 3 * kFarBasis;
    for (int e = tid; e < st; e += kP2mThreads) {
        R *s = &s_a[0][0][0][0] + e, v = s[0];
#pragma unroll
        for (int q = 1; q < kP2mWaves; q++) v += s[q * st];
        s[0] = v;
    }
    __syncthreads();
    const R ih = (R)(ns / lv.side);
    const long base = (lv.off[l] - lv.off[2] + cell) * M * nc;
    for (int e = tid; e < M * nc; e += kP2mThreads) {
        const int m0 = e / nc, i = e % nc;
        R v = R(0);
        if (i < (p + 1) * (p + 1) - 1) {
            int n, m;
            bool im;
            degree_of(i, n, m, im);
            const R(*A)[kFarBasis] = s_a[0][m0];
            const int d = (n - 1) * (n - 1);
            // Re / Im of order q of degree n - 1; zero past the degree and for Im of order 0
            auto re = [&](int c, int q) { return q <= n - 1 ? A[c][d + (q == 0 ? 0 : 2 * q - 1)] : R(0); };
            auto imag = [&](int c, int q) { return q >= 1 && q <= n - 1 ? A[c][d + 2 * q] : R(0); };
            if (m == 0) v = re(2, 0) - re(0, 1) - imag(1, 1);
            else if (!im)
                v = R(0.5) * (re(0, m - 1) - re(0, m + 1)) - R(0.5) * (imag(1, m - 1) + imag(1, m + 1)) + re(2, m);
            else
                v = R(0.5) * (imag(0, m - 1) - imag(0, m + 1)) + R(0.5) * (re(1, m - 1) + re(1, m + 1)) + imag(2, m);
            v *= ih;
        }
        mom[base + e] = init ? init[base + e] + v : v;
    }
}

// Field expansion of one cell: the splits' sums l, then G with E_c = sum_i B_i G_c,i,
// the transpose of the derivatives above times -1 / h^2.
template <typename R, int M>
__global__ __launch_bounds__(kBlock) void k_far_field(FarLevels lv, int p, int nc, int nsplit, int ngroups, int width,
                                                      const int *__restrict__ gcell, const int *__restrict__ glevel,
                                                      const R *__restrict__ part, R *__restrict__ grad,
                                                      const CgState *__restrict__ skip) {
    if (all_done(skip, M)) return;
    const int slot = blockIdx.x, g = slot / width;
    const int cell = gcell[slot];
    if (cell < 0) return;
    __shared__ R s_l[M][16 * kFarMaxTiles];
    const int l = glevel[g];
    for (int e = threadIdx.x; e < M * nc; e += kBlock) {
        const R *s = part + ((long)g * 32 + slot % width * M + e / nc) * nc + e % nc;
        R v = R(0);
        for (int q = 0; q < nsplit; q++) v += s[(long)q * ngroups * 32 * nc];
        s_l[e / nc][e % nc] = v;
    }
    __syncthreads();
    const double h = lv.side / (1 << l);
    const R f = (R)(-1.0 / (h * h));
    R *out = grad + (lv.off[l] - lv.off[2] + cell) * M * 3 * kFarBasis;
    for (int e = threadIdx.x; e < M * 3 * kFarBasis; e += kBlock) {
        const int m0 = e / (3 * kFarBasis), c = e / kFarBasis % 3, i = e % kFarBasis;
        R v = R(0);
        if (i < p * p) {
            int n = 0;
            while ((n + 1) * (n + 1) <= i) n++;
            const int r = i - n * n, m = (r + 1) / 2, d = (n + 1) * (n + 1) - 1;  // degree n + 1 in l
            const bool im = r > 0 && (r & 1) == 0;
            const R *L = s_l[m0];
            auto re = [&](int q) { return L[d + (q == 0 ? 0 : 2 * q - 1)]; };
            auto imag = [&](int q) { return q >= 1 ? L[d + 2 * q] : R(0); };
            const R h2 = R(0.5), down = m == 1 ? R(1) : R(0.5);
            if (c == 2) v = im ? imag(m) : re(m);
            else if (c == 0)
                v = im ? h2 * imag(m + 1) - (m >= 2 ? h2 * imag(m - 1) : R(0))
                       : h2 * re(m + 1) - (m >= 1 ? down * re(m - 1) : R(0));
            else
                v = im ? -h2 * re(m + 1) - down * re(m - 1)
                       : h2 * imag(m + 1) + (m >= 2 ? h2 * imag(m - 1) : R(0));
        }
        out[e] = v * f;
    }
}

// T targets of a leaf and its 27 leaves: thread (t, s) meets every (256 / T)-th source
// from the s-th for target t.  Sources pass through LDS, read there by T lanes at once.
// Damped pairs (a few per thread, in half of a wave's steps) are left out of the sweep:
// each thread lists its own within a tile and does them at the tile's end, where the
// exact argument decides (cutoffs as in row_sweep.h); a full list damps in place.
//
// Bound by the vector unit.  One target per thread keeps its data in registers and
// leaves three sums per thread and column to add up.  With the sources over the threads
// instead (as the per-target matvec, which sweeps thousands of them) each of 8 targets'
// sums went over 256 threads: half of the instructions at the 500 sources of a leaf of
// 29 sites.  120,000 sites FP64, one column: 497 -> 267 us (187 of them vector issue);
// FP32, two columns: 20,001 sites 72 -> 53, 60,000 sites in leaves of 171: 353 -> 336
// (292 issue, 37 instructions per pair).
constexpr int kNearCap = 12;  // listed pairs per thread and tile
template <typename R> constexpr int kNearTile = sizeof(R) == 8 ? 256 : 512;  // sources in LDS

template <typename R, int M, bool AMOEBA, int T>
__global__ __launch_bounds__(kBlock) void k_far_near(
    FarLevels lv, int npol, const int2 *__restrict__ blocks, const int *__restrict__ leaf_start,
    const int *__restrict__ order, const typename V4<R>::t *__restrict__ pos, const R *__restrict__ adamp,
    const R *__restrict__ rc2, const typename V4<R>::t *__restrict__ xs, const R *__restrict__ basis,
    const R *__restrict__ grad, const double4 *__restrict__ ps, const double *__restrict__ pa,
    const double *__restrict__ alpha, const int *__restrict__ pp_ri, const int *__restrict__ pp_ci,
    const double *__restrict__ pp_f, const double *__restrict__ x, long xstride, double *__restrict__ y, long ystride,
    int dodiag, double *__restrict__ dotpart, const CgState *__restrict__ skip) {
    using R4 = typename V4<R>::t;
    constexpr int C = 3 * M, NS = kBlock / T, TILE = kNearTile<R>, NB = kFarBasis / NS;
    static_assert(T <= 32 && NB >= 1, "whole slices per wave");
    if (all_done(skip, M)) return;
    __shared__ R4 s_pos[TILE], s_x[M][TILE];
    __shared__ unsigned short s_list[kNearCap][kBlock];
    __shared__ double s_sum[kBlock / 64][T][C], s_dot[T][C];
    const int tid = threadIdx.x, tt = tid % T, sl = tid / T;
    const int leaf = blocks[blockIdx.x].x, t0 = blocks[blockIdx.x].y;
    const int nl = 1 << lv.levels, lx = leaf & (nl - 1), ly = leaf >> lv.levels & (nl - 1), lz = leaf >> 2 * lv.levels;
    const int nt = min(T, leaf_start[leaf + 1] - t0);
    // targets past the leaf's end repeat the last one; their results are not written
    const int ti = t0 + min(tt, nt - 1), site = order[ti];
    const R4 pt = pos[ti];
    const R at = adamp[ti], rc = rc2[site];
    R f[M][3];
#pragma unroll
    for (int m = 0; m < M; m++) f[m][0] = f[m][1] = f[m][2] = R(0);
    // far field of every level: NB basis functions per thread
    for (int l = 2; l <= lv.levels; l++) {
        const int k = lv.levels - l, ns = 1 << l;
        const long cell = lv.off[l] - lv.off[2] + ((long)(lz >> k) * ns + (ly >> k)) * ns + (lx >> k);
        const R *g = grad + cell * C * kFarBasis + sl * NB;
        const R *bas = basis + ((long)(l - 2) * npol + ti) * kFarBasis + sl * NB;
#pragma unroll
        for (int i = 0; i < NB; i++) {
            const R bv = bas[i];
#pragma unroll
            for (int c = 0; c < C; c++) f[c / 3][c % 3] += bv * g[c * kFarBasis + i];
        }
    }
    // near field: nine runs of sites (three leaves along x each)
    int start[9], before[10];
    before[0] = 0;
    const int x0 = max(lx - 1, 0), x1 = min(lx + 1, nl - 1);
#pragma unroll
    for (int r = 0; r < 9; r++) {
        const int yy = ly + r % 3 - 1, zz = lz + r / 3 - 1;
        const bool in = yy >= 0 && yy < nl && zz >= 0 && zz < nl;
        const int row = in ? (zz * nl + yy) * nl : 0;
        start[r] = in ? leaf_start[row + x0] : 0;
        before[r + 1] = before[r] + (in ? leaf_start[row + x1 + 1] - start[r] : 0);
    }
    const int total = before[9];
    for (int tile = 0; tile < total; tile += TILE) {
        const int cnt = min(TILE, total - tile), cntp = (cnt + NS - 1) / NS * NS;
        __syncthreads();
        for (int q = tid; q < cntp; q += kBlock) {
            R4 p, v[M];
            if (q < cnt) {
                int i = start[0] + tile + q;
#pragma unroll
                for (int r = 1; r < 9; r++)
                    if (tile + q >= before[r]) i = start[r] + tile + q - before[r];
                p = pos[i];
#pragma unroll
                for (int m = 0; m < M; m++) v[m] = xs[(long)m * npol + i];
            } else {
                p.x = p.y = p.z = R(1e15);
                p.w = R(1);
#pragma unroll
                for (int m = 0; m < M; m++) {
                    v[m].x = v[m].y = v[m].z = R(0);
                    v[m].w = R(0.39);
                }
            }
            s_pos[q] = p;
#pragma unroll
            for (int m = 0; m < M; m++) s_x[m][q] = v[m];
        }
        __syncthreads();
        int n = 0;
        for (int q = sl; q < cntp; q += NS) {
            const R4 p = s_pos[q];
            R4 v[M];
#pragma unroll
            for (int m = 0; m < M; m++) v[m] = s_x[m][q];
            R dx, dy, dz, k2, k3;
            const bool in = pair_bare<R>(pt, p, dx, dy, dz, k2, k3) < rc;  // the target itself among them
            if (__ballot(in)) {
                if (in) {
                    if (n < kNearCap) {
                        s_list[n++][tid] = (unsigned short)q;
                        k2 = k3 = R(0);
                    } else {
                        R arg;
                        bool near;
                        pair_geom<R, AMOEBA>(pt, at, p, v[0].w, dx, dy, dz, k2, k3, arg, near);
                        pair_damp<R, AMOEBA>(arg, near, k2, k3);
                    }
                }
            }
            pair_accum<R, M>(f, v, dx, dy, dz, k2, k3);
        }
        for (int e = 0; __ballot(e < n); e++) {
            if (e >= n) continue;
            const int q = s_list[e][tid];
            const R4 p = s_pos[q];
            R4 v[M];
#pragma unroll
            for (int m = 0; m < M; m++) v[m] = s_x[m][q];
            R dx, dy, dz, k2, k3, arg;
            bool near;
            pair_geom<R, AMOEBA>(pt, at, p, v[0].w, dx, dy, dz, k2, k3, arg, near);  // 0 for itself
            pair_damp<R, AMOEBA>(arg, near, k2, k3);
            pair_accum<R, M>(f, v, dx, dy, dz, k2, k3);
        }
    }
    // screened pairs (FP64), then the sum over the slices
    double sum[C];
#pragma unroll
    for (int c = 0; c < C; c++) sum[c] = -(double)f[c / 3][c % 3];
    screened_pairs<AMOEBA, M>(site, sl, NS, ps, pa, pp_ri, pp_ci, pp_f, x, xstride, sum);
#pragma unroll
    for (int mask = T; mask < 64; mask <<= 1)
#pragma unroll
        for (int c = 0; c < C; c++) sum[c] += __shfl_xor(sum[c], mask, 64);
    if ((tid & 63) < T) {
#pragma unroll
        for (int c = 0; c < C; c++) s_sum[tid >> 6][tt][c] = sum[c];
    }
    __syncthreads();
    if (tid < T * C) {
        const int t = tid / C, c = tid % C;
        double out = 0.0;
        if (t < nt) {
            const int j = order[t0 + t];
            const double xj = x[c / 3 * xstride + 3L * j + c % 3];
            double v = s_sum[0][t][c];
#pragma unroll
            for (int q = 1; q < kBlock / 64; q++) v += s_sum[q][t][c];
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
        for (int t = 0; t < T; t++) d += (s_dot[t][3 * tid] + s_dot[t][3 * tid + 1]) + s_dot[t][3 * tid + 2];
        dotpart[tid * (long)gridDim.x + blockIdx.x] = d;
    }
}

// The workgroups' y.x partials of column blockIdx.y as kFarDots sums, in a fixed
// order: the tens of thousands of a large system are read by every workgroup of
// the CG update (120,000 sites: 36 us of it, 6 us + 4 us with this).
__global__ __launch_bounds__(kBlock) void k_far_dots(int n, const double *__restrict__ dots,
                                                     double *__restrict__ out, const CgState *__restrict__ skip,
                                                     int M) {
    if (all_done(skip, M)) return;
    __shared__ double sh[4];
    double v = 0.0;
    for (int i = blockIdx.x * kBlock + threadIdx.x; i < n; i += kFarDots * kBlock) v += dots[(long)blockIdx.y * n + i];
    v = block_sum_all(v, sh);
    if (threadIdx.x == 0) out[blockIdx.y * kFarDots + blockIdx.x] = v;
}

template <typename R>
void sort(hipStream_t st, const FarDev<R> &f, const int *order, int M, const double *x, long xs, const CgState *skip) {
    hipLaunchKernelGGL(k_far_sort<R>, dim3((unsigned)((f.npol + kBlock - 1) / kBlock), M), dim3(kBlock), 0, st, f.npol,
                       order, f.a, x, xs, f.xs, skip, M);
    HIP_CHECK(hipGetLastError());
}

template <typename R, int M, bool MONO>
void m2l(hipStream_t st, const FarDev<R> &f, const FarGroups &tgt, const int *cnt_src, const R *mom,
         const CgState *skip) {
    const dim3 grid(tgt.n, f.nsplit), block(kBlock);
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, block, 0, st, f.lv, f.nsplit, f.zero, tgt.cell, tgt.level, cnt_src,
                           f.K, f.K0, mom, f.mom0, f.part, skip);
        HIP_CHECK(hipGetLastError());
    };
    switch (f.nc / 16) {
        case 1: go(k_far_m2l<R, M, 1, MONO>); break;
        case 2: go(k_far_m2l<R, M, 2, MONO>); break;
        case 3: go(k_far_m2l<R, M, 3, MONO>); break;
        case 4: go(k_far_m2l<R, M, 4, MONO>); break;
        case 5: go(k_far_m2l<R, M, 5, MONO>); break;
        default: fatal("Internal error: expansion order of the far-field transfer");
    }
}

template <typename R, int M, bool AMOEBA>
void matvec_t(hipStream_t st, const FarDev<R> &f, const int *cnt, const double4 *ps64, const double *pa64,
              const double *alpha, const CsrDev &pp, const double *x, long xs, double *y, long ys, bool dodiag,
              double *dotpart, const CgState *skip) {
    const int places = f.groups.n * f.groups.width;
    sort<R>(st, f, f.order, M, x, xs, skip);
    if (f.groups.n > 0) {
        hipLaunchKernelGGL((k_far_p2m<R, M>), dim3(places), dim3(kP2mThreads), 0, st, f.lv, f.p, f.nc, f.npol,
                           f.groups.width, f.groups.cell, f.groups.level, f.leaf_start, f.basis, f.xs,
                           (const R *)nullptr, f.mom, skip);
        HIP_CHECK(hipGetLastError());
        m2l<R, M, false>(st, f, f.groups, cnt, f.mom, skip);
        hipLaunchKernelGGL((k_far_field<R, M>), dim3(places), dim3(kBlock), 0, st, f.lv, f.p, f.nc, f.nsplit,
                           f.groups.n, f.groups.width, f.groups.cell, f.groups.level, f.part, f.grad, skip);
        HIP_CHECK(hipGetLastError());
    }
    auto near = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, dim3(f.nblocks), dim3(kBlock), 0, st, f.lv, f.npol, f.blocks, f.leaf_start, f.order,
                           f.pos, f.a, f.rc2, f.xs, f.basis, f.grad, ps64, pa64, alpha, pp.ri, pp.ci, pp.f, x, xs, y,
                           ys, (int)dodiag, dotpart ? f.dots : nullptr, skip);
    };
    if (f.near == 16) near(k_far_near<R, M, AMOEBA, 16>);
    else near(k_far_near<R, M, AMOEBA, 32>);
    if (dotpart)
        hipLaunchKernelGGL(k_far_dots, dim3(kFarDots, M), dim3(kBlock), 0, st, f.nblocks, f.dots, dotpart, skip, M);
    HIP_CHECK(hipGetLastError());
}

}  // namespace

void far_launch_moments(hipStream_t st, const FarDev<double> &f, const double2 *mexp) {
    const long nm = f.cells * f.nc;
    hipLaunchKernelGGL(k_far_moments, dim3((unsigned)((nm + kBlock - 1) / kBlock)), dim3(kBlock), 0, st, f.lv, f.p,
                       f.nc, f.cells, mexp, f.mom_static, f.mom0);
    HIP_CHECK(hipGetLastError());
}

void far_launch_locals(hipStream_t st, const FarDev<double> &f, const FarGroups &tgt, const FarGroups &src,
                       const int *cnt_src, bool with_static, const double *dip, double2 *loc) {
    const long nl = f.cells * (f.p + 1) * (f.p + 1);
    const double *mom = with_static && !dip ? f.mom_static : f.mom;
    hipLaunchKernelGGL(k_far_zero, dim3((unsigned)((nl + kBlock - 1) / kBlock)), dim3(kBlock), 0, st, nl,
                       loc + f.lv.off[2] * (f.p + 1) * (f.p + 1));
    if (dip && src.n > 0) {
        sort<double>(st, f, nullptr, 1, dip, 0L, nullptr);
        hipLaunchKernelGGL((k_far_p2m<double, 1>), dim3(src.n * src.width), dim3(kP2mThreads), 0, st, f.lv, f.p, f.nc,
                           f.npol, src.width, src.cell, src.level, f.leaf_start, f.basis, f.xs,
                           with_static ? f.mom_static : nullptr, f.mom, (const CgState *)nullptr);
    }
    HIP_CHECK(hipGetLastError());
    if (tgt.n == 0) return;
    if (with_static) m2l<double, 1, true>(st, f, tgt, cnt_src, mom, nullptr);
    else m2l<double, 1, false>(st, f, tgt, cnt_src, mom, nullptr);
    hipLaunchKernelGGL(k_far_locals, dim3(tgt.n * tgt.width), dim3(kBlock), 0, st, f.lv, f.p, f.nc, f.nsplit, tgt.n,
                       tgt.cell, tgt.level, f.part, loc);
    HIP_CHECK(hipGetLastError());
}

template <typename R> void far_launch_basis(hipStream_t st, const FarDev<R> &f, const double4 *ps) {
    if (f.lv.levels < 2) return;
    const long n = (long)f.npol * f.p * (f.lv.levels - 1);
    hipLaunchKernelGGL(k_far_basis<R>, dim3((unsigned)((n + kBlock - 1) / kBlock)), dim3(kBlock), 0, st, f.lv, f.p,
                       f.npol, f.order, f.leaf, ps, f.basis);
    HIP_CHECK(hipGetLastError());
}
template void far_launch_basis<double>(hipStream_t, const FarDev<double> &, const double4 *);
template void far_launch_basis<float>(hipStream_t, const FarDev<float> &, const double4 *);

template <typename R>
void far_launch_matvec(hipStream_t st, const FarDev<R> &f, bool amoeba, int M, const int *cnt, const double4 *ps64,
                       const double *pa64, const double *alpha, const CsrDev &pp, const double *x, long xstride,
                       double *y, long ystride, bool dodiag, double *dotpart, const CgState *skip) {
    auto go = [&](auto m, auto am) {
        matvec_t<R, decltype(m)::value, decltype(am)::value>(st, f, cnt, ps64, pa64, alpha, pp, x, xstride, y,
                                                             ystride, dodiag, dotpart, skip);
    };
    auto cols = [&](auto am) {
        if (M == 1) go(std::integral_constant<int, 1>{}, am);
        else go(std::integral_constant<int, 2>{}, am);
    };
    if (amoeba) cols(std::true_type{});
    else cols(std::false_type{});
}
template void far_launch_matvec<double>(hipStream_t, const FarDev<double> &, bool, int, const int *, const double4 *,
                                        const double *, const double *, const CsrDev &, const double *, long,
                                        double *, long, bool, double *, const CgState *);
template void far_launch_matvec<float>(hipStream_t, const FarDev<float> &, bool, int, const int *, const double4 *,
                                       const double *, const double *, const CsrDev &, const double *, long, double *,
                                       long, bool, double *, const CgState *);

}  // namespace ommp
