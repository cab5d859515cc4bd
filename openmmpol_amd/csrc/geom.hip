// Per-geometry device work: the site records of the uploaded coordinates, the
// check for coincident sites and the neighbour lists of the near-field
// preconditioner, all from one uniform grid of cells at least kNbCut wide over
// the MM atoms (only the 27 cells around a site can hold its neighbours).
//
// The grid is a counting sort: atoms counted per cell, counts scanned, atoms
// placed.  The order inside a cell depends on the atomics, what is made of it
// does not: the check is a flag, and every list row is put in site order by rank.
// kLanes lanes share a site; along x the three cells are one run of the sorted
// atoms, so a site has nine runs of ~8 candidates each.
//
// On the host (hash grid and sorted rows, one thread) this took 2.6 ms at 5,003
// sites and 15 ms at 20,001 per geometry, more than the solve on the device; here
// 30 us of small launches at 648 sites (3-10 us each, bound by latency) and 90 us
// at 20,001 (two scans of 17 us by one workgroup, 15 us for each pass over the
// candidates).
#include <hip/hip_runtime.h>

#include "device.h"

namespace ommp {

namespace {

constexpr int kLanes = 16, kSites = kBlock / kLanes, kRowCap = 64;

__global__ __launch_bounds__(kBlock) void k_geom_sites(int nmm, const double *__restrict__ c,
                                                       const double *__restrict__ w, const int *__restrict__ mm_polar,
                                                       double4 *__restrict__ ms, double4 *__restrict__ ps,
                                                       float4 *__restrict__ ps32) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= nmm) return;
    const double4 s = make_double4(c[3L * i], c[3L * i + 1], c[3L * i + 2], w[i]);
    ms[i] = s;
    const int p = mm_polar[i];
    if (p < 0) return;
    ps[p] = s;
    ps32[p] = make_float4((float)s.x, (float)s.y, (float)s.z, (float)s.w);
}

__device__ __forceinline__ int axis_cell(double x, double lo, double inv_h, int dim) {
    return (int)fmin(fmax(floor((x - lo) * inv_h), 0.0), (double)(dim - 1));  // a NaN goes to cell 0
}

__global__ __launch_bounds__(kBlock) void k_cell_zero(long n, int *__restrict__ count, int *__restrict__ flags) {
    const long k = (long)blockIdx.x * kBlock + threadIdx.x;
    if (k < n) count[k] = 0;
    if (k < 2) flags[k] = 0;
}

__global__ __launch_bounds__(kBlock) void k_cell_count(int nmm, GridGeom g, const double4 *__restrict__ ms,
                                                       int *__restrict__ cell, int *__restrict__ rank,
                                                       int *__restrict__ count) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= nmm) return;
    const double4 s = ms[i];
    const int c = (axis_cell(s.z, g.lo[2], g.inv_h, g.dim[2]) * g.dim[1] + axis_cell(s.y, g.lo[1], g.inv_h, g.dim[1])) *
                      g.dim[0] + axis_cell(s.x, g.lo[0], g.inv_h, g.dim[0]);
    cell[i] = c;
    rank[i] = atomicAdd(count + c, 1);
}

// out[k] = sum of in[0..k), out[n] = the total; one workgroup, kScanPer values
// per thread and round.
constexpr int kScanThreads = 1024, kScanPer = 8;
__global__ __launch_bounds__(kScanThreads) void k_scan(long n, const int *__restrict__ in, int *__restrict__ out,
                                                       int *__restrict__ total) {
    __shared__ int s_wave[kScanThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    int base = 0;
    for (long b = 0; b < n; b += (long)kScanThreads * kScanPer) {
        const long k0 = b + (long)tid * kScanPer;
        int v[kScanPer], sum = 0;
#pragma unroll
        for (int q = 0; q < kScanPer; q++) {
            v[q] = k0 + q < n ? in[k0 + q] : 0;
            sum += v[q];
        }
        int inc = sum;  // inclusive over the wave
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int t = __shfl_up(inc, off, 64);
            if (lane >= off) inc += t;
        }
        if (lane == 63) s_wave[w] = inc;
        __syncthreads();
        int before = base + inc - sum, all = 0;
#pragma unroll
        for (int q = 0; q < kScanThreads / 64; q++) {
            if (q < w) before += s_wave[q];
            all += s_wave[q];
        }
#pragma unroll
        for (int q = 0; q < kScanPer; q++) {
            if (k0 + q < n) out[k0 + q] = before;
            before += v[q];
        }
        base += all;
        __syncthreads();
    }
    if (tid == 0) {
        out[n] = base;
        if (total) *total = base;
    }
}

__global__ __launch_bounds__(kBlock) void k_cell_fill(int nmm, const int *__restrict__ cell,
                                                      const int *__restrict__ rank, const int *__restrict__ start,
                                                      int *__restrict__ order) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < nmm) order[start[cell[i]] + rank[i]] = i;
}

// f(j, d2) for every MM atom j != i in the 27 cells around atom i that this lane takes.
template <typename F>
__device__ __forceinline__ void each_candidate(const GridGeom &g, int i, const double4 &s, int lane,
                                               const int *__restrict__ start, const int *__restrict__ order,
                                               const double4 *__restrict__ ms, F &&f) {
    const int cx = axis_cell(s.x, g.lo[0], g.inv_h, g.dim[0]), cy = axis_cell(s.y, g.lo[1], g.inv_h, g.dim[1]),
              cz = axis_cell(s.z, g.lo[2], g.inv_h, g.dim[2]);
    const int x0 = max(cx - 1, 0), x1 = min(cx + 1, g.dim[0] - 1);
    for (int z = max(cz - 1, 0); z <= min(cz + 1, g.dim[2] - 1); z++)
        for (int y = max(cy - 1, 0); y <= min(cy + 1, g.dim[1] - 1); y++) {
            const int row = (z * g.dim[1] + y) * g.dim[0];
            const int q1 = start[row + x1 + 1];
            for (int q = start[row + x0] + lane; q < q1; q += kLanes) {
                const int j = order[q];
                const double4 t = ms[j];
                const double dx = s.x - t.x, dy = s.y - t.y, dz = s.z - t.z;
                // one rounding order for every caller: the counted and the written rows agree
                if (j != i) f(j, fma(dz, dz, fma(dy, dy, dx * dx)));
            }
        }
}

// Neighbours of every polarizable site (polarizable, closer than the cut), their
// number in count[p]; *bad = 1 where a site coincides with any MM atom
// (distance below eps_rp, mod_electrostatics.F90:1003-1008).
__global__ __launch_bounds__(kBlock) void k_nb_count(int npol, GridGeom g, const int *__restrict__ polar_mm,
                                                     const int *__restrict__ mm_polar,
                                                     const double4 *__restrict__ ms, const int *__restrict__ start,
                                                     const int *__restrict__ order, int *__restrict__ count,
                                                     int *__restrict__ bad) {
    const int p = blockIdx.x * kSites + threadIdx.x / kLanes, lane = threadIdx.x % kLanes;
    if (p >= npol) return;
    const int i = polar_mm[p];
    int n = 0, hit = 0;
    each_candidate(g, i, ms[i], lane, start, order, ms, [&](int j, double d2) {
        if (d2 < kNbCut * kNbCut && mm_polar[j] >= 0) n++;
        if (sqrt(d2) < kEpsRpDev) hit = 1;
    });
#pragma unroll
    for (int m = kLanes / 2; m > 0; m >>= 1) n += __shfl_xor(n, m, 64);
    if (lane == 0) count[p] = n;
    if (hit) *bad = 1;
}

// The rows: ci in ascending order and rowi = p.  The hits of a site are gathered
// in LDS in any order, each is written at its rank; a row of more than kRowCap is
// written smallest first by repeated passes over the candidates.
__global__ __launch_bounds__(kBlock) void k_nb_fill(int npol, GridGeom g, const int *__restrict__ polar_mm,
                                                    const int *__restrict__ mm_polar, const double4 *__restrict__ ms,
                                                    const int *__restrict__ start, const int *__restrict__ order,
                                                    const int *__restrict__ row_ptr, int *__restrict__ ci,
                                                    int *__restrict__ rowi) {
    __shared__ int s_n[kSites], s_hit[kSites][kRowCap];
    const int g0 = threadIdx.x / kLanes, p = blockIdx.x * kSites + g0, lane = threadIdx.x % kLanes;
    if (lane == 0) s_n[g0] = 0;
    __syncthreads();
    const int i = p < npol ? polar_mm[p] : 0, r0 = p < npol ? row_ptr[p] : 0, n = p < npol ? row_ptr[p + 1] - r0 : 0;
    if (n > 0 && n <= kRowCap)
        each_candidate(g, i, ms[i], lane, start, order, ms, [&](int j, double d2) {
            if (d2 < kNbCut * kNbCut && mm_polar[j] >= 0) s_hit[g0][atomicAdd(&s_n[g0], 1)] = mm_polar[j];
        });
    __syncthreads();
    if (n <= kRowCap) {
        for (int e = lane; e < n; e += kLanes) {
            const int q = s_hit[g0][e];
            int rank = 0;
            for (int k = 0; k < n; k++) rank += s_hit[g0][k] < q;
            ci[r0 + rank] = q;
            rowi[r0 + rank] = p;
        }
        return;
    }
    int last = -1;
    for (int e = 0; e < n; e++) {
        int best = 0x7fffffff;
        each_candidate(g, i, ms[i], lane, start, order, ms, [&](int j, double d2) {
            const int q = mm_polar[j];
            if (d2 < kNbCut * kNbCut && q > last) best = min(best, q);
        });
#pragma unroll
        for (int m = kLanes / 2; m > 0; m >>= 1) best = min(best, __shfl_xor(best, m, 64));
        if (lane == 0) {
            ci[r0 + e] = best;
            rowi[r0 + e] = p;
        }
        last = best;
    }
}

int blocks(long n, int per) { return (int)((n + per - 1) / per); }

}  // namespace

void launch_geom_sites(hipStream_t st, int nmm, const double *c, const double *w, const int *mm_polar, double4 *ms,
                       double4 *ps, float4 *ps32) {
    if (nmm == 0) return;
    hipLaunchKernelGGL(k_geom_sites, dim3(blocks(nmm, kBlock)), dim3(kBlock), 0, st, nmm, c, w, mm_polar, ms, ps,
                       ps32);
    HIP_CHECK(hipGetLastError());
}

void launch_grid(hipStream_t st, int nmm, int npol, const GridDev &g, const int *polar_mm, const int *mm_polar,
                 const double4 *ms, int *row_ptr) {
    const long ncell = (long)g.geom.dim[0] * g.geom.dim[1] * g.geom.dim[2];
    hipLaunchKernelGGL(k_cell_zero, dim3(blocks(ncell, kBlock)), dim3(kBlock), 0, st, ncell, g.count, g.flags);
    hipLaunchKernelGGL(k_cell_count, dim3(blocks(nmm, kBlock)), dim3(kBlock), 0, st, nmm, g.geom, ms, g.cell, g.rank,
                       g.count);
    hipLaunchKernelGGL(k_scan, dim3(1), dim3(kScanThreads), 0, st, ncell, g.count, g.start, nullptr);
    hipLaunchKernelGGL(k_cell_fill, dim3(blocks(nmm, kBlock)), dim3(kBlock), 0, st, nmm, g.cell, g.rank, g.start,
                       g.order);
    hipLaunchKernelGGL(k_nb_count, dim3(blocks(npol, kSites)), dim3(kBlock), 0, st, npol, g.geom, polar_mm, mm_polar,
                       ms, g.start, g.order, g.rows, g.flags);
    hipLaunchKernelGGL(k_scan, dim3(1), dim3(kScanThreads), 0, st, (long)npol, g.rows, row_ptr, g.flags + 1);
    HIP_CHECK(hipGetLastError());
}

void launch_nb_lists(hipStream_t st, int npol, const GridDev &g, const int *polar_mm, const int *mm_polar,
                     const double4 *ms, const int *row_ptr, int *ci, int *rowi) {
    if (npol == 0) return;
    hipLaunchKernelGGL(k_nb_fill, dim3(blocks(npol, kSites)), dim3(kBlock), 0, st, npol, g.geom, polar_mm, mm_polar,
                       ms, g.start, g.order, row_ptr, ci, rowi);
    HIP_CHECK(hipGetLastError());
}

}  // namespace ommp
