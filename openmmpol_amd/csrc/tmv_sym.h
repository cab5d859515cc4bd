// Pair-once sweep of one block pair: the body shared by the single-system T
// matvec (tmv_sym.hip) and the batched solver (batch_kernels.hip).
//
// Sites are grouped in blocks of kSymBlock = 256 (four 64-site sub-tiles, one per
// wave).  For the block pair (I <= J), wave w holds the targets of sub-tile w of
// I in registers; the 256 sites of J are staged in LDS.  For sub-tile k of J,
// lane l meets source (l + s) mod 64 at step s = 0..63, so at every step the 64
// lanes touch 64 distinct sources: the target side accumulates in registers, and
// so does the source side, each lane holding the sum of its current source and
// taking over the next lane's after every step (a DPP wave rotate, on the vector
// ALU); after 64 steps every source-side sum is back at its source's lane.
// Every sum has a fixed order (results bitwise reproducible).  Measured
// alternatives for the source side, both slower: LDS float atomics into a
// per-wave row (FP32 ones were 14x slower here) and lane shuffles through the
// LDS crossbar.  Scale 1 for every pair (the finalize kernels apply the screening
// corrections), self excluded.
//
// A diagonal block pair (I = J) has its ten sub-tile pairs spread evenly: wave w
// sweeps sub-tile w against itself over s = 1..32 (at s = 32 lanes 0..31 alone),
// against w + 1 over all 64 steps and against w + 2 over the half that wave w + 2
// does not (indices mod 4): 128 steps, as many as off the diagonal.  Skipping the
// mirror images (k < w) instead gave wave 0 255 steps, nearly all of them with
// damped pairs, one long dependent chain each: at 8,000 sites of a chain in FP64 it
// took 120 of the sweep's 122 us.
//
// Bound by the vector unit's issue (instructions per pair at 60,000 sites: FP64 one / two
// columns 45 / 67, FP32 37 / 58).  us per sweep, before these diagonals and the cutoffs of
// pair_damp_v and now: FP64 one / two columns at 8,000 sites 113 / 144 and 77 / 105, at
// 15,000 (water) 221 / 309 and 189 / 270, at 60,000 2895 / 4260 and 2565 / 3945; FP32 two
// columns at 15,000 164 and 147, at 60,000 2190 and 2015.
#pragma once

#include <hip/hip_runtime.h>

#include "device.h"
#include "pair_math.h"

namespace ommp {

constexpr int kSymWaves = kSymBlock / 64;

// Index of block pair (I <= J) of nb blocks in the partial sums (the order in which
// the pairs are dispatched is another: the diagonal ones first).
__device__ __forceinline__ long sym_pair_index(int nb, int I, int J) {
    return (long)I * nb - (long)I * (I - 1) / 2 + J - I;
}

// Steps [s, s + n) and sub-tile k of wave w in phase ph of a diagonal block pair.
constexpr int kSymDiagPhases = 3;
__device__ __forceinline__ void sym_diag_phase(int w, int ph, int &k, int &s, int &n) {
    k = (w + ph) & 3;
    s = ph == 0 || (ph == 2 && w >= 2) ? 1 : 0;
    n = ph == 1 ? 64 : 32;
}

// Lane l + 1's value at lane l (wave rotate by one lane, DPP).
__device__ __forceinline__ float lane_next(float v) {
    return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x134, 0xf, 0xf, false));
}
__device__ __forceinline__ double lane_next(double v) {
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_mov_dpp((int)(b & 0xffffffffLL), 0x134, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), 0x134, 0xf, 0xf, false);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// LDS of sym_block_pair for up to M columns (bytes): the block's sources
// (position, damping, dipoles) and the per-wave rows of source-side sums.
template <typename R, int M>
constexpr int sym_lds_bytes() {
    return (int)(sizeof(typename V4<R>::t) * kSymBlock * (1 + M) + sizeof(R) * kSymWaves * M * 3 * 64);
}

// Damps the kernels of a pair of distinct sites at distance^2 r2 (pair_bare) where
// its argument says so.  Beyond the target's cutoff rc2 (row_sweep.h) no pair is
// damped, so that callers decide by one compare per pair and come here only where a
// lane of the wave is inside; the exponential is formed only where its argument says so
// (one site of larger polarizability or smaller damping factor widens every cutoff:
// 15,000 sites, FP64 one column, a polarizability of 300 bohr^3 among them 226 -> 212 us,
// a damping factor of 0 340 -> 239).  AMOEBA: w holds w^3 (vi vj r^3 = u^3).
template <typename R, bool AMOEBA>
__device__ __forceinline__ void pair_damp_v(const typename V4<R>::t &pj, R aj, const typename V4<R>::t &pi, R ai,
                                            R r2, R &k2, R &k3) {
    const R r = r2 * fast_rsqrt(r2);
    R arg;
    bool near;
    if (AMOEBA) {
        arg = pos_min(ai, aj) * ((r * r2) * (pi.w * pj.w));
        near = arg < R(50);
    } else {
        arg = r * (pi.w * pj.w);
        near = arg < R(1);
    }
    if (__ballot(near)) pair_damp<R, AMOEBA>(arg, near, k2, k3);
}

// Both directions' accumulation of one pair: E_i += k3 (x_j.d) d - k2 x_j at the
// target, E_j += k3 (x_i.d) d - k2 x_i at the source, with q = k3 d formed once.
template <typename R, int M>
__device__ __forceinline__ void pair_accum2(R (&acc)[M][3], R *jacc, const typename V4<R>::t *xv,
                                            const R (&xi)[M][3], R dx, R dy, R dz, R k2, R k3) {
    const R qx = k3 * dx, qy = k3 * dy, qz = k3 * dz, nk2 = -k2;
#pragma unroll
    for (int m = 0; m < M; m++) {
        const R c = fmaa(xv[m].z, qz, fmaa(xv[m].y, qy, xv[m].x * qx));
        acc[m][0] = fmaa(c, dx, fmaa(nk2, xv[m].x, acc[m][0]));
        acc[m][1] = fmaa(c, dy, fmaa(nk2, xv[m].y, acc[m][1]));
        acc[m][2] = fmaa(c, dz, fmaa(nk2, xv[m].z, acc[m][2]));
        const R cj = fmaa(xi[m][2], qz, fmaa(xi[m][1], qy, xi[m][0] * qx));
        jacc[3 * m + 0] = fmaa(cj, dx, fmaa(nk2, xi[m][0], jacc[3 * m + 0]));
        jacc[3 * m + 1] = fmaa(cj, dy, fmaa(nk2, xi[m][1], jacc[3 * m + 1]));
        jacc[3 * m + 2] = fmaa(cj, dz, fmaa(nk2, xi[m][2], jacc[3 * m + 2]));
    }
}

// Sources of a block pair: the sites of J to LDS.  Padding sites (past npol, in the
// last block only) sit far away at distinct points with zero dipoles, so that no pair
// but the skipped self pair has a zero distance.
template <typename R, int M, bool AMOEBA>
__device__ __forceinline__ void sym_sources(int npol, int J, const typename V4<R>::t *__restrict__ site,
                                            const R *__restrict__ adamp, const double *const (&xcol)[M],
                                            typename V4<R>::t *s_pos, typename V4<R>::t (*s_x)[kSymBlock]) {
    const R far = R(1e15), gap = R(1e9);
    const int tid = threadIdx.x, jj = J * kSymBlock + tid;
    typename V4<R>::t p, v[M];
    if (jj < npol) {
        p = site[jj];
        if (AMOEBA) p.w = p.w * p.w * p.w;  // w^3 (pair_damp_v)
#pragma unroll
        for (int m = 0; m < M; m++) {
            v[m].x = (R)xcol[m][3L * jj + 0];
            v[m].y = (R)xcol[m][3L * jj + 1];
            v[m].z = (R)xcol[m][3L * jj + 2];
            v[m].w = m == 0 ? adamp[jj] : R(0);
        }
    } else {
        p.x = p.y = p.z = far + gap * (R)tid;
        p.w = R(1);
#pragma unroll
        for (int m = 0; m < M; m++) {
            v[m].x = v[m].y = v[m].z = R(0);
            v[m].w = R(0.39);
        }
    }
    s_pos[tid] = p;
#pragma unroll
    for (int m = 0; m < M; m++) s_x[m][tid] = v[m];
}

// Target li of block I: position (w^3 for AMOEBA), damping, cutoff, dipoles.
template <typename R, int M, bool AMOEBA>
__device__ __forceinline__ void sym_target(int npol, int I, int li, const typename V4<R>::t *__restrict__ site,
                                           const R *__restrict__ adamp, const R *__restrict__ rc2,
                                           const double *const (&xcol)[M], typename V4<R>::t &p, R &a, R &rc,
                                           R (&x)[M][3]) {
    const R far = R(1e15), gap = R(1e9);
    const int i = I * kSymBlock + li;
    if (i < npol) {
        p = site[i];
        if (AMOEBA) p.w = p.w * p.w * p.w;
        a = adamp[i];
        rc = rc2[i];
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int c = 0; c < 3; c++) x[m][c] = (R)xcol[m][3L * i + c];
    } else {
        p.x = p.y = p.z = far + gap * (R)li;
        p.w = R(1);
        a = R(0.39);
        rc = R(0);
#pragma unroll
        for (int m = 0; m < M; m++) x[m][0] = x[m][1] = x[m][2] = R(0);
    }
}

// One wave's sweep of sub-tile k (its sources at pos_k, x_k) over steps s .. s + n - 1
// (n even), two sources at a time: their two dependent chains keep a lone wave busy.
// jacc ends at the sum of source (l + s + n) & 63.  half: the last step is the one
// that meets every pair twice; lanes 0..31 keep theirs.
template <typename R, int M, bool AMOEBA>
__device__ __forceinline__ void sym_sweep(int s, int n, bool half, const typename V4<R>::t &pj, R aj, R rj,
                                          const R (&xi)[M][3], const typename V4<R>::t *pos_k,
                                          const typename V4<R>::t *x_k, R (&acc)[M][3], R (&jacc)[M * 3]) {
    using R4 = typename V4<R>::t;
    const int l = threadIdx.x & 63, end = s + n;
    for (; s < end; s += 2) {
        R4 xv[2][M], ps[2];
        R dx[2], dy[2], dz[2], k2[2], k3[2], r2[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const int js = (l + s + u) & 63;
#pragma unroll
            for (int m = 0; m < M; m++) xv[u][m] = x_k[m * kSymBlock + js];
            ps[u] = pos_k[js];
            r2[u] = pair_bare<R>(pj, ps[u], dx[u], dy[u], dz[u], k2[u], k3[u]);
        }
        if (__ballot(r2[0] < rj || r2[1] < rj)) {
#pragma unroll
            for (int u = 0; u < 2; u++) pair_damp_v<R, AMOEBA>(pj, aj, ps[u], xv[u][0].w, r2[u], k2[u], k3[u]);
        }
        if (half && s + 2 == end && l >= 32) k2[1] = k3[1] = R(0);
#pragma unroll
        for (int u = 0; u < 2; u++) {
            pair_accum2<R, M>(acc, jacc, xv[u], xi, dx[u], dy[u], dz[u], k2[u], k3[u]);
#pragma unroll
            for (int c = 0; c < M * 3; c++) jacc[c] = lane_next(jacc[c]);
        }
    }
}

// Pair (I, J) of blocks with a kSymBlock-thread workgroup: xcol[m] = column m's
// dipoles [npol][3] (FP64); the target-side sums of component c of column m go
// to out_i[m][c * kSymBlock + t] (t = the site's index in I), the source-side
// ones to out_j[m][c * kSymBlock + t] (t in J).  lds: sym_lds_bytes<R, M>()
// bytes, 16-byte aligned (the caller's, so that bodies of different widths in
// one kernel share it); the body ends with a workgroup barrier.
template <typename R, int M, bool AMOEBA>
__device__ __forceinline__ void sym_block_pair(int npol, int I, int J, const typename V4<R>::t *__restrict__ site,
                                               const R *__restrict__ adamp, const R *__restrict__ rc2,
                                               const double *const (&xcol)[M], R *const (&out_i)[M],
                                               R *const (&out_j)[M], char *lds) {
    using R4 = typename V4<R>::t;
    R4 *s_pos = reinterpret_cast<R4 *>(lds);
    R4(*s_x)[kSymBlock] = reinterpret_cast<R4(*)[kSymBlock]>(s_pos + kSymBlock);  // x, y, z; w of column 0: a
    R(*s_acc)[M * 3][64] = reinterpret_cast<R(*)[M * 3][64]>(s_x + M);
    const int tid = threadIdx.x, l = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave index, uniform
    sym_sources<R, M, AMOEBA>(npol, J, site, adamp, xcol, s_pos, s_x);
    R4 pj;
    R aj, rj, xi[M][3], acc[M][3];
    sym_target<R, M, AMOEBA>(npol, I, tid, site, adamp, rc2, xcol, pj, aj, rj, xi);
#pragma unroll
    for (int m = 0; m < M; m++) acc[m][0] = acc[m][1] = acc[m][2] = R(0);
    __syncthreads();
    const bool diag = I == J;
    R jown[M * 3];  // diagonal: the source-side sum of this thread's site
#pragma unroll
    for (int c = 0; c < M * 3; c++) jown[c] = R(0);
    const int phases = diag ? kSymDiagPhases : kSymWaves;
    for (int ph = 0; ph < phases; ph++) {
        int k = ph, s = 0, n = 64;
        if (diag) sym_diag_phase(w, ph, k, s, n);
        R jacc[M * 3];
#pragma unroll
        for (int c = 0; c < M * 3; c++) jacc[c] = R(0);
        sym_sweep<R, M, AMOEBA>(s, n, diag && ph == 0, pj, aj, rj, xi, s_pos + k * 64, &s_x[0][k * 64], acc, jacc);
#pragma unroll
        for (int c = 0; c < M * 3; c++) s_acc[w][c][(l + s + n) & 63] = jacc[c];
        __syncthreads();
        if (diag) {
#pragma unroll
            for (int c = 0; c < M * 3; c++) jown[c] += s_acc[(w - ph) & 3][c][l];
        } else {
            // source side of sub-tile k: the waves' rows added in wave order
            for (int e = tid; e < M * 3 * 64; e += kSymBlock) {
                const int c = e >> 6, jl = e & 63;
                R sum = s_acc[0][c][jl];
#pragma unroll
                for (int q = 1; q < kSymWaves; q++) sum += s_acc[q][c][jl];
                out_j[c / 3][(c % 3) * kSymBlock + k * 64 + jl] = sum;
            }
        }
        __syncthreads();
    }
#pragma unroll
    for (int m = 0; m < M; m++)
#pragma unroll
        for (int c = 0; c < 3; c++) {
            out_i[m][c * kSymBlock + tid] = acc[m][c];
            if (diag) out_j[m][c * kSymBlock + tid] = jown[3 * m + c];
        }
}

// Off-diagonal block pair (I < J) with two targets per lane: wave w holds the
// targets of sub-tiles 2 (w & 1) and 2 (w & 1) + 1 of I and sweeps sub-tiles
// 2 (w >> 1) and 2 (w >> 1) + 1 of J, so that every sub-tile pair is met by one
// wave and each source read from LDS, and each source-side sum rotated, serves
// two pairs.  A target's sum is split over the two waves holding it, a source's
// over the two waves sweeping it; both are added in wave order.  Same interface,
// LDS and outputs as sym_block_pair.
template <typename R, int M, bool AMOEBA>
__device__ __forceinline__ void sym_block_pair2(int npol, int I, int J, const typename V4<R>::t *__restrict__ site,
                                                const R *__restrict__ adamp, const R *__restrict__ rc2,
                                               const double *const (&xcol)[M],
                                                R *const (&out_i)[M], R *const (&out_j)[M], char *lds) {
    using R4 = typename V4<R>::t;
    static_assert(kSymWaves == 4, "two target and two source halves");
    static_assert(M <= 2, "the target-side rows reuse the sources' LDS");
    R4 *s_pos = reinterpret_cast<R4 *>(lds);
    R4(*s_x)[kSymBlock] = reinterpret_cast<R4(*)[kSymBlock]>(s_pos + kSymBlock);
    R(*s_acc)[M * 3][64] = reinterpret_cast<R(*)[M * 3][64]>(s_x + M);
    const int tid = threadIdx.x, l = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int th = w & 1, sh = w >> 1;
    sym_sources<R, M, AMOEBA>(npol, J, site, adamp, xcol, s_pos, s_x);
    // targets: sites 128 th + l and 128 th + 64 + l of I
    R4 pt[2];
    R at[2], rt[2], xt[2][M][3];
#pragma unroll
    for (int h = 0; h < 2; h++)
        sym_target<R, M, AMOEBA>(npol, I, 128 * th + 64 * h + l, site, adamp, rc2, xcol, pt[h], at[h], rt[h], xt[h]);
    R acc[2][M][3];
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int m = 0; m < M; m++) acc[h][m][0] = acc[h][m][1] = acc[h][m][2] = R(0);
    __syncthreads();
    constexpr int kRow = 64 * (int)sizeof(R4);
#pragma unroll
    for (int kk = 0; kk < 2; kk++) {
        const int k = 2 * sh + kk;
        R jacc[M * 3];
#pragma unroll
        for (int c = 0; c < M * 3; c++) jacc[c] = R(0);
        const char *pos_k = reinterpret_cast<const char *>(s_pos + k * 64);
        const char *x_k = reinterpret_cast<const char *>(&s_x[0][k * 64]);
        int jo = l * (int)sizeof(R4);
        for (int s = 0; s < 64; s++) {
            R4 xv[M];
#pragma unroll
            for (int m = 0; m < M; m++)
                xv[m] = *reinterpret_cast<const R4 *>(x_k + m * kSymBlock * (int)sizeof(R4) + jo);
            const R4 ps = *reinterpret_cast<const R4 *>(pos_k + jo);
            // both targets' kernels before the branch: two chains for the few waves
            R dx[2], dy[2], dz[2], k2[2], k3[2], r2[2];
#pragma unroll
            for (int h = 0; h < 2; h++) r2[h] = pair_bare<R>(pt[h], ps, dx[h], dy[h], dz[h], k2[h], k3[h]);
#pragma unroll
            for (int h = 0; h < 2; h++)
                if (__ballot(r2[h] < rt[h]))
                    pair_damp_v<R, AMOEBA>(pt[h], at[h], ps, xv[0].w, r2[h], k2[h], k3[h]);
#pragma unroll
            for (int h = 0; h < 2; h++)
                pair_accum2<R, M>(acc[h], jacc, xv, xt[h], dx[h], dy[h], dz[h], k2[h], k3[h]);
#pragma unroll
            for (int c = 0; c < M * 3; c++) jacc[c] = lane_next(jacc[c]);
            jo = (jo + (int)sizeof(R4)) & (kRow - 1);
        }
#pragma unroll
        for (int c = 0; c < M * 3; c++) s_acc[w][c][l] = jacc[c];
        __syncthreads();
        // source sides of sub-tiles kk and 2 + kk: rows of waves (0, 1) and (2, 3)
        for (int e = tid; e < 2 * M * 3 * 64; e += kSymBlock) {
            const int hh = e / (M * 3 * 64), r = e - hh * (M * 3 * 64), c = r >> 6, jl = r & 63;
            const R sum = s_acc[2 * hh][c][jl] + s_acc[2 * hh + 1][c][jl];
            out_j[c / 3][(c % 3) * kSymBlock + (2 * hh + kk) * 64 + jl] = sum;
        }
        __syncthreads();
    }
    // target sides: waves th and th + 2 hold the same targets (the sources' LDS
    // is free now): rows [wave][half][component][lane]
    R(*s_t)[2][M * 3][64] = reinterpret_cast<R(*)[2][M * 3][64]>(lds);
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int m = 0; m < M; m++)
#pragma unroll
            for (int c = 0; c < 3; c++) s_t[w][h][3 * m + c][l] = acc[h][m][c];
    __syncthreads();
    for (int e = tid; e < 4 * M * 3 * 64; e += kSymBlock) {
        const int ts = e / (M * 3 * 64), r = e - ts * (M * 3 * 64), c = r >> 6, jl = r & 63;
        const int t2 = ts >> 1, h = ts & 1;
        const R sum = s_t[t2][h][c][jl] + s_t[t2 + 2][h][c][jl];
        out_i[c / 3][(c % 3) * kSymBlock + ts * 64 + jl] = sum;
    }
    __syncthreads();
}

// Two targets per lane: FP32 (one or two columns) and FP64 with one or two
// columns, 4-6% faster at 15,000 sites (FP64 two columns: 146 registers, three
// workgroups per CU instead of four, 0.306 -> 0.294 ms per sweep); wider FP64
// groups keep one target per lane.
template <typename R, int M>
constexpr bool kSymTwoTargets = sizeof(R) == 4 || M <= 2;

// The body for block pair (I, J): two targets per lane off the diagonal where
// the width allows it, one otherwise.
template <typename R, int M, bool AMOEBA>
__device__ __forceinline__ void sym_block_pair_any(int npol, int I, int J, const typename V4<R>::t *__restrict__ site,
                                                   const R *__restrict__ adamp, const R *__restrict__ rc2,
                                               const double *const (&xcol)[M],
                                                   R *const (&out_i)[M], R *const (&out_j)[M], char *lds) {
    if constexpr (kSymTwoTargets<R, M>) {
        if (I != J) {
            sym_block_pair2<R, M, AMOEBA>(npol, I, J, site, adamp, rc2, xcol, out_i, out_j, lds);
            return;
        }
    }
    sym_block_pair<R, M, AMOEBA>(npol, I, J, site, adamp, rc2, xcol, out_i, out_j, lds);
}

}  // namespace ommp
