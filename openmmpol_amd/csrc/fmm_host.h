// Host-built octree and translation tables of the fast multipole path (see
// fmm.h for the device layout they are uploaded into).
#pragma once

#include <hip/hip_runtime.h>

#include <complex>
#include <vector>

#include "fmm.h"

namespace ommp {

struct System;

struct FmmHost {
    int levels = 0, p_pol = 8, p_static = 8, p_tab = 8, ncoef_tab = 81, ncoef2_tab = 289;
    double side = 0.0, leaf_h = 0.0, origin[3] = {0.0, 0.0, 0.0};
    std::vector<long> cell_off;
    std::vector<int> pol_order, pol_leaf, pol_mmself, pol_leaf_start;
    std::vector<int> mm_order, mm_leaf, mm_leaf_start;
    std::vector<int> cnt_pol, cnt_mm;
    std::vector<double2> tab_m2m, tab_l2l, tab_m2l;
};

// Whether trees of L levels and order p use the matrix-core transfer and matvec
// (far.h): orders up to 8, and up to 6 levels, where their per-cell arrays take about
// 1 GB at order 8 (moments twice 0.19, field expansions 0.46, partial sums up to 0.19)
// beside 512 bytes per site and level; others use the complex kernels and tables.
inline bool fmm_uses_far(int L, int p) { return L <= 6 && far_order(p); }

// i^e
inline std::complex<double> fmm_ipow(int e) {
    switch (e & 3) {
        case 0: return {1.0, 0.0};
        case 1: return {0.0, 1.0};
        case 2: return {-1.0, 0.0};
        default: return {0.0, -1.0};
    }
}

// T_n^m(v), n <= p and all m, into out[n^2 + n + m].
void fmm_transfer(int p, const double v[3], double2 *out);

// Octree with leaves of side >= max(min_cell, distance) (bohr) over the MM
// atoms of s, at most kFmmMaxLevels levels below the root.
FmmHost fmm_build(const System &s, int p_pol, int p_static, double min_cell, double distance);

}  // namespace ommp
