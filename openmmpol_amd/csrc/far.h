// Far field of a uniform octree on the matrix cores: the T matvec through
// multipole expansions (FP64 for the fast multipoles, FP32 for the inner solves
// of the mixed solver), and the transfer step alone for the other passes of the
// fast multipoles (fmm_kernels.hip).
//
// Real solid harmonics B_i(v): degree n >= 0, Re Phi_n^0 | Re Phi_n^m | Im Phi_n^m
// at i = n^2 + (0 | 2m - 1 | 2m) (Phi as in fmm_kernels.hip).  Expansions leave out
// degree 0, i.e. hold coefficient i + 1 at i: a local expansion's constant does not
// act on fields, and only charges have a monopole, which is kept apart.  In units
// of a level's cell side h a cell's moments M = sum D B(v / h) and its local
// expansion l, V = (1 / h) sum l B(v / h), are related by one matrix per cell
// offset for every level,
//   l_target = sum over its interaction list of K(offset) M_source,
// offset = source - target cell.  Cells are numbered (z ns + y) ns + x in a level
// of ns = 2^l cells per side, level l after level l - 1; sites are sorted by leaf,
// so that cells next to each other along x are one run of sites.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>
#include <vector>

#include "device.h"

namespace ommp {

constexpr int kFarMaxLevels = 7;
constexpr int kFarOffsets = 343;  // (dz + 3) 49 + (dy + 3) 7 + dx + 3
constexpr int kFarMaxTiles = 5;   // tiles of 16 coefficients: orders up to 8
constexpr int kFarBasis = 64;     // basis functions of degree < p, p <= 8
constexpr int kFarDots = 64;      // y.x partials per column of the matvec

inline int far_coefs(int p) { return ((p + 1) * (p + 1) - 1 + 15) / 16 * 16; }
inline bool far_order(int p) { return p >= 1 && far_coefs(p) <= 16 * kFarMaxTiles; }

struct FarLevels {
    int levels = 0;
    double side = 0.0, origin[3] = {0.0, 0.0, 0.0};
    long off[kFarMaxLevels + 2] = {0};  // first cell of level l
};

// Target cells by group: cells of one level and one place in their parent (so that
// they have the same interaction list), `width` per group, -1 past the last.
struct FarGroups {
    int n = 0, width = 32;
    int *cell = nullptr;   // [n * width] cell within the level, or -1
    int *level = nullptr;  // [n]; 0: no cells
};

// Transfer state of one tree, R = double or float.  Per-cell arrays over the
// levels 2 .. levels, index off[l] - off[2] + cell.
template <typename R> struct FarDev {
    int p = 0, nc = 0, nsplit = 1;
    FarLevels lv;
    long cells = 0;
    R *K = nullptr;                // [offset][nc / 16][..][64 lanes][16 bytes]
    R *K0 = nullptr;               // [offset][nc / 16][64 lanes]: the monopole's column (FP64 trees)
    R *mom = nullptr, *mom_static = nullptr, *mom0 = nullptr;  // [cells][M][nc], [cells][nc], [cells]
    R *zero = nullptr;             // [nc] zeros
    R *part = nullptr;             // [nsplit][groups][32][nc]
    // T matvec: sites by leaf
    int npol = 0, nblocks = 0, near = 16;  // near: sites per workgroup of the near field, 16 or 32
    int *leaf_start = nullptr, *order = nullptr, *leaf = nullptr;  // leaf: of every sorted site
    typename std::conditional<sizeof(R) == 8, double4, float4>::type *pos = nullptr;
    R *a = nullptr;
    typename std::conditional<sizeof(R) == 8, double4, float4>::type *xs = nullptr;  // [M][npol] the dipoles sorted; w of column 0: a
    const R *rc2 = nullptr;        // damping cutoffs, by polarizable site (row_sweep.h)
    int2 *blocks = nullptr;        // (leaf, first sorted site) of every workgroup of the near field
    R *basis = nullptr;            // [levels - 1][npol][kFarBasis]: B(v / h), degree < p, sorted sites
    R *grad = nullptr;             // [cells][M][3][kFarBasis]: the field's expansion
    double *dots = nullptr;        // [M][nblocks]
    FarGroups groups;              // cells with sites
};

// Transfer matrices of order p in the device layout: made once per order and
// process (they depend on nothing else).
template <typename R> struct FarTables {
    std::vector<R> K, K0;
};
template <typename R> const FarTables<R> &far_tables(int p);
int far_splits(int ngroups);
// Workgroups of the near field: f.near and (leaf, first sorted site) of each.
template <typename R> std::vector<int2> far_blocks(FarDev<R> &f, const std::vector<int> &leaf_start);

// Groups of the cells with cnt != 0 of the levels 2 .. levels (host tree).
void far_group_cells(const FarLevels &lv, const std::vector<int> &cnt, int width, std::vector<int> &cell,
                     std::vector<int> &level);

// f.mom_static and f.mom0 from the complex moments mexp[cell][(p + 1)^2] of the
// static multipoles, all cells of the tree.
void far_launch_moments(hipStream_t st, const FarDev<double> &f, const double2 *mexp);
// Complex local expansions loc (layout of mexp) of the levels 2 .. levels from the
// static multipoles (with_static) and / or the dipoles dip[npol][3] of the sorted
// sites; cells of no group of tgt get zeros.  src, cnt_src: the sources' groups and
// number per cell.
void far_launch_locals(hipStream_t st, const FarDev<double> &f, const FarGroups &tgt, const FarGroups &src,
                       const int *cnt_src, bool with_static, const double *dip, double2 *loc);

// f.basis from the sites ps (once per geometry).
template <typename R> void far_launch_basis(hipStream_t st, const FarDev<R> &f, const double4 *ps);
// y = T x of M columns (corrections, diagonal and kFarDots y.x partials per column,
// as the per-target matvec): far field by expansions, the 27 leaves
// around a target directly.  One column, or two when
// f.groups has 16 cells a group.  cnt: sites per cell of every level.
template <typename R>
void far_launch_matvec(hipStream_t st, const FarDev<R> &f, bool amoeba, int M, const int *cnt, const double4 *ps64,
                       const double *pa64, const double *alpha, const CsrDev &pp, const double *x, long xstride,
                       double *y, long ystride, bool dodiag, double *dotpart, const CgState *skip);

}  // namespace ommp
