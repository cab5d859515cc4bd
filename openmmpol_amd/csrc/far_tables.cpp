// Transfer matrices of the real solid harmonics (far.h), from the complex
// convolution of fmm_kernels.hip: L_j^k = sum O_n^m T_{j+n}^{m-k}, with the source
// moments R_n^+-m and the local functions S_j^+-k written in Re and Im Phi; and
// the grouping of target cells.
#include <algorithm>
#include <cmath>
#include <complex>
#include <mutex>
#include <type_traits>

#include "fmm_host.h"

namespace ommp {

namespace {

using cplx = std::complex<double>;

// Coefficients of Re and Im Phi in the complex functions of +m and -m.
struct Term {
    int m;
    cplx f;
};
std::vector<Term> source_terms(int m, bool im) {
    // R^m = (-i)^m (c - i s), R^-m = (-i)^m (c + i s)
    std::vector<Term> out = {{m, fmm_ipow(-m) * (im ? cplx(0.0, -1.0) : cplx(1.0))}};
    if (m > 0) out.push_back({-m, fmm_ipow(-m) * (im ? cplx(0.0, 1.0) : cplx(1.0))});
    return out;
}
std::vector<Term> local_terms(int j, int k, bool im) {
    // S^k = i^-k (-1)^j (c + i s), S^-k = i^-k (-1)^j (c - i s)
    const cplx f = fmm_ipow(-k) * ((j & 1) ? -1.0 : 1.0);
    std::vector<Term> out = {{k, f * (im ? cplx(0.0, 1.0) : cplx(1.0))}};
    if (k > 0) out.push_back({-k, f * (im ? cplx(0.0, -1.0) : cplx(1.0))});
    return out;
}

template <typename R> void make_tables(int p, FarTables<R> &out) {
    constexpr int vec = 16 / sizeof(R);  // elements of a lane's load
    const int nc = far_coefs(p), ncoef = (p + 1) * (p + 1) - 1, tiles = nc / 16, per = nc / 4;
    out.K.assign((size_t)kFarOffsets * nc * nc, R(0));
    out.K0.assign((size_t)kFarOffsets * tiles * 64, R(0));
    std::vector<std::vector<Term>> src(ncoef), loc(ncoef);
    std::vector<int> deg(ncoef);
    for (int i = 0; i < ncoef; i++) {
        int n = 1;
        while ((n + 1) * (n + 1) - 1 <= i) n++;
        const int r = i - (n * n - 1), m = (r + 1) / 2;
        const bool im = r > 0 && r % 2 == 0;
        deg[i] = n;
        src[i] = source_terms(m, im);
        loc[i] = local_terms(n, m, im);
    }
    for (int o = 0; o < kFarOffsets; o++) {
        const int d[3] = {o % 7 - 3, o / 7 % 7 - 3, o / 49 - 3};
        if (std::abs(d[0]) <= 1 && std::abs(d[1]) <= 1 && std::abs(d[2]) <= 1) continue;
        const double v[3] = {(double)d[0], (double)d[1], (double)d[2]};
        std::vector<double2> tv((2 * p + 1) * (2 * p + 1));
        fmm_transfer(2 * p, v, tv.data());
        auto t = [&](int k) { return cplx(tv[k].x, tv[k].y); };
        for (int row = 0; row < ncoef; row++) {
            for (int col = 0; col < ncoef; col++) {
                const int n = deg[row] + deg[col];
                cplx s = 0.0;
                for (const Term &a : loc[row])
                    for (const Term &b : src[col]) s += a.f * b.f * t(n * n + n + b.m - a.m);
                // lane (row % 16, col / per), element col % per in vectors of 16 bytes
                const int lane = row % 16 + 16 * (col / per), e = col % per;
                out.K[((((size_t)o * tiles + row / 16) * (per / vec) + e / vec) * 64 + lane) * vec + e % vec] =
                    (R)s.real();
            }
            cplx s = 0.0;
            const int n = deg[row];
            for (const Term &a : loc[row]) s += a.f * t(n * n + n - a.m);
            out.K0[((size_t)o * tiles + row / 16) * 64 + row % 16] = (R)s.real();
        }
    }
}

}  // namespace

template <typename R> const FarTables<R> &far_tables(int p) {
    static std::once_flag made[9];
    static FarTables<R> tables[9];
    std::call_once(made[p], [p] { make_tables(p, tables[p]); });
    return tables[p];
}
template const FarTables<double> &far_tables<double>(int p);
template const FarTables<float> &far_tables<float>(int p);

template <typename R> std::vector<int2> far_blocks(FarDev<R> &f, const std::vector<int> &leaf_start) {
    int occupied = 0;
    for (size_t k = 0; k + 1 < leaf_start.size(); k++) occupied += leaf_start[k + 1] > leaf_start[k];
    // 32 sites share a workgroup's sources where most leaves have several such groups
    f.near = f.npol > 96L * occupied ? 32 : 16;
    std::vector<int2> blocks;
    for (int k = 0; k + 1 < (int)leaf_start.size(); k++)
        for (int t = leaf_start[k]; t < leaf_start[k + 1]; t += f.near) blocks.push_back(make_int2(k, t));
    f.nblocks = (int)blocks.size();
    return blocks;
}
template std::vector<int2> far_blocks<double>(FarDev<double> &, const std::vector<int> &);
template std::vector<int2> far_blocks<float>(FarDev<float> &, const std::vector<int> &);

// Enough workgroups to fill the chip when a tree has few groups of cells.
int far_splits(int ngroups) {
    const int s = (1024 + ngroups - 1) / std::max(ngroups, 1);
    return std::min(std::max(s, 1), 12);
}

void far_group_cells(const FarLevels &lv, const std::vector<int> &cnt, int width, std::vector<int> &cell,
                     std::vector<int> &level) {
    cell.clear();
    level.clear();
    for (int l = 2; l <= lv.levels; l++) {
        const int ns = 1 << l;
        for (int c = 0; c < 8; c++) {
            for (int z = c >> 2; z < ns; z += 2)
                for (int y = c >> 1 & 1; y < ns; y += 2)
                    for (int x = c & 1; x < ns; x += 2) {
                        const int k = (z * ns + y) * ns + x;
                        if (cnt[lv.off[l] + k] != 0) cell.push_back(k);
                    }
            while (cell.size() % width) cell.push_back(-1);
            level.resize(cell.size() / width, l);
        }
    }
}

}  // namespace ommp
