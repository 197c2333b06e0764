// SO(4)/SNAP bispectrum kernels for gfx950 (FP64, wave64).
//
// Device layout (HBM), per atom i (tile t = i/64, lane = i%64):
//   utot[t][nhalf][lane] complex  U_tot half rows (mb <= l/2), self term,
//                                 u_norm (tile-major; the Z, B and Y kernels
//                                 run one atom per lane)
//   z[t][nz][lane]  complex  Z in the reference's idxz order, tile-major
//   b[i][nb]        real     B in the reference's idxb order
//   y[i][nhalf]     complex  adjoint Y (dE/dB-weighted Z, half weights,
//                            factor 2 and u_norm folded in)
// per image e (centre i, neighbour j, translation T): r_e[3], dE/dr_e[3].
//
// The Wigner-U recursion (compute_uarray_recursive / compute_duarray_recursive,
// SNAP.py:870-1017) is run "one lane per row": a group of G = 2J/2+1 lanes
// serves one neighbour image, lane mb carrying row mb of every level in
// registers.  Row mb of level l only needs row mb of level l-1, so the lanes
// never exchange data; lane mb starts from row 0 (which it recurses up to
// level mb) and turns it into row mb of level mb with the inversion symmetry
// u[l][l-mb][l-ma] = (-1)^(ma+mb) conj(u[l][mb][ma]) (SNAP.py:908-925).
// Every lane executes the same fully unrolled instruction stream
// (sum_l l recursion steps), so groups never diverge.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <cmath>
#include <cstring>
#include <map>
#include <atomic>
#include <mutex>
#include <numeric>
#include <tuple>
#include <utility>
#include <vector>

#include "pxff_common.h"
#include "so4_dev.h"
#include "so4_tables.h"

namespace pxff {

namespace {
std::mutex g_tab_mutex;
std::map<std::pair<int, int>, So4Dev> g_tabs;  // (device, 2J*2+norm)

template <typename T>
int upload(const std::vector<T> &v, T **dst) {
    size_t n = v.size() ? v.size() : 1;
    PXFF_HIP_CHECK(hipMalloc((void **)dst, n * sizeof(T)));
    if (!v.empty()) PXFF_HIP_CHECK(hipMemcpy(*dst, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    return 0;
}
}  // namespace

// Tables of the matrix-core dB/dr kernel (so4_dbdr_centre_kernel).
static int db_tables(const So4HostTables &t, So4Dev &d) {
    // the kernel's LDS is sized at compile time by these counts
    bool as_compiled = t.nb == nb_of(t.twol);
    for (int l = 0; l < t.ldim; l++)
        as_compiled = as_compiled && t.blk_level_start[l + 1] - t.blk_level_start[l] == nblk_level(t.twol, l);
    if (!as_compiled) {
        set_error("block counts of the 2J tables differ from those the dB/dr kernel is built for");
        return PXFF_EINVAL;
    }
    const int nw = db_waves(t.twol), tw = ((t.nb + 3) / 4 + nw - 1) / nw, nslot = nw * tw * 4;
    // stages: runs of levels whose values share a W row
    std::vector<int> stage(t.ldim, 0);
    for (int l = 1; l < t.ldim; l++) stage[l] = stage[l - 1] + (db_stage_first(t.twol, l) == l ? 1 : 0);
    const int nstage = stage[t.ldim - 1] + 1;
    // the levels that hold a block of b
    std::vector<unsigned> lev(nslot, 0u);
    for (int l = 0; l < t.ldim; l++)
        for (int k = t.blk_level_start[l]; k < t.blk_level_start[l + 1]; k++)
            for (int q = 0; q < 3; q++)
                if (t.blk_tb[3 * k + q] >= 0) lev[t.blk_tb[3 * k + q]] |= 1u << l;
    // Components to the places (wavefront, tile, row): a tile costs the union
    // of its components' levels, and the wavefronts wait for each other
    // after every stage, so the cost is the sum over the stages of the
    // busiest wavefront's steps (then the steps of all).  Exchanges while
    // they do not cost more, from the components in order of their levels.
    // On the host at the first call of a 2J: the steps of every union are
    // tabulated, and an exchange changes the work of its two tiles only (2J =
    // 6 / 8 / 10: 0.2 / 1 / 2 ms, 4 / 8 / 10 with every exchange summed anew).
    std::vector<int> place(nslot);
    std::iota(place.begin(), place.end(), 0);
    std::stable_sort(place.begin(), place.end(), [&](int a, int b) { return lev[a] > lev[b]; });
    // deal the tiles out in turn
    {
        std::vector<int> p(place.size());
        for (int k = 0; k < nw * tw; k++)
            for (int q = 0; q < 4; q++) p[((k % nw) * tw + k / nw) * 4 + q] = place[4 * k + q];
        place = p;
    }
    // steps[m][s]: of the levels of the set m in stage s
    std::vector<int> steps((size_t)nstage << t.ldim, 0);
    for (unsigned m = 1; m < 1u << t.ldim; m++) {
        const int l = __builtin_ctz(m);
        for (int s = 0; s < nstage; s++) steps[m * nstage + s] = steps[(m & (m - 1)) * nstage + s];
        steps[m * nstage + stage[l]] += db_steps(l);
    }
    std::vector<unsigned> at(nslot), uni(nw * tw, 0u);  // levels of a place's component, of a tile
    for (int k = 0; k < nslot; k++) {
        at[k] = lev[place[k]];
        uni[k / 4] |= at[k];
    }
    std::vector<int> work(8 * nstage, 0);  // [stage][wavefront], the last four unused below 2J = 10
    long sum = 0;
    for (int k = 0; k < nw * tw; k++)
        for (int s = 0; s < nstage; s++) {
            work[8 * s + k / tw] += steps[uni[k] * nstage + s];
            sum += steps[uni[k] * nstage + s];
        }
    auto peak = [&]() {
        long p = 0;
        for (int s = 0; s < nstage; s++) {
            const int *w = &work[8 * s];
            p += std::max(std::max(std::max(w[0], w[1]), std::max(w[2], w[3])),
                          std::max(std::max(w[4], w[5]), std::max(w[6], w[7])));
        }
        return p;
    };
    uint32_t rnd = 12345u;
    auto next = [&](int n) {
        rnd = rnd * 1664525u + 1013904223u;
        return (int)((rnd >> 8) % (uint32_t)n);
    };
    auto others = [&](int k) {  // levels of the other three places of k's tile
        const int b = k & ~3;
        return at[b + ((k + 1) & 3)] | at[b + ((k + 2) & 3)] | at[b + ((k + 3) & 3)];
    };
    long best = peak() * 4096 + sum;
    // 2J = 8: the last gain is at 30,000 of 32,768; 2J = 10: 40,000 come within 1e-4 of twice as many
    const int trials = std::min(8 * nslot * nslot, 40000);
    for (int it = 0; it < trials; it++) {
        const int i = next(nslot), j = next(nslot), a = i / 4, b = j / 4;
        if (a == b || at[i] == at[j]) continue;
        const unsigned ma = others(i) | at[j], mb = others(j) | at[i];
        if (ma == uni[a] && mb == uni[b]) {  // costs what it did
            std::swap(at[i], at[j]);
            std::swap(place[i], place[j]);
            continue;
        }
        const int *na = &steps[ma * nstage], *oa = &steps[uni[a] * nstage];
        const int *nb = &steps[mb * nstage], *ob = &steps[uni[b] * nstage];
        int *wa = &work[a / tw], *wb = &work[b / tw];
        long d = 0;
        for (int s = 0; s < nstage; s++) {
            wa[8 * s] += na[s] - oa[s];
            wb[8 * s] += nb[s] - ob[s];
            d += (na[s] - oa[s]) + (nb[s] - ob[s]);
        }
        const long now = peak() * 4096 + sum + d;
        if (now > best) {
            for (int s = 0; s < nstage; s++) {
                wa[8 * s] -= na[s] - oa[s];
                wb[8 * s] -= nb[s] - ob[s];
            }
            continue;
        }
        best = now;
        sum += d;
        uni[a] = ma;
        uni[b] = mb;
        std::swap(at[i], at[j]);
        std::swap(place[i], place[j]);
    }
    // levels of every tile, then the component of every slot (-1 none)
    std::vector<int> tile, where(t.nb, 0);
    for (int k = 0; k < nw * tw; k++) {
        unsigned m = 0;
        for (int q = 0; q < 4; q++) m |= lev[place[4 * k + q]];
        tile.push_back((int)m);
    }
    for (int k = 0; k < nslot; k++) {
        tile.push_back(place[k] < t.nb ? place[k] : -1);
        if (place[k] < t.nb) where[place[k]] = k;
    }
    // LDS row of the block of every (level, slot) (the zero row without one)
    // and its factor 2 f norm_l; Z elements in level order: their Z offset,
    // then place in the stage's LDS rows and twice the half weight
    const int zero = db_stage_zlds(t.twol) - db_stride(t.twol);
    std::vector<int> row((size_t)t.ldim * nslot, zero), zmap, first;
    std::vector<double> fac((size_t)t.ldim * nslot, 0.0);
    int z = 0, c = 0;
    for (int l = 0; l < t.ldim; l++) {
        if (l == 0 || stage[l] != stage[l - 1]) {
            first.push_back(z);
            first.push_back(c);
            first.push_back(l);
        }
        const int base = db_level_zbase(t.twol, l), st = db_level_stride(l);
        for (int k = t.blk_level_start[l]; k < t.blk_level_start[l + 1]; k++) {
            const int at = base + (k - t.blk_level_start[l]) * st;
            for (int q = 0; q < 3; q++) {
                const int b = t.blk_tb[3 * k + q];
                if (b < 0) continue;
                const size_t e = (size_t)l * nslot + where[b];
                if (row[e] != zero) {
                    set_error("two blocks of one level target one bispectrum component");
                    return PXFF_EINVAL;
                }
                row[e] = at;
                fac[e] = t.blk_tf[3 * k + q] * 2.0 * t.lnorm[l];
            }
            for (int loc = 0; loc < (l / 2 + 1) * (l + 1); loc++) {
                zmap.push_back(t.blk_zoff[k] + loc);
                zmap.push_back((at + 2 * loc) | (int)(2.0 * t.h_weight[t.hoff[l] + loc]) << 16);
            }
        }
        z += (t.blk_level_start[l + 1] - t.blk_level_start[l]) * (l / 2 + 1) * (l + 1);
        c += db_steps(l) * 16;
    }
    first.push_back(z);
    first.push_back(c);
    first.push_back(t.ldim);
    // coefficients (C1, C2) of V_q at element k of a level (re / im of half
    // element loc, times W's sqrt factor s): V_q[k] = C1 Z[k + off1] + C2 Z[k + off2]
    std::vector<double> coef;
    auto f = [](int n) {
        double v = 1.0;
        for (int k = 2; k <= n; k++) v *= k;
        return v;
    };
    for (int l = 0; l < t.ldim; l++)
        for (int k = 0; k < 4 * db_steps(l); k++) {
            const int loc = k / 2, mb = loc / (l + 1), m = loc - mb * (l + 1);
            const bool in = loc < (l / 2 + 1) * (l + 1);
            const double s = in ? std::sqrt(f(m) * f(l - m) / (f(mb) * f(l - mb))) : 0.0;
            const double up = in ? std::sqrt((double)((m + 1) * (l - m))) : 0.0;
            const double dn = in ? std::sqrt((double)(m * (l - m + 1))) : 0.0;
            const double sg = k & 1 ? -1.0 : 1.0;
            const double cc[4][2] = {{s, 0.0}, {sg * s * (l - 2 * m), 0.0}, {s * up, -s * dn}, {sg * s * up, sg * s * dn}};
            for (int q = 0; q < 4; q++) {
                coef.push_back(cc[q][0]);
                coef.push_back(cc[q][1]);
            }
        }
    d.db_nstage = nstage;
    int rc = 0;
    if ((rc = upload(tile, &d.db_tile))) return rc;
    if ((rc = upload(row, &d.db_row))) return rc;
    if ((rc = upload(fac, &d.db_fac))) return rc;
    if ((rc = upload(zmap, &d.db_zmap))) return rc;
    if ((rc = upload(first, &d.db_stage))) return rc;
    return upload(coef, &d.db_coef);
}

int find_so4_tables(int twol, int norm, const So4Dev **out) {
    int dev = 0;
    PXFF_HIP_CHECK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_tab_mutex);
    auto it = g_tabs.find(std::make_pair(dev, twol * 2 + (norm ? 1 : 0)));
    if (it == g_tabs.end()) {
        set_error("the 2J=" + std::to_string(twol) + " tables are not built on this device yet: call any allocating "
                  "SO4 entry point (e.g. pxff_so4_tangent) with the same 2J and normalisation once first");
        return PXFF_EINVAL;
    }
    *out = &it->second;
    return 0;
}

int get_so4_tables(int twol, int norm, const So4Dev **out) {
    int dev = 0;
    PXFF_HIP_CHECK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_tab_mutex);
    auto key = std::make_pair(dev, twol * 2 + (norm ? 1 : 0));
    auto it = g_tabs.find(key);
    if (it != g_tabs.end()) {
        *out = &it->second;
        return 0;
    }
    So4HostTables t;
    if (!build_so4_tables(twol, norm, t)) {
        set_error("unsupported 2J=" + std::to_string(twol) + " (even 2J in 0..10 supported)");
        return PXFF_ENOTIMPL;
    }
    So4Dev d;
    d.twol = twol;
    d.nu = t.nu;
    d.nhalf = t.nhalf;
    d.nz = t.nz;
    d.nb = t.nb;
    d.ncg = t.ncg;
    d.nblk = t.nblk;
    int rc = 0;
    if ((rc = upload(t.cglist, &d.cg))) return rc;
    if ((rc = upload(t.blk_level_start, &d.blk_level_start))) return rc;
    if ((rc = upload(t.blk_zoff, &d.blk_zoff))) return rc;
    if ((rc = upload(t.blk_tb, &d.blk_tb))) return rc;
    if ((rc = upload(t.blk_tf, &d.blk_tf))) return rc;
    if ((rc = upload(t.b_zoff, &d.b_zoff))) return rc;
    if ((rc = upload(t.b_level, &d.b_level))) return rc;
    if ((rc = upload(t.rootpq, &d.rootpq))) return rc;
    if ((rc = upload(t.lnorm, &d.lnorm))) return rc;
    if ((rc = upload(t.hoff, &d.hoff))) return rc;
    if ((rc = upload(t.h_level, &d.h_level))) return rc;
    if ((rc = upload(t.h_diag, &d.h_diag))) return rc;
    if ((rc = upload(t.h_weight, &d.h_weight))) return rc;
    if ((rc = upload(t.idxu_block, &d.idxu_block))) return rc;
    d.nbrow = t.nbrow;
    if ((rc = upload(t.b_brow0, &d.b_brow0))) return rc;
    d.nzgroups = t.nzgroups;
    if ((rc = upload(t.zgroups, &d.zgroups))) return rc;
    // inverse of the block targets: the (block, factor) pairs of each b
    std::vector<int> bsrc(3 * (size_t)t.nb, -1);
    std::vector<double> bsrcf(3 * (size_t)t.nb, 0.0);
    for (int k = 0; k < t.nblk; k++)
        for (int q = 0; q < 3; q++) {
            const int b = t.blk_tb[3 * k + q];
            if (b < 0) continue;
            int slot = 0;
            while (slot < 3 && bsrc[3 * b + slot] >= 0) slot++;
            if (slot == 3) {
                set_error("more than three blocks target one bispectrum component");
                return PXFF_EINVAL;
            }
            bsrc[3 * b + slot] = k;
            bsrcf[3 * b + slot] = t.blk_tf[3 * k + q];
        }
    if ((rc = upload(bsrc, &d.b_src))) return rc;
    if ((rc = upload(bsrcf, &d.b_srcf))) return rc;
    // half-U element of each Z element: Z block (l1, l2, l) element loc pairs
    // with U^l element loc (same (mb, ma), mb <= l/2)
    std::vector<int> zh((size_t)t.nz, 0);
    for (int k = 0; k < t.nblk; k++) {
        int l = 0;
        while (l + 1 < t.ldim && k >= t.blk_level_start[l + 1]) l++;
        const int nloc = (l / 2 + 1) * (l + 1);
        for (int q = 0; q < nloc; q++) {
            zh[t.blk_zoff[k] + q] = t.hoff[l] + q;
        }
    }
    if ((rc = upload(zh, &d.zh))) return rc;
    std::vector<double> hscale((size_t)t.nhalf, 0.0);
    for (int h = 0; h < t.nhalf; h++) hscale[h] = 2.0 * t.h_weight[h] * t.lnorm[t.h_level[h]];
    if ((rc = upload(hscale, &d.hscale))) return rc;
    // Y tasks, most blocks first (longest wavefronts start first)
    std::vector<std::array<int, YTASK_STRIDE>> yt;
    for (int l = 0; l < t.ldim; l++) {
        const int nloc = (l / 2 + 1) * (l + 1);
        for (int loc0 = 0; loc0 < nloc; loc0 += YTASK_ROWS)
            yt.push_back({l, loc0, std::min(YTASK_ROWS, nloc - loc0), t.blk_level_start[l],
                          t.blk_level_start[l + 1], t.hoff[l] + loc0});
    }
    std::stable_sort(yt.begin(), yt.end(), [](const std::array<int, YTASK_STRIDE> &a,
                                              const std::array<int, YTASK_STRIDE> &b) {
        return (a[4] - a[3]) * a[2] > (b[4] - b[3]) * b[2];
    });
    std::vector<int> ytf;
    for (auto &q : yt) ytf.insert(ytf.end(), q.begin(), q.end());
    d.nytask = (int)yt.size();
    if ((rc = upload(ytf, &d.ytask))) return rc;
    if ((rc = db_tables(t, d))) return rc;
    g_tabs[key] = d;
    *out = &g_tabs[key];
    return 0;
}

// Cayley-Klein parameters of one image (compute_uarray_recursive,
// SNAP.py:909-914) and their gradients (compute_duarray_recursive,
// SNAP.py:965-976).
struct CK {
    cd ca, cb;          // conj(a), conj(b)
    cd cda[3], cdb[3];  // conj(da/dr_k), conj(db/dr_k)
};

__device__ inline void cayley_klein(double x, double y, double z, double r, double psi, bool grad, CK &ck) {
    double sinpsi, cospsi;
    sincos(psi, &sinpsi, &cospsi);
    // a = cos psi - i sin psi z/r ; b = sin psi/r (y - i x)
    ck.ca = cmake(cospsi, sinpsi / r * z);
    ck.cb = cmake(sinpsi / r * y, sinpsi / r * x);
    if (grad) {
        double g[3] = {x / r, y / r, z / r};
        double rr = r * r;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            // da = -sinpsi*psi/r*g - i*z*cospsi/r^2*psi*g + i*z*sinpsi/r^2*g  (+ -i sinpsi/r on z)
            double dre = -sinpsi * psi / r * g[k];
            double dim = -z * cospsi / rr * psi * g[k] + z * sinpsi / rr * g[k];
            if (k == 2) dim += -sinpsi / r;
            ck.cda[k] = cmake(dre, -dim);
            // db = cospsi/r^2*psi*(y - i x)*g - sinpsi/r^2*(y - i x)*g  (+ sinpsi/r on y, -i sinpsi/r on x)
            double f = cospsi / rr * psi * g[k] - sinpsi / rr * g[k];
            double bre = f * y, bim = -f * x;
            if (k == 1) bre += sinpsi / r;
            if (k == 0) bim += -sinpsi / r;
            ck.cdb[k] = cmake(bre, -bim);
        }
    }
}

// One level of the row recursion, in place, descending ma.
//   new[m] = rootpq[l-m][q] ca old[m] - rootpq[m][q] cb old[m-1],  q = l - mb
// (SNAP.py:921-931) and, with GRAD, its derivative (SNAP.py:982-991).
template <int TWOJ, bool GRAD>
__device__ inline void row_step(int l, int q, const double *__restrict__ rpq, const CK &ck, cd *u, cd (*du)[TWOJ + 1]) {
#pragma unroll
    for (int m = TWOJ; m >= 0; --m) {
        if (m > l) continue;
        cd un = cmake(0.0, 0.0);
        cd dn[3] = {cmake(0, 0), cmake(0, 0), cmake(0, 0)};
        // the coefficient is folded into one factor of each product (c1 ca,
        // c1 u), so every derivative term is a complex multiply-add
        if (m < l) {
            double c1 = rpq[(l - m) * (TWOJ + 1) + q];
            cd c1a = cscale(ck.ca, c1);
            un = cmul(c1a, u[m]);
            if (GRAD) {
                const cd c1u = cscale(u[m], c1);
#pragma unroll
                for (int k = 0; k < 3; k++) dn[k] = cmadd(c1a, du[k][m], cmul(ck.cda[k], c1u));
            }
        }
        if (m >= 1) {
            double c2 = rpq[m * (TWOJ + 1) + q];
            cd c2b = cscale(ck.cb, -c2);
            un = cmadd(c2b, u[m - 1], un);
            if (GRAD) {
                const cd c2u = cscale(u[m - 1], -c2);
#pragma unroll
                for (int k = 0; k < 3; k++) dn[k] = cmadd(c2b, du[k][m - 1], cmadd(ck.cdb[k], c2u, dn[k]));
            }
        }
        u[m] = un;
        if (GRAD) {
#pragma unroll
            for (int k = 0; k < 3; k++) du[k][m] = dn[k];
        }
    }
}

// Row 0 -> row l of the same level: new[m] = (-1)^(l-m) conj(old[l-m]).
template <int TWOJ, bool GRAD>
__device__ inline void row_flip(int l, cd *u, cd (*du)[TWOJ + 1]) {
    cd tu[TWOJ + 1];
    cd td[3][TWOJ + 1];
#pragma unroll
    for (int m = 0; m <= TWOJ; m++) {
        if (m > l) continue;
        double s = ((l - m) & 1) ? -1.0 : 1.0;
        cd o = u[l - m];
        tu[m] = cmake(s * o.re, -s * o.im);
        if (GRAD) {
#pragma unroll
            for (int k = 0; k < 3; k++) {
                cd od = du[k][l - m];
                td[k][m] = cmake(s * od.re, -s * od.im);
            }
        }
    }
#pragma unroll
    for (int m = 0; m <= TWOJ; m++) {
        if (m > l) continue;
        u[m] = tu[m];
        if (GRAD) {
#pragma unroll
            for (int k = 0; k < 3; k++) du[k][m] = td[k][m];
        }
    }
}

// Sweep the levels of one image.  After every level l all lanes call
// f(l, u_row, du_row, half) with half = (2 mb <= l), i.e. whether the lane's
// row is one of the half rows the bispectrum uses.  Lanes whose row is not a
// half row still run the recursion, so control flow stays uniform.
template <int TWOJ, bool GRAD, typename F>
__device__ inline void sweep_rows(int mb, const double *__restrict__ rpq, const CK &ck, F &&f) {
    cd u[TWOJ + 1];
    cd du[3][TWOJ + 1];
#pragma unroll
    for (int m = 0; m <= TWOJ; m++) {
        u[m] = cmake(0.0, 0.0);
#pragma unroll
        for (int k = 0; k < 3; k++) du[k][m] = cmake(0.0, 0.0);
    }
    u[0] = cmake(1.0, 0.0);
    f(0, u, du, mb == 0);
#pragma unroll
    for (int l = 1; l <= TWOJ; l++) {
        // without derivative rows: keep the coefficient loads of a level
        // inside it (hoisted loads of later levels would hold registers
        // across the whole sweep)
        if (!GRAD) asm volatile("" ::: "memory");
        const int mbe = (l <= mb) ? 0 : mb;
        row_step<TWOJ, GRAD>(l, l - mbe, rpq, ck, u, du);
        if (l == mb) row_flip<TWOJ, GRAD>(l, u, du);
        f(l, u, du, 2 * mb <= l);
    }
}

// The same sweep with the recursion coefficients taken out.  The
// coefficients are sqrt(p / q) (init_rootpqarray, SNAP.py:861-868):
// c1 = sqrt(l - m) / sqrt(q), c2 = sqrt(m) / sqrt(q) with q = l - mb (q = l
// on row 0), so with
//   u^l_mb[m] = sqrt(m! (l - m)! / (mb! (l - mb)!)) W^l[m]
// the row recursion becomes W^l[m] = ca W^{l-1}[m] - cb W^{l-1}[m-1]
// (binomial, no coefficients: W^l on row 0 is C(l, m) ca^(l-m) (-cb)^m),
// and the inversion flip keeps its form (the factor is symmetric under
// m <-> l - m).  f(l, w, half) receives W; the factor (so4_wscale) is
// image-independent, so sums over images take it once.  |W| <= C(l, l/2)
// (252 at 2J = 10).
template <int TWOJ, typename F>
__device__ inline void sweep_rows_w(int mb, const CK &ck, F &&f) {
    cd w[TWOJ + 1];
#pragma unroll
    for (int m = 0; m <= TWOJ; m++) w[m] = cmake(0.0, 0.0);
    w[0] = cmake(1.0, 0.0);
    f(0, w, mb == 0);
    const cd mcb = cmake(-ck.cb.re, -ck.cb.im);
#pragma unroll
    for (int l = 1; l <= TWOJ; l++) {
#pragma unroll
        for (int m = TWOJ; m >= 0; --m) {
            if (m > l) continue;
            if (m == l)
                w[m] = cmul(mcb, w[m - 1]);
            else if (m >= 1)
                w[m] = cmadd(mcb, w[m - 1], cmul(ck.ca, w[m]));
            else
                w[m] = cmul(ck.ca, w[m]);
        }
        if (l == mb) {
            cd t[TWOJ + 1];
#pragma unroll
            for (int m = 0; m <= TWOJ; m++) {
                if (m > l) continue;
                const cd o = w[l - m];
                t[m] = ((l - m) & 1) ? cmake(-o.re, o.im) : cmake(o.re, -o.im);
            }
#pragma unroll
            for (int m = 0; m <= TWOJ; m++)
                if (m <= l) w[m] = t[m];
        }
        f(l, w, 2 * mb <= l);
    }
}

// sqrt(m! (l - m)! / (mb! (l - mb)!)), the factor of sweep_rows_w, from
// sf[k] = sqrt(k!) and isf[k] = 1 / sqrt(k!).
__device__ inline double so4_wscale(int l, int m, int mb, const double *sf, const double *isf) {
    return (sf[m] * sf[l - m]) * (isf[mb] * isf[l - mb]);
}

// ------------------------------------------------------ su(2) generators
// U^l is a representation of SU(2): U^l(g h) = U^l(g) U^l(h) for the
// Cayley-Klein matrix g = [[conj a, -conj b], [b, a]] of an image.  Hence
// dU^l/dr_k = U^l M^l(xi_k) with xi_k = g^-1 dg/dr_k = [[i p, q], [-conj q,
// -i p]] in su(2), and M^l(xi) is tridiagonal in the column index:
//   M[m][m] = i p (l - 2m),  M[m][m+1] = c_m q,  M[m+1][m] = -c_m conj q,
//   c_m = sqrt((m + 1)(l - m)).
// Right multiplication keeps the row, so on the half rows the adjoint
// contraction of compute_duarray_recursive / compute_dbidrj (SNAP.py:
// 958-1017, 1143-1257) with Y becomes
//   Re sum conj(dU_k) Y = p_k A1 + Re q_k A2 + Im q_k A3,
//   A1 = sum (l-2m) Im(conj U_m Y_m),
//   A2 = sum c_m Re(conj U_m Y_m+1 - conj U_m+1 Y_m),
//   A3 = sum c_m Im(conj U_m Y_m+1 + conj U_m+1 Y_m),
// so the sweep needs U alone (no dU recursion, no derivative registers).
// p_k, q_k from a, b and their gradients: i p = a conj(da) + conj(b) db,
// q = conj(b) da - a conj(db).
__device__ inline void su2_generators(const CK &ck, double p[3], cd q[3]) {
#pragma unroll
    for (int k = 0; k < 3; k++) {
        const cd ca = ck.ca, cb = ck.cb, cda = ck.cda[k], cdb = ck.cdb[k];  // conjugates of a, b, da, db
        p[k] = (ca.re * cda.im - ca.im * cda.re) + (cb.im * cdb.re - cb.re * cdb.im);
        q[k] = cmake((cb.re * cda.re + cb.im * cda.im) - (ca.re * cdb.re + ca.im * cdb.im),
                     (cb.im * cda.re - cb.re * cda.im) - (ca.re * cdb.im - ca.im * cdb.re));
    }
}

// Accumulate A_u = sum Re(conj U_m Y_m) and A1..A3 (above) of one half row
// of level l (u: the row, y: Y of the same row).
template <int TWOJ>
__device__ inline void generator_dots(int l, const cd *u, const cd *y, double &au, double &a1, double &a2,
                                      double &a3) {
#pragma unroll
    for (int m = 0; m <= TWOJ; m++) {
        if (m > l) continue;
        au = fma(u[m].re, y[m].re, fma(u[m].im, y[m].im, au));
        if (l != 2 * m) a1 = fma((double)(l - 2 * m), u[m].re * y[m].im - u[m].im * y[m].re, a1);
        if (m < l) {
            const double c = sqrt((double)((m + 1) * (l - m)));  // folded per (l, m)
            const double t1 = fma(u[m].re, y[m + 1].re, u[m].im * y[m + 1].im) -
                              fma(u[m + 1].re, y[m].re, u[m + 1].im * y[m].im);
            const double t2 = fma(u[m].re, y[m + 1].im, -u[m].im * y[m + 1].re) +
                              fma(u[m + 1].re, y[m].im, -u[m + 1].im * y[m].re);
            a2 = fma(c, t1, a2);
            a3 = fma(c, t2, a3);
        }
    }
}

// One level of the W rows with nothing but multiplications: row mb of level l
// is the coefficients in x of (b + a x)^mb (conj a - conj b x)^(l - mb) (the
// inversion of row 0 of level mb is the first power), so every level
// multiplies by one of the two factors.  w[m] is zero for m > l - 1 on entry.
template <int TWOJ>
__device__ __forceinline__ void row_step_w(int l, int mb, const CK &ck, cd *w) {
    const bool up = l <= mb;
    const cd f0 = up ? cconj(ck.cb) : ck.ca, f1 = up ? cconj(ck.ca) : cmake(-ck.cb.re, -ck.cb.im);
#pragma unroll
    for (int m = TWOJ; m >= 1; m--)
        if (m <= l) w[m] = cmadd(f1, w[m - 1], cmul(f0, w[m]));
    w[0] = cmul(f0, w[0]);
}

// ---------------------------------------------------------------- U_tot
// One wavefront per centre (64 threads); NG groups of G lanes each take one
// image per round; per-group partial sums live in LDS and are reduced in a
// fixed order at the end (deterministic).  With TANGENT the kernel instead
// accumulates dU_tot . dr_e (forward-mode derivative of U_tot).
// The U_tot sums hold no derivative rows: registers are kept within three
// wavefronts per SIMD (the tangent variant needs more than that).
template <int TWOJ, bool TANGENT, bool TILED, int MODE>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(3))) void so4_accum_kernel(int64_t natoms, const int64_t *__restrict__ img_start,
                                                        const int64_t *__restrict__ img_j,
                                                        const double *__restrict__ img_r,
                                                        const double *__restrict__ atom_w,
                                                        const double *__restrict__ site_w,
                                                        const double *__restrict__ dr,
                                                        const int64_t *__restrict__ work_order, const double *rootpq_g,
                                                        const double *lnorm_g, double rcut, double rfac0, int cutoff_id,
                                                        double fcut0, double *__restrict__ out) {
    constexpr int G = TWOJ / 2 + 1;
    constexpr int NG = 64 / G;
    constexpr int NH = nhalf_of(TWOJ);
    // MODE 0: each group keeps its own partial array, summed in group order
    // at the end.  MODE 1: all groups add into one LDS array (ds_add_f64;
    // one wavefront per centre issues every add, so the order is fixed).
    // MODE 2 / 3: MODE groups share each partial array (groups g, g + NP,
    // g + 2 NP, ...); they add in MODE masked passes of one wavefront, in
    // program order: 1/MODE of the LDS, so more resident wavefronts.
    constexpr bool LDSADD = MODE == 1;
    constexpr int NPASS = MODE >= 2 ? MODE : 1;
    constexpr int NP = MODE == 1 ? 1 : (NG + NPASS - 1) / NPASS;
    __shared__ cd part[NP][NH];
    __shared__ double rpq[(TWOJ + 1) * (TWOJ + 1)];
    __shared__ double lnorm[TWOJ + 1];
    // staged per image (64 at a time): ca, cb, fc w (0: no image); with
    // TANGENT ca, cb, w fc p(eta), w fc q(eta), w dfc (rhat . dr), valid
    __shared__ double stg[TANGENT ? 9 : 5][64];
    const int lane = threadIdx.x;
    const int g = lane / G, mb = lane % G;
    for (int k = lane; k < (TWOJ + 1) * (TWOJ + 1); k += 64) rpq[k] = rootpq_g[k];
    for (int k = lane; k <= TWOJ; k += 64) lnorm[k] = lnorm_g[k];
    if (TILED && blockIdx.x == 0 && (natoms & 63)) {
        // padding lanes of the last tile (read by the Z kernel) are zero
        cd *last = reinterpret_cast<cd *>(out) + (size_t)(natoms >> 6) * NH * 64;
        for (int k = lane; k < NH * 64; k += 64)
            if ((k & 63) >= (natoms & 63)) last[k] = cmake(0.0, 0.0);
    }

    for (int64_t c = blockIdx.x; c < natoms; c += gridDim.x) {
        const int64_t i = work_order ? work_order[c] : c;
        __syncthreads();
        for (int k = lane; k < NP * NH; k += 64) (&part[0][0])[k] = cmake(0.0, 0.0);
        __syncthreads();
        const int64_t s = img_start[i], e = img_start[i + 1];
        if constexpr (!TANGENT) {
            // up to 64 images at a time: their Cayley-Klein parameters and
            // weights, one lane each, staged in LDS for the row sweeps (the G
            // lanes of an image would otherwise each compute them)
            for (int64_t b64 = s; b64 < e; b64 += 64) {
                const int64_t e64 = b64 + 64 < e ? b64 + 64 : e;
                {
                    const int64_t img = b64 + lane;
                    bool ok = img < e64;
                    double x = 0, y = 0, z = 1.0, r = 1.0, w = 0.0;
                    if (ok) {
                        x = img_r[3 * img];
                        y = img_r[3 * img + 1];
                        z = img_r[3 * img + 2];
                        r = sqrt(x * x + y * y + z * z);
                        w = atom_w[img_j[img]];
                        if (r < 1e-8) ok = false;  // SNAP.py:1487 (padding rows)
                    }
                    if (!ok) {
                        x = 0;
                        y = 0;
                        z = 1.0;
                        r = 1.0;
                    }
                    double fc, dfc;
                    cutoff_fdf(cutoff_id, r, rcut, fc, dfc);
                    CK ck;
                    cayley_klein(x, y, z, r, rfac0 * M_PI * r / rcut, false, ck);
                    stg[0][lane] = ck.ca.re;
                    stg[1][lane] = ck.ca.im;
                    stg[2][lane] = ck.cb.re;
                    stg[3][lane] = ck.cb.im;
                    stg[4][lane] = ok ? fc * w : 0.0;  // a zero weight adds nothing either way
                }
                __syncthreads();
                for (int64_t base = b64; base < e64; base += NG) {
                    const int64_t img = base + g;
                    const int si = (g < NG && img < e64) ? (int)(img - b64) : 0;
                    const bool valid = (g < NG) && (img < e64) && stg[4][si] != 0.0;
                    CK ck;
                    ck.ca = cmake(stg[0][si], stg[1][si]);
                    ck.cb = cmake(stg[2][si], stg[3][si]);
                    const double sc = stg[4][si];
                    const int pidx = g < NG ? g % NP : 0;  // index the __shared__ array itself: LDS atomics
                    sweep_rows<TWOJ, false>(mb, rpq, ck, [&](int l, const cd *u, const cd(*du)[TWOJ + 1], bool half) {
                        const bool act = valid && half;
                        const int h0 = hoff_of(l) + mb * (l + 1);
#pragma unroll
                        for (int pass = 0; pass < NPASS; pass++) {
                            // MODE >= 2: the groups sharing an array add in
                            // separate passes, ordered by workgroup barriers
                            if (act && (NPASS == 1 || g / NP == pass)) {
#pragma unroll
                                for (int m = 0; m <= TWOJ; m++) {
                                    if (m > l) continue;
                                    if (LDSADD) {
                                        atomicAdd(&part[pidx][h0 + m].re, sc * u[m].re);
                                        atomicAdd(&part[pidx][h0 + m].im, sc * u[m].im);
                                    } else {
                                        cd v = part[pidx][h0 + m];
                                        part[pidx][h0 + m] = cmake(v.re + sc * u[m].re, v.im + sc * u[m].im);
                                    }
                                }
                            }
                            if (NPASS > 1) __syncthreads();
                        }
                    });
                }
                __syncthreads();  // the next 64 images reuse the stage
            }
        } else {
            // forward-mode: dU . dr_e = U M(eta_e) with eta_e = sum_k dr_k xi_k
            // (the su(2) generators of the adjoint kernel), so a row needs U
            // alone: (U M(eta))_m = i p (l-2m) U_m + c_m-1 q U_m-1 - c_m conj(q) U_m+1
            for (int64_t b64 = s; b64 < e; b64 += 64) {
                const int64_t e64 = b64 + 64 < e ? b64 + 64 : e;
                {
                    const int64_t img = b64 + lane;
                    bool ok = img < e64;
                    double x = 0, y = 0, z = 0, r = 1.0, w = 0.0;
                    if (ok) {
                        x = img_r[3 * img];
                        y = img_r[3 * img + 1];
                        z = img_r[3 * img + 2];
                        r = sqrt(x * x + y * y + z * z);
                        w = atom_w[img_j[img]];
                        if (r < 1e-8) ok = false;  // SNAP.py:1487 (padding rows)
                    }
                    if (!ok) {
                        x = 0;
                        y = 0;
                        z = 1.0;
                        r = 1.0;
                    }
                    double fc, dfc;
                    cutoff_fdf(cutoff_id, r, rcut, fc, dfc);
                    CK ck;
                    cayley_klein(x, y, z, r, rfac0 * M_PI * r / rcut, true, ck);
                    double p[3];
                    cd q[3];
                    su2_generators(ck, p, q);
                    double d0 = 0, d1 = 0, d2 = 0;
                    if (ok) {
                        d0 = dr[3 * img];
                        d1 = dr[3 * img + 1];
                        d2 = dr[3 * img + 2];
                    }
                    const double wf = ok ? w * fc : 0.0;
                    stg[0][lane] = ck.ca.re;
                    stg[1][lane] = ck.ca.im;
                    stg[2][lane] = ck.cb.re;
                    stg[3][lane] = ck.cb.im;
                    stg[4][lane] = wf * (p[0] * d0 + p[1] * d1 + p[2] * d2);
                    stg[5][lane] = wf * (q[0].re * d0 + q[1].re * d1 + q[2].re * d2);
                    stg[6][lane] = wf * (q[0].im * d0 + q[1].im * d1 + q[2].im * d2);
                    // D . dr = fc (dU . dr) + dfc (rhat . dr) U
                    stg[7][lane] = ok ? w * dfc * (x * d0 + y * d1 + z * d2) / r : 0.0;
                    stg[8][lane] = ok ? 1.0 : 0.0;
                }
                __syncthreads();
                for (int64_t base = b64; base < e64; base += NG) {
                    const int64_t img = base + g;
                    const int si = (g < NG && img < e64) ? (int)(img - b64) : 0;
                    const bool valid = (g < NG) && (img < e64) && stg[8][si] != 0.0;
                    CK ck;
                    ck.ca = cmake(stg[0][si], stg[1][si]);
                    ck.cb = cmake(stg[2][si], stg[3][si]);
                    const double P = stg[4][si], Qr = stg[5][si], Qi = stg[6][si], Gu = stg[7][si];
                    const int pidx = g < NG ? g % NP : 0;  // index the __shared__ array itself: LDS atomics
                    sweep_rows<TWOJ, false>(mb, rpq, ck, [&](int l, const cd *u, const cd(*du)[TWOJ + 1], bool half) {
                        const bool act = valid && half;
                        const int h0 = hoff_of(l) + mb * (l + 1);
#pragma unroll
                        for (int pass = 0; pass < NPASS; pass++) {
                            if (act && (NPASS == 1 || g / NP == pass)) {
#pragma unroll
                                for (int m = 0; m <= TWOJ; m++) {
                                    if (m > l) continue;
                                    const double pm = P * (double)(l - 2 * m);
                                    double re = fma(-pm, u[m].im, Gu * u[m].re);
                                    double im = fma(pm, u[m].re, Gu * u[m].im);
                                    if (m >= 1) {
                                        const double c = sqrt((double)(m * (l - m + 1)));  // c_(m-1)
                                        re = fma(c, Qr * u[m - 1].re - Qi * u[m - 1].im, re);
                                        im = fma(c, Qr * u[m - 1].im + Qi * u[m - 1].re, im);
                                    }
                                    if (m < l) {
                                        const double c = sqrt((double)((m + 1) * (l - m)));  // c_m
                                        re = fma(-c, Qr * u[m + 1].re + Qi * u[m + 1].im, re);
                                        im = fma(-c, Qr * u[m + 1].im - Qi * u[m + 1].re, im);
                                    }
                                    if (LDSADD) {
                                        atomicAdd(&part[pidx][h0 + m].re, re);
                                        atomicAdd(&part[pidx][h0 + m].im, im);
                                    } else {
                                        cd v = part[pidx][h0 + m];
                                        part[pidx][h0 + m] = cmake(v.re + re, v.im + im);
                                    }
                                }
                            }
                            if (NPASS > 1) __syncthreads();
                        }
                    });
                }
                __syncthreads();  // the next 64 images reuse the stage
            }
        }
        __syncthreads();
        for (int h = lane; h < NH; h += 64) {
            cd acc = cmake(0.0, 0.0);
            for (int q = 0; q < NP; q++) acc = cadd(acc, part[q][h]);
            // level / row / column of h (compile-time level offsets and
            // divisors: compares and selects instead of loops and divisions)
            int l = 0, hm = 0, hma = 0;
#pragma unroll
            for (int L = 0; L <= TWOJ; L++)
                if (h >= hoff_of(L) && h < hoff_of(L + 1)) {
                    l = L;
                    hm = (h - hoff_of(L)) / (L + 1);
                    hma = (h - hoff_of(L)) % (L + 1);
                }
            if (!TANGENT && hm == hma) acc.re += fcut0 * site_w[i];  // addself_uarraytot
            acc = cscale(acc, lnorm[l]);                               // ulisttot *= u_norm
            if (TILED)  // [atom / 64][h][atom % 64], the layout of the Z kernel's loads
                reinterpret_cast<cd *>(out)[((size_t)(i >> 6) * NH + h) * 64 + (i & 63)] = acc;
            else
                reinterpret_cast<cd *>(out)[(size_t)i * NH + h] = acc;
        }
    }
}

// The per-image values the U_tot sweeps read (compute_uarray_recursive's
// a, b, SNAP.py:1515-1555, with the cutoff and weight of add_uarraytot):
// conj(a), conj(b) and w fc (0 for coincident atoms, SNAP.py:1487), and for
// the tangent w fc p(eta), w fc q(eta), w dfc (rhat . dr) and a valid flag
// in place of w fc.
template <bool TANGENT>
__device__ inline void so4_stage_image(bool ok, int64_t img, const int64_t *__restrict__ img_j,
                                       const double *__restrict__ img_r, const double *__restrict__ atom_w,
                                       const double *__restrict__ dr, double rcut, double rfac0, int cutoff_id,
                                       double *v) {
    double x = 0, y = 0, z = 1.0, r = 1.0, w = 0.0;
    if (ok) {
        x = img_r[3 * img];
        y = img_r[3 * img + 1];
        z = img_r[3 * img + 2];
        r = sqrt(x * x + y * y + z * z);
        w = atom_w[img_j[img]];
        if (r < 1e-8) ok = false;  // SNAP.py:1487 (padding rows)
    }
    if (!ok) {
        x = 0;
        y = 0;
        z = 1.0;
        r = 1.0;
    }
    double fc, dfc;
    cutoff_fdf(cutoff_id, r, rcut, fc, dfc);
    CK ck;
    cayley_klein(x, y, z, r, rfac0 * M_PI * r / rcut, TANGENT, ck);
    v[0] = ck.ca.re;
    v[1] = ck.ca.im;
    v[2] = ck.cb.re;
    v[3] = ck.cb.im;
    if constexpr (!TANGENT) {
        v[4] = ok ? fc * w : 0.0;  // a zero weight adds nothing either way
    } else {
        double p[3];
        cd q[3];
        su2_generators(ck, p, q);
        double d0 = 0, d1 = 0, d2 = 0;
        if (ok) {
            d0 = dr[3 * img];
            d1 = dr[3 * img + 1];
            d2 = dr[3 * img + 2];
        }
        const double wf = ok ? w * fc : 0.0;
        v[4] = wf * (p[0] * d0 + p[1] * d1 + p[2] * d2);
        v[5] = wf * (q[0].re * d0 + q[1].re * d1 + q[2].re * d2);
        v[6] = wf * (q[0].im * d0 + q[1].im * d1 + q[2].im * d2);
        // D . dr = fc (dU . dr) + dfc (rhat . dr) U
        v[7] = ok ? w * dfc * (x * d0 + y * d1 + z * d2) / r : 0.0;
        v[8] = ok ? 1.0 : 0.0;
    }
}

// Record stride (doubles) of the staged values: 5 (9 with the tangent) used,
// padded to 16-byte multiples.
template <bool TANGENT>
constexpr int so4_stage_stride() { return TANGENT ? 10 : 6; }

// The staged values of every image e < min(img_start[natoms], cap), one
// thread per image (grid stride): the U_tot sweep kernel then reads one
// record per image instead of evaluating the cutoff and the Cayley-Klein
// parameters between its sweeps.
template <bool TANGENT>
__global__ __launch_bounds__(256) void so4_stage_kernel(int64_t natoms, int64_t cap,
                                                        const int64_t *__restrict__ img_start,
                                                        const int64_t *__restrict__ img_j,
                                                        const double *__restrict__ img_r,
                                                        const double *__restrict__ atom_w,
                                                        const double *__restrict__ dr, double rcut, double rfac0,
                                                        int cutoff_id, double *__restrict__ stage) {
    constexpr int NS = so4_stage_stride<TANGENT>();
    const int64_t n = img_start[natoms] < cap ? img_start[natoms] : cap;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (int64_t)gridDim.x * blockDim.x) {
        double v[TANGENT ? 9 : 5];
        so4_stage_image<TANGENT>(true, e, img_j, img_r, atom_w, dr, rcut, rfac0, cutoff_id, v);
        double *o = stage + e * NS;
#pragma unroll
        for (int k = 0; k < (TANGENT ? 9 : 5); k++) o[k] = v[k];
    }
}

// U_tot (and its tangent) with the partial sums in registers.  One
// wavefront per centre, G = 2J/2+1 lanes per image as in so4_accum_kernel,
// but lane (g, mb) adds row mb of every level of all its images into
// registers (one slot per (l, m), 45 complex at 2J=8), so a centre's images
// cost no LDS traffic; once per centre the NG groups' sums are reduced in
// LDS in a fixed order (groups g < NP store, groups g + NP add, then the NP
// arrays are summed in order: deterministic).  2J <= 8 (at 2J=10 the
// register partials would exceed the register file; so4_accum_kernel).
template <int TWOJ, bool TANGENT, bool STAGED>
__device__ __forceinline__ void so4_utot_body(
    int64_t natoms, const int64_t *__restrict__ img_start, const int64_t *__restrict__ img_j,
    const double *__restrict__ img_r, const double *__restrict__ atom_w, const double *__restrict__ site_w,
    const double *__restrict__ dr, const int64_t *__restrict__ work_order, const double *rootpq_g,
    const double *lnorm_g, double rcut, double rfac0, int cutoff_id, double fcut0, double *__restrict__ out,
    const double *__restrict__ stage) {
    constexpr int G = TWOJ / 2 + 1;
    constexpr int NG = 64 / G;
    constexpr int NH = nhalf_of(TWOJ);
    constexpr int NSLOT = (TWOJ + 1) * (TWOJ + 2) / 2;  // (l, m <= l) of every level
    constexpr int NP = (NG + 1) / 2;                    // LDS partial arrays
    __shared__ cd part[NP][NH];
    __shared__ double sf[TWOJ + 1], isf[TWOJ + 1];  // sqrt(k!), 1 / sqrt(k!)
    __shared__ double lnorm[TWOJ + 1];
    // staged per image: ca, cb, fc w (0: no image); with TANGENT ca, cb,
    // w fc p(eta), w fc q(eta), w dfc (rhat . dr), valid
    __shared__ double stg[TANGENT ? 9 : 5][64];
    const int lane = threadIdx.x;
    const int g = lane / G, mb = lane % G;
    (void)rootpq_g;  // the W recursion has no coefficients
    if (lane <= TWOJ) {
        double f = 1.0;
        for (int q = 2; q <= lane; q++) f *= q;
        sf[lane] = sqrt(f);
        isf[lane] = 1.0 / sqrt(f);
    }
    for (int k = lane; k <= TWOJ; k += 64) lnorm[k] = lnorm_g[k];
    if (blockIdx.x == 0 && (natoms & 63)) {
        // padding lanes of the last tile (read by the Z kernel) are zero
        cd *last = reinterpret_cast<cd *>(out) + (size_t)(natoms >> 6) * NH * 64;
        for (int k = lane; k < NH * 64; k += 64)
            if ((k & 63) >= (natoms & 63)) last[k] = cmake(0.0, 0.0);
    }
    __syncthreads();
    for (int64_t c = blockIdx.x; c < natoms; c += gridDim.x) {
        // without a work order, the eight centres of a 64-atom tile whose
        // elements share a 128-byte line of the tile-major output run on one
        // XCD (workgroups go to the XCDs round-robin, and the grid is a
        // multiple of 8 or a single round): swap the 3-bit fields c % 8 and
        // (c / 8) % 8, a bijection on every whole tile (a partial last tile
        // keeps the identity)
        const int64_t cx = (c & ~(int64_t)63) | ((c & 7) << 3) | ((c >> 3) & 7);
        const int64_t i = work_order ? work_order[c] : ((c | 63) < natoms ? cx : c);
        const int64_t s = img_start[i], e = img_start[i + 1];
        const double wself = TANGENT ? 0.0 : site_w[i];  // loaded ahead of the sweeps
        if (s == e) {  // no image: the partial arrays start (and stay) at zero
            for (int k = lane; k < NP * NH; k += 64) part[k / NH][k % NH] = cmake(0.0, 0.0);
            __syncthreads();
        }
        for (int64_t b64 = s; b64 < e; b64 += 64) {
            const int64_t e64 = b64 + 64 < e ? b64 + 64 : e;
            if constexpr (!STAGED) {
                const int64_t img = b64 + lane;
                double v[TANGENT ? 9 : 5];
                so4_stage_image<TANGENT>(img < e64, img, img_j, img_r, atom_w, dr, rcut, rfac0, cutoff_id, v);
#pragma unroll
                for (int q = 0; q < (TANGENT ? 9 : 5); q++) stg[q][lane] = v[q];
            }
            if constexpr (!STAGED) __syncthreads();
            // the chunk's sums: live only over its sweeps (not across the
            // staging above), flushed to the partial arrays below
            cd acc[NSLOT];
#pragma unroll
            for (int q = 0; q < NSLOT; q++) acc[q] = cmake(0.0, 0.0);
            constexpr int NV = TANGENT ? 9 : 5;
            for (int64_t base = b64; base < e64; base += NG) {
                const int64_t img = base + g;
                const int si = (g < NG && img < e64) ? (int)(img - b64) : 0;
                double sv[NV];
                if constexpr (STAGED) {
                    // the group's record (loaded where it is used: a copy
                    // loaded one pass ahead costs registers, and its spills
                    // cost more than the wait: 39 against 36 us)
                    const bool ok = g < NG && img < e64;
                    const double *rec = stage + (ok ? img : b64) * so4_stage_stride<TANGENT>();
#pragma unroll
                    for (int q = 0; q < NV; q++) sv[q] = ok ? rec[q] : 0.0;
                } else {
#pragma unroll
                    for (int q = 0; q < NV; q++) sv[q] = stg[q][si];
                }
                const bool valid = (g < NG) && (img < e64) && sv[TANGENT ? 8 : 4] != 0.0;
                CK ck;
                ck.ca = cmake(sv[0], sv[1]);
                ck.cb = cmake(sv[2], sv[3]);
                if constexpr (!TANGENT) {
                    const double sc = sv[4];
                    sweep_rows_w<TWOJ>(mb, ck, [&](int l, const cd *u, bool half) {
                        if (!(valid && half)) return;
                        const int q0 = l * (l + 1) / 2;
#pragma unroll
                        for (int m = 0; m <= TWOJ; m++) {
                            if (m > l) continue;
                            acc[q0 + m].re = fma(sc, u[m].re, acc[q0 + m].re);
                            acc[q0 + m].im = fma(sc, u[m].im, acc[q0 + m].im);
                        }
                    });
                } else {
                    // dU . dr_e = U M(eta_e): (U M)_m = i p (l-2m) U_m + c_m-1 q U_m-1 - c_m conj(q) U_m+1,
                    // c_m = sqrt((m+1)(l-m)); on W (U_m = s_m W_m, s_m-1 / s_m = sqrt((l-m+1)/m))
                    // the coefficients become c_m-1 s_m-1 / s_m = l-m+1 and c_m s_m+1 / s_m = m+1
                    const double P = sv[4], Qr = sv[5], Qi = sv[6], Gu = sv[7];
                    sweep_rows_w<TWOJ>(mb, ck, [&](int l, const cd *u, bool half) {
                        if (!(valid && half)) return;
                        const int q0 = l * (l + 1) / 2;
#pragma unroll
                        for (int m = 0; m <= TWOJ; m++) {
                            if (m > l) continue;
                            const double pm = P * (double)(l - 2 * m);
                            double re = fma(-pm, u[m].im, Gu * u[m].re);
                            double im = fma(pm, u[m].re, Gu * u[m].im);
                            if (m >= 1) {
                                const double cc = (double)(l - m + 1);
                                re = fma(cc, Qr * u[m - 1].re - Qi * u[m - 1].im, re);
                                im = fma(cc, Qr * u[m - 1].im + Qi * u[m - 1].re, im);
                            }
                            if (m < l) {
                                const double cc = (double)(m + 1);
                                re = fma(-cc, Qr * u[m + 1].re + Qi * u[m + 1].im, re);
                                im = fma(-cc, Qr * u[m + 1].im - Qi * u[m + 1].re, im);
                            }
                            acc[q0 + m].re += re;
                            acc[q0 + m].im += im;
                        }
                    });
                }
            }
            __syncthreads();  // the next 64 images reuse the stage
            // reduce the NG groups' register sums: g < NP store (add after
            // the centre's first chunk), g >= NP add
#pragma unroll
            for (int pass = 0; pass < 2; pass++) {
                const bool mine = g < NG && (pass == 0 ? g < NP : g >= NP);
                const bool store = pass == 0 && b64 == s;
                const int pidx = g < NG ? (pass == 0 ? g : g - NP) : 0;
                if (mine) {
#pragma unroll
                    for (int l = 0; l <= TWOJ; l++) {
                        if (2 * mb > l) continue;
                        const int h0 = hoff_of(l) + mb * (l + 1), q0 = l * (l + 1) / 2;
#pragma unroll
                        for (int m = 0; m <= l; m++) {
                            const cd v = cscale(acc[q0 + m], so4_wscale(l, m, mb, sf, isf));
                            if (store)
                                part[pidx][h0 + m] = v;
                            else
                                part[pidx][h0 + m] = cadd(part[pidx][h0 + m], v);
                        }
                    }
                }
                __syncthreads();  // (odd NG: array NP - 1 has no second group)
            }
        }
        for (int h = lane; h < NH; h += 64) {
            cd a = cmake(0.0, 0.0);
            for (int q = 0; q < NP; q++) a = cadd(a, part[q][h]);
            int l = 0, hm = 0, hma = 0;
#pragma unroll
            for (int L = 0; L <= TWOJ; L++)
                if (h >= hoff_of(L) && h < hoff_of(L + 1)) {
                    l = L;
                    hm = (h - hoff_of(L)) / (L + 1);
                    hma = (h - hoff_of(L)) % (L + 1);
                }
            if (!TANGENT && hm == hma) a.re += fcut0 * wself;  // addself_uarraytot
            a = cscale(a, lnorm[l]);                                 // ulisttot *= u_norm
            reinterpret_cast<cd *>(out)[((size_t)(i >> 6) * NH + h) * 64 + (i & 63)] = a;
        }
        __syncthreads();  // the next centre rewrites part
    }
}

template <int TWOJ, bool TANGENT>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(1))) void so4_utot_kernel(
    int64_t natoms, const int64_t *__restrict__ img_start, const int64_t *__restrict__ img_j,
    const double *__restrict__ img_r, const double *__restrict__ atom_w, const double *__restrict__ site_w,
    const double *__restrict__ dr, const int64_t *__restrict__ work_order, const double *rootpq_g,
    const double *lnorm_g, double rcut, double rfac0, int cutoff_id, double fcut0, double *__restrict__ out) {
    so4_utot_body<TWOJ, TANGENT, false>(natoms, img_start, img_j, img_r, atom_w, site_w, dr, work_order, rootpq_g,
                                        lnorm_g, rcut, rfac0, cutoff_id, fcut0, out, nullptr);
}

// U_tot from the staged per-image records (so4_stage_kernel): without the
// cutoff and Cayley-Klein evaluation between its sweeps the kernel fits two
// wavefronts per SIMD.  A wavefront per centre: for lists too short to fill
// the chip with the wavefronts of so4_utot_group_kernel.
template <int TWOJ>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void so4_utot_staged_kernel(
    int64_t natoms, const int64_t *__restrict__ img_start, const double *__restrict__ site_w,
    const int64_t *__restrict__ work_order, const double *lnorm_g, double fcut0, const double *__restrict__ stage,
    double *__restrict__ out) {
    so4_utot_body<TWOJ, false, true>(natoms, img_start, nullptr, nullptr, nullptr, site_w, nullptr, work_order,
                                     nullptr, lnorm_g, 0.0, 0.0, 1, fcut0, out, stage);
}

// The same for long lists.  G lanes (one
// per row mb) go through images as in so4_utot_body, sums in registers, but a
// centre gets only `split` of the wavefront's NG lane groups, and the
// wavefront NG / split centres: with one group per centre nothing is summed
// across lanes at all, and every centre fewer groups saves their share of the
// LDS traffic of that sum, which took longer than the sweeps.  The groups of
// a centre are added in halves (fixed order).  Neighbouring centres share a
// wavefront, so their elements of the tile-major output share lines.
// Two wavefronts per SIMD (registers: 45 complex sums at 2J = 8).
// Against the wavefront per centre (with the staging of the records): 4096
// atoms (28 images, 2J = 8, three groups to a centre) 36 -> 29 us, 32768 233 ->
// 121, 110592 760 -> 396, 120000 of 32 images on average 851 -> 547; 4096 atoms
// at 2J = 6 22 -> 20.  The tangent (with the dB sum, 2J = 8): 4096 atoms 129 ->
// 113 us, 32768 718 -> 525, 33000 of 32 images 808 -> 670.
template <int TWOJ, bool TANGENT>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(2))) void so4_utot_group_kernel(
    int64_t natoms, int split, const int64_t *__restrict__ img_start, const double *__restrict__ site_w,
    const double *__restrict__ lnorm_g, double fcut0, int64_t cap, const double *__restrict__ stage,
    double *__restrict__ out) {
    constexpr int G = TWOJ / 2 + 1;
    constexpr int NG = 64 / G;
    constexpr int NH = nhalf_of(TWOJ);
    constexpr int NSLOT = (TWOJ + 1) * (TWOJ + 2) / 2;  // (l, m <= l) of every level
    constexpr int NS = so4_stage_stride<TANGENT>();
    __shared__ cd part[NG / 2][NH];
    __shared__ double sf[TWOJ + 1], isf[TWOJ + 1];  // sqrt(k!), 1 / sqrt(k!)
    const int lane = threadIdx.x;
    const int g = lane / G, mb = lane % G;
    if (lane <= TWOJ) {
        double f = 1.0;
        for (int q = 2; q <= lane; q++) f *= q;
        sf[lane] = sqrt(f);
        isf[lane] = 1.0 / sqrt(f);
    }
    if (blockIdx.x == 0 && (natoms & 63)) {
        // padding lanes of the last tile (read by the Z kernel) are zero
        cd *last = reinterpret_cast<cd *>(out) + (size_t)(natoms >> 6) * NH * 64;
        for (int k = lane; k < NH * 64; k += 64)
            if ((k & 63) >= (natoms & 63)) last[k] = cmake(0.0, 0.0);
    }
    const int cpw = NG / split, c = g / split, p = g - c * split;
    const int64_t i = (int64_t)blockIdx.x * cpw + c;
    const bool mine = c < cpw && i < natoms;
    // images past the cap staged records have none
    const int64_t s = mine ? img_start[i] : 0, s1 = mine ? min(img_start[i + 1], cap) : 0;
    const int n = s1 > s ? (int)(s1 - s) : 0;
    const double wself = mine && !TANGENT ? site_w[i] : 0.0;
    cd acc[NSLOT];
#pragma unroll
    for (int q = 0; q < NSLOT; q++) acc[q] = cmake(0.0, 0.0);
    // the wavefront's longest centre bounds the loop: with a bound per lane
    // the sums were held twice around it (140 spilled registers)
    int most = n;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o));
    most = __builtin_amdgcn_readfirstlane(most);
#pragma unroll 1
    for (int k0 = 0; k0 < most; k0 += split) {
        const int k = k0 + p;
        const bool ok = k < n;
        const double *rec = stage + (s + (ok ? k : 0)) * NS;
        CK ck;
        ck.ca = cmake(1.0, 0.0);
        ck.cb = cmake(0.0, 0.0);
        double sc = 0.0, Qr = 0.0, Qi = 0.0, Gu = 0.0;  // TANGENT: sc is p(eta)
        if (ok) {
            ck.ca = cmake(rec[0], rec[1]);
            ck.cb = cmake(rec[2], rec[3]);
            sc = rec[4];
            if (TANGENT) {
                Qr = rec[5];
                Qi = rec[6];
                Gu = rec[7];
            }
        }
        cd w[TWOJ + 1];
#pragma unroll
        for (int m = 0; m <= TWOJ; m++) w[m] = cmake(m == 0 ? 1.0 : 0.0, 0.0);
        // (the rows above the half add to sums that are not written)
#pragma unroll
        for (int l = 0; l <= TWOJ; l++) {
            if (l > 0) row_step_w<TWOJ>(l, mb, ck, w);
            const int q0 = l * (l + 1) / 2;
#pragma unroll
            for (int m = 0; m <= TWOJ; m++) {
                if (m > l) continue;
                cd &a = acc[q0 + m];
                if constexpr (!TANGENT) {
                    a.re = fma(sc, w[m].re, a.re);
                    a.im = fma(sc, w[m].im, a.im);
                } else {
                    // (U M(eta))_m on W as in so4_utot_body
                    const double pm = sc * (double)(l - 2 * m);
                    double re = fma(-pm, w[m].im, Gu * w[m].re);
                    double im = fma(pm, w[m].re, Gu * w[m].im);
                    if (m >= 1) {
                        const double cc = (double)(l - m + 1);
                        re = fma(cc, Qr * w[m - 1].re - Qi * w[m - 1].im, re);
                        im = fma(cc, Qr * w[m - 1].im + Qi * w[m - 1].re, im);
                    }
                    if (m < l) {
                        const double cc = (double)(m + 1);
                        re = fma(-cc, Qr * w[m + 1].re + Qi * w[m + 1].im, re);
                        im = fma(-cc, Qr * w[m + 1].im - Qi * w[m + 1].re, im);
                    }
                    a.re += re;
                    a.im += im;
                }
            }
        }
    }
    // groups [half, cnt) of every centre into its groups [0, cnt - half)
    for (int cnt = split; cnt > 1;) {
        const int half = (cnt + 1) / 2, src = p - half;
        __syncthreads();
        if (c < cpw && src >= 0 && p < cnt) {
            cd *o = part[c * (split / 2) + src];
#pragma unroll
            for (int l = 0; l <= TWOJ; l++)
#pragma unroll
                for (int m = 0; m <= l; m++)
                    if (2 * mb <= l) o[hoff_of(l) + mb * (l + 1) + m] = acc[l * (l + 1) / 2 + m];
        }
        __syncthreads();
        {
            // no branch around the additions: the sums of both ways would be
            // held side by side
            const bool add = c < cpw && p + half < cnt;
            const cd *o = part[add ? c * (split / 2) + p : 0];
#pragma unroll
            for (int l = 0; l <= TWOJ; l++)
#pragma unroll
                for (int m = 0; m <= l; m++) {
                    const bool on = add && 2 * mb <= l;
                    const cd v = o[on ? hoff_of(l) + mb * (l + 1) + m : 0];
                    cd &t = acc[l * (l + 1) / 2 + m];
                    t.re += on ? v.re : 0.0;
                    t.im += on ? v.im : 0.0;
                }
        }
        cnt = half;
    }
    __syncthreads();  // sf, isf
    if (!mine || p != 0) return;
    cd *o = reinterpret_cast<cd *>(out) + (size_t)(i >> 6) * NH * 64 + (i & 63);
#pragma unroll
    for (int l = 0; l <= TWOJ; l++) {
        if (2 * mb > l) continue;
        const double ln = lnorm_g[l];
#pragma unroll
        for (int m = 0; m <= l; m++) {
            cd a = cscale(acc[l * (l + 1) / 2 + m], so4_wscale(l, m, mb, sf, isf));
            if (!TANGENT && m == mb) a.re += fcut0 * wself;  // addself_uarraytot
            o[(size_t)(hoff_of(l) + mb * (l + 1) + m) * 64] = cscale(a, ln);  // ulisttot *= u_norm
        }
    }
}

// B (compute_bi, SNAP.py:1101-1141) from the tile-major U_tot and Z: one
// atom per lane (64-atom tiles, so the U_tot loads are coalesced), the
// components b spread over the wavefronts of a tile (grid.y); loop bounds
// are wave-uniform.
template <int TWOJ>
__global__ __launch_bounds__(256) void so4_b_kernel(int64_t natoms, const double *__restrict__ utile,
                                                     const double *__restrict__ z, int nz, int nb,
                                                     const int *__restrict__ b_zoff, const int *__restrict__ b_level,
                                                     double *__restrict__ bout) {
    constexpr int NH = nhalf_of(TWOJ);
    const int lane = threadIdx.x & 63;
    const int w = blockIdx.y * 4 + (threadIdx.x >> 6), nw = gridDim.y * 4;
    const int64_t tile = blockIdx.x;
    const int64_t i = tile * 64 + lane;
    if (i >= natoms) return;
    const cd *ut = reinterpret_cast<const cd *>(utile) + (size_t)tile * NH * 64 + lane;
    const cd *zi = reinterpret_cast<const cd *>(z) + (size_t)tile * nz * 64 + lane;  // Z tile-major
    for (int b = w; b < nb; b += nw) {
        const int l = __builtin_amdgcn_readfirstlane(b_level[b]);
        const int z0 = __builtin_amdgcn_readfirstlane(b_zoff[b]);
        const int h0 = hoff_of(l);
        // rows mb < l/2 in full, then (l even) the middle row up to the
        // diagonal, whose element counts half
        const int nfull = ((l + 1) / 2) * (l + 1);
        double s = 0.0;
#pragma unroll 8
        for (int q = 0; q < nfull; q++) s += cdotre(ut[(size_t)(h0 + q) * 64], zi[(size_t)(z0 + q) * 64]);
        if ((l & 1) == 0) {
            const int mb = l / 2;
#pragma unroll 4
            for (int q = nfull; q < nfull + mb; q++)
                s += cdotre(ut[(size_t)(h0 + q) * 64], zi[(size_t)(z0 + q) * 64]);
            s += 0.5 * cdotre(ut[(size_t)(h0 + nfull + mb) * 64], zi[(size_t)(z0 + nfull + mb) * 64]);
        }
        bout[(size_t)i * nb + b] = 2.0 * s;
    }
}

// ---------------------------------------------------------------------- Y
// Y[h] = 2 hw(h) norm_l sum_{blocks k at level l} c_k Z[k][loc(h)],
// c_k = sum_targets f beta[b].  One atom per lane over a 64-atom tile, like
// the Z kernel whose tile-major output it reads: a wavefront owns one task
// (a run of at most YTASK_ROWS half elements of one level), loops over the
// level's blocks in order (fixed summation order, no atomics) and adds
// c_k Z[k][loc] into register accumulators; every Z load is a coalesced
// 1 KB row and every Z element is read by exactly one wavefront.  The four
// wavefronts of a workgroup take four tasks of the same tile and share its
// dE/dB rows, staged in LDS.
__global__ __launch_bounds__(256) void so4_yi_kernel(int64_t natoms, int ntasks, int nz, int nb, int nhalf,
                                                      const int *__restrict__ ytask, const double *__restrict__ z,
                                                      const double *__restrict__ beta,
                                                      const int *__restrict__ blk_zoff, const int *__restrict__ blk_tb,
                                                      const double *__restrict__ blk_tf,
                                                      const double *__restrict__ hscale, double *__restrict__ y) {
    extern __shared__ double sb[];  // [64][nb] dE/dB of the tile (zero beyond natoms)
    const int tg = (ntasks + 3) / 4;
    const int64_t tile = blockIdx.x / tg;
    const int task = (int)(blockIdx.x % tg) * 4 + (threadIdx.x >> 6);
    const int lane = threadIdx.x & 63;
    const int64_t a0 = tile * 64;
    const int64_t nv = (natoms - a0 < 64 ? natoms - a0 : 64) * nb;
    for (int64_t k = threadIdx.x; k < 64 * (int64_t)nb; k += blockDim.x) sb[k] = k < nv ? beta[a0 * nb + k] : 0.0;
    __syncthreads();
    if (task >= ntasks) return;
    const int *T = ytask + YTASK_STRIDE * task;
    const int loc0 = __builtin_amdgcn_readfirstlane(T[1]);
    const int cnt = __builtin_amdgcn_readfirstlane(T[2]);
    const int k0 = __builtin_amdgcn_readfirstlane(T[3]);
    const int k1 = __builtin_amdgcn_readfirstlane(T[4]);
    const int h0 = __builtin_amdgcn_readfirstlane(T[5]);
    const double *bl = sb + lane * nb;
    const cd *zt = reinterpret_cast<const cd *>(z) + (size_t)tile * nz * 64 + lane;
    cd acc[YTASK_ROWS];
#pragma unroll
    for (int q = 0; q < YTASK_ROWS; q++) acc[q] = cmake(0.0, 0.0);
    // YB blocks per step, so that their Z loads are in flight together
    constexpr int YB = 4;
    for (int kb = k0; kb < k1; kb += YB) {
        double c[YB];
        cd v[YB][YTASK_ROWS];
#pragma unroll
        for (int u = 0; u < YB; u++) {
            const int k = kb + u;
            c[u] = 0.0;
            if (k < k1) {
                const cd *zk = zt + (size_t)(__builtin_amdgcn_readfirstlane(blk_zoff[k]) + loc0) * 64;
#pragma unroll
                for (int q = 0; q < YTASK_ROWS; q++)
                    if (q < cnt) v[u][q] = zk[q * 64];
#pragma unroll
                for (int t = 0; t < 3; t++) {
                    const int b = __builtin_amdgcn_readfirstlane(blk_tb[3 * k + t]);
                    if (b >= 0) c[u] += blk_tf[3 * k + t] * bl[b];
                }
            }
        }
#pragma unroll
        for (int u = 0; u < YB; u++)
            if (kb + u < k1) {
#pragma unroll
                for (int q = 0; q < YTASK_ROWS; q++)
                    if (q < cnt) {
                        acc[q].re += c[u] * v[u][q].re;
                        acc[q].im += c[u] * v[u][q].im;
                    }
            }
    }
    if (a0 + lane < natoms) {
        cd *yo = reinterpret_cast<cd *>(y) + (size_t)(a0 + lane) * nhalf + h0;
#pragma unroll
        for (int q = 0; q < YTASK_ROWS; q++)
            if (q < cnt) yo[q] = cscale(acc[q], hscale[h0 + q]);
    }
}

// -------------------------------------------------------- adjoint dE/dr
constexpr int DEIDRJ_NST = 16;  // staged doubles per image of the dE/dr kernel
// Flat over images: a wavefront serves NB = nr x NG images (any centres).
// It first stages, one lane per image, the Cayley-Klein parameters and the
// per-image factors of the generator contraction in LDS (the G lanes of an
// image would otherwise each compute them), then sweeps them in nr rounds
// of NG images (nr is chosen by the launch so that the grid holds enough
// wavefronts to hide latency):
//   dE/dr_k = w fc (p_k A1 + Re q_k A2 + Im q_k A3) + w dfc rhat_k A_u.
template <int TWOJ>
__global__ __launch_bounds__(256) void so4_deidrj_kernel(int64_t nimg, const int64_t *__restrict__ img_atom,
                                                           const int64_t *__restrict__ img_j,
                                                           const double *__restrict__ img_r,
                                                           const double *__restrict__ atom_w,
                                                           const double *__restrict__ y, const double *rootpq_g,
                                                           double rcut, double rfac0, int cutoff_id,
                                                           double *__restrict__ dedr,
                                                           const int64_t *__restrict__ d_count, int nr) {
    constexpr int G = TWOJ / 2 + 1;
    constexpr int NG = 64 / G;
    const int NB = NG * nr;  // images per wavefront (nr rounds, nr <= 64 / NG)
    constexpr int NST = DEIDRJ_NST;
    constexpr int NH = nhalf_of(TWOJ);
    __shared__ double rpq[(TWOJ + 1) * (TWOJ + 1)];
    // per wavefront (dynamic, sized by the launch's wavefronts per block):
    // NST x 64 staged doubles, 64 x 4 partial sums, 64 centre indices
    extern __shared__ double dsm[];
    // with d_count the grid covers an image capacity and the images in use
    // are counted on the device
    if (d_count) {
        const int64_t c = *d_count;
        nimg = c < nimg ? c : nimg;
    }
    const int tid = threadIdx.x;
    const int wv = tid >> 6, lane = tid & 63;
    const int wpb = blockDim.x >> 6;
    const int g = lane / G, mb = lane % G;
    for (int k = tid; k < (TWOJ + 1) * (TWOJ + 1); k += blockDim.x) rpq[k] = rootpq_g[k];
    __syncthreads();
    const int64_t base = ((int64_t)blockIdx.x * wpb + wv) * NB;
    // a wavefront past the images in use (a launch over an image capacity)
    // has nothing to do; the later synchronisation is wavefront-local
    if (base >= nimg) return;
    double(*S)[64] = reinterpret_cast<double(*)[64]>(dsm + (size_t)wv * (NST + 5) * 64);
    double(*red)[4] = reinterpret_cast<double(*)[4]>(dsm + (size_t)wv * (NST + 5) * 64 + NST * 64);
    int64_t *s_at = reinterpret_cast<int64_t *>(dsm + (size_t)wv * (NST + 5) * 64 + (NST + 4) * 64);
    {
        const int64_t img = base + lane;
        bool ok = lane < NB && img < nimg;
        double x = 0, yy = 0, zz = 1.0, r = 1.0, w = 0.0;
        int64_t i = -1;
        if (ok) {
            x = img_r[3 * img];
            yy = img_r[3 * img + 1];
            zz = img_r[3 * img + 2];
            r = sqrt(x * x + yy * yy + zz * zz);
            w = atom_w[img_j[img]];
            i = img_atom[img];
            if (r < 1e-8) ok = false;  // SNAP.py:1487 (padding rows)
        }
        if (!ok) {
            x = 0;
            yy = 0;
            zz = 1.0;
            r = 1.0;
        }
        double fc, dfc;
        cutoff_fdf(cutoff_id, r, rcut, fc, dfc);
        CK ck;
        cayley_klein(x, yy, zz, r, rfac0 * M_PI * r / rcut, true, ck);
        double p[3];
        cd q[3];
        su2_generators(ck, p, q);
        S[0][lane] = ck.ca.re;
        S[1][lane] = ck.ca.im;
        S[2][lane] = ck.cb.re;
        S[3][lane] = ck.cb.im;
        const double wf = w * fc, wd = w * dfc / r;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            S[4 + k][lane] = wf * p[k];
            S[7 + k][lane] = wf * q[k].re;
            S[10 + k][lane] = wf * q[k].im;
        }
        S[13][lane] = wd * x;
        S[14][lane] = wd * yy;
        S[15][lane] = wd * zz;
        s_at[lane] = ok ? i : -1;
    }
    // the rounds read lanes of the same wavefront only
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    for (int rd = 0; rd < nr; rd++) {
        if (base + rd * NG >= nimg) break;  // uniform
        const int slot = rd * NG + (g < NG ? g : 0);
        const int64_t i = s_at[slot];
        const bool valid = g < NG && i >= 0;
        CK ck;
        ck.ca = cmake(S[0][slot], S[1][slot]);
        ck.cb = cmake(S[2][slot], S[3][slot]);
        const cd *yi = reinterpret_cast<const cd *>(y) + (size_t)(valid ? i : 0) * NH;
        double au = 0.0, a1 = 0.0, a2 = 0.0, a3 = 0.0;
        sweep_rows<TWOJ, false>(mb, rpq, ck, [&](int l, const cd *u, const cd(*du)[TWOJ + 1], bool half) {
            if (!valid || !half) return;
            const cd *yr = yi + hoff_of(l) + mb * (l + 1);
            cd yv[TWOJ + 1];
#pragma unroll
            for (int m = 0; m <= TWOJ; m++)
                if (m <= l) yv[m] = yr[m];
            generator_dots<TWOJ>(l, u, yv, au, a1, a2, a3);
        });
        red[lane][0] = au;
        red[lane][1] = a1;
        red[lane][2] = a2;
        red[lane][3] = a3;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        if (valid && mb == 0) {
            double sm[4] = {0, 0, 0, 0};
            for (int qq = 0; qq < G; qq++)
                for (int k = 0; k < 4; k++) sm[k] += red[lane + qq][k];
            const int64_t img = base + slot;
            for (int k = 0; k < 3; k++)
                dedr[3 * img + k] = S[4 + k][slot] * sm[1] + S[7 + k][slot] * sm[2] + S[10 + k][slot] * sm[3] +
                                    S[13 + k][slot] * sm[0];
        } else if (g < NG && mb == 0 && base + slot < nimg) {
            // an image of coincident atoms (r < 1e-8) contributes nothing, as
            // the reference skips it (SNAP.py:1487)
            const int64_t img = base + slot;
            for (int k = 0; k < 3; k++) dedr[3 * img + k] = 0.0;
        }
        // the next round rewrites red
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
}

// --------------------------------------------------- plain dB/dr per image
// One wavefront per NG images.  Level by level the groups put their D rows
// (D_k = fc dU_k + dfc rhat_k U, i.e. dU_tot/dr without w and u_norm) into
// LDS; then all 64 lanes form the block inner products
// p[blk][k] = Re <D_k^l, 2 hw norm_l Z^blk> of that level and add w f p to
// every (b, factor) target of the block -- the three terms of
// compute_dbidrj (SNAP.py:1143-1257).  Within one level a (b, k) output
// receives at most one block, so the accumulation needs no atomics.
template <int TWOJ>
__global__ __launch_bounds__(64) void so4_dbdr_kernel(
    int64_t nimg, const int64_t *__restrict__ img_atom, const int64_t *__restrict__ img_j,
    const double *__restrict__ img_r, const double *__restrict__ atom_w, const double *__restrict__ z, int nz, int nb,
    const double *rootpq_g, const double *__restrict__ lnorm, const int *__restrict__ blk_level_start,
    const int *__restrict__ blk_zoff, const int *__restrict__ blk_tb, const double *__restrict__ blk_tf, double rcut,
    double rfac0, int cutoff_id, double *__restrict__ dbdr) {
    constexpr int G = TWOJ / 2 + 1;
    constexpr int NG = 64 / G;
    constexpr int NL = (TWOJ / 2 + 1) * (TWOJ + 1);
    constexpr int NBMAX = nb_of(TWOJ);
    __shared__ double rpq[(TWOJ + 1) * (TWOJ + 1)];
    __shared__ cd Dl[NG][3][NL];
    __shared__ double acc[NG][NBMAX * 3];
    __shared__ int64_t s_atom[NG];
    __shared__ double s_w[NG];
    const int lane = threadIdx.x;
    const int g = lane / G, mb = lane % G;
    for (int k = lane; k < (TWOJ + 1) * (TWOJ + 1); k += 64) rpq[k] = rootpq_g[k];
    for (int k = lane; k < NG * NBMAX * 3; k += 64) (&acc[0][0])[k] = 0.0;
    const int64_t img = (int64_t)blockIdx.x * NG + g;
    bool valid = (g < NG) && (img < nimg);
    double x = 0, yy = 0, zz = 1.0, r = 1.0, w = 0.0;
    if (valid) {
        x = img_r[3 * img];
        yy = img_r[3 * img + 1];
        zz = img_r[3 * img + 2];
        r = sqrt(x * x + yy * yy + zz * zz);
        w = atom_w[img_j[img]];
        if (r < 1e-8) {
            valid = false;
            x = 0;
            yy = 0;
            zz = 1.0;
            r = 1.0;
        }
    }
    if (g < NG && mb == 0) {
        s_atom[g] = valid ? img_atom[img] : -1;
        s_w[g] = w;
    }
    double fc, dfc;
    cutoff_fdf(cutoff_id, r, rcut, fc, dfc);
    const double rh[3] = {x / r, yy / r, zz / r};
    CK ck;
    cayley_klein(x, yy, zz, r, rfac0 * M_PI * r / rcut, true, ck);
    __syncthreads();
    sweep_rows<TWOJ, true>(mb, rpq, ck, [&](int l, const cd *u, const cd(*du)[TWOJ + 1], bool half) {
        if (g < NG && half) {
#pragma unroll
            for (int m = 0; m <= TWOJ; m++) {
                if (m > l) continue;
#pragma unroll
                for (int k = 0; k < 3; k++)
                    Dl[g][k][mb * (l + 1) + m] = cmake(fc * du[k][m].re + dfc * rh[k] * u[m].re,
                                                       fc * du[k][m].im + dfc * rh[k] * u[m].im);
            }
        }
        __syncthreads();
        const int b0 = blk_level_start[l], nbl = blk_level_start[l + 1] - b0;
        const int nloc = (l / 2 + 1) * (l + 1);
        const double nrm2 = 2.0 * lnorm[l];
        for (int it = lane; it < NG * nbl * 3; it += 64) {
            const int gg = it / (nbl * 3);
            const int rem = it - gg * nbl * 3;
            const int bk = rem / 3, k = rem - bk * 3;
            const int64_t a = s_atom[gg];
            if (a < 0) continue;
            const int blk = b0 + bk;
            // atom-major Z: each lane walks one contiguous block row
            const cd *zb = reinterpret_cast<const cd *>(z) + (size_t)a * nz + blk_zoff[blk];
            double p = 0.0;
            int loc = 0;
            for (int hm = 0; 2 * hm < l; hm++)
                for (int ma = 0; ma <= l; ma++, loc++) p += cdotre(Dl[gg][k][loc], zb[loc]);
            if ((l & 1) == 0) {
                const int hm = l / 2;
                for (int ma = 0; ma < hm; ma++, loc++) p += cdotre(Dl[gg][k][loc], zb[loc]);
                p += 0.5 * cdotre(Dl[gg][k][loc], zb[loc]);
            }
            (void)nloc;
            p *= nrm2 * s_w[gg];
#pragma unroll
            for (int s = 0; s < 3; s++) {
                const int b = blk_tb[3 * blk + s];
                if (b >= 0) acc[gg][3 * b + k] += blk_tf[3 * blk + s] * p;
            }
        }
        __syncthreads();
    });
    for (int gg = 0; gg < NG; gg++) {
        const int64_t im = (int64_t)blockIdx.x * NG + gg;
        if (im >= nimg) break;
        for (int k = lane; k < nb * 3; k += 64) dbdr[(size_t)im * nb * 3 + k] = acc[gg][k];
    }
}

// --------------------------------------- plain dB/dr, one centre per workgroup
// dB/dr of every image of a centre on the FP64 matrix cores.  With the su(2)
// generators of an image (su2_generators) and W the rows of sweep_rows_w,
//   dB_b/dr_k = w [fc (p_k A1 + Re q_k A2 + Im q_k A3) + dfc rhat_k Au]_b,
// each A_q of component b a real inner product over the half elements of
// three levels: of W of the image with
//   V_q = sum over the blocks targeting b (compute_dbidrj, SNAP.py:1143-1257)
//         of 2 f norm_l (generator q applied to the block's weighted Z rows),
// and V_q depends on the centre only.  So per centre it is a product of a
// matrix with four rows (q) per b by a matrix with a column per image, the
// sum running over (level, half element, re / im).  Level by level the
// workgroup puts the images' W rows (one thread per image and row) and the
// centre's Z blocks (half weights applied) into LDS; a wavefront forms the
// operand V_q of its tiles of four b from two Z values and two coefficients
// (generator, sqrt factors of W) and keeps the sums of up to 16 b and 48
// images in registers over all levels, so the outputs are written once.
// Rows of a 16x16x4 tile are (q, b), so that a lane ends up with all four
// sums of its (b, image).
// Levels go in stages, runs of levels whose values share a W row, so that the
// workgroup meets at a barrier twice per stage and not per level.
// A tile of four b costs the union of their levels: the b are grouped for
// small unions (2J = 8: 440 steps of four products per 16 images against 304
// for each b alone and 523 in index order).
// Bound by latency, two workgroups per CU (registers): of 95k cycles of a
// workgroup at 2J = 8 the products take 48k, the W rows and their barriers
// 30k, the prologue 16k.  4096 atoms (115k images), 2J = 8: 620 -> 398 us;
// 1728 atoms: 264 -> 180 us.  The
// forerunner summed one (image, block) per lane on the vector units and added
// to the output rows level by level (0.9 GB read and 0.9 GB written for 157 MB
// of output).  Measured beside it (4096 atoms): eight wavefronts of half the
// tiles 525 us, a stage per level 474 us.
typedef double db_d4 __attribute__((ext_vector_type(4)));
template <int TWOJ>
struct DbDim {
    static constexpr int NW = db_waves(TWOJ);
    static constexpr int T = 64 * NW;
    static constexpr int G = TWOJ / 2 + 1;
    static constexpr int NT = TWOJ <= 8 ? 3 : 2;  // tiles of 16 images per pass
    static constexpr int NI = 16 * NT;
    static constexpr int KS = db_stride(TWOJ);  // W row: the values of the longest stage
    static constexpr int TW = ((nb_of(TWOJ) + 3) / 4 + NW - 1) / NW;  // tiles per wavefront
    static constexpr int NSLOT = NW * TW * 4;
    static constexpr int ZP = (db_stage_zmax(TWOJ) + T - 1) / T;       // Z elements of a stage per thread
    static constexpr int CP = (db_steps(TWOJ) * 16 + T - 1) / T;       // coefficient pairs
    static_assert(NI * G <= T, "one thread per (image, row)");
    static_assert(16 * 3 * nb_of(TWOJ) <= NI * KS, "the output tile reuses the W rows");
};

struct DbArgs {
    const int64_t *__restrict__ img_start, *__restrict__ img_j;
    const double *__restrict__ img_r, *__restrict__ atom_w, *__restrict__ zt;
    int nz, cutoff_id, z_atom_major, nstage;
    const int *__restrict__ db_tile, *__restrict__ db_row;
    const double *__restrict__ db_fac, *__restrict__ db_coef;
    const int *__restrict__ db_zmap, *__restrict__ db_stage;
    double rcut, rfac0;
};

// One pass: images [e0, e0 + ne), ne <= NI, of centre c.
template <int TWOJ>
__device__ __forceinline__ void so4_dbdr_pass(const DbArgs &A, int64_t c, int64_t e0, int ne, double *__restrict__ dbdr) {
    using D = DbDim<TWOJ>;
    constexpr int T = D::T, G = D::G, NT = D::NT, NI = D::NI, KS = D::KS, TW = D::TW;
    constexpr int NB = nb_of(TWOJ), NSLOT = D::NSLOT, ZP = D::ZP, CP = D::CP, NL = TWOJ + 1;
    // the operand loads run up to five steps past a level's last (their
    // values are not used): slack behind each array
    constexpr int PAD = 5 * 4, ZLEN = db_stage_zlds(TWOJ) + PAD;
    __shared__ __attribute__((aligned(16))) double Ul[NI * KS + PAD];
    __shared__ __attribute__((aligned(16))) double Zl[ZLEN];
    __shared__ double2 Cl[(db_steps(TWOJ) + 5) * 16];
    __shared__ double s_fac[NL * NSLOT];
    __shared__ int s_row[NL * NSLOT], s_b[NSLOT];
    __shared__ double sc[NI][12];  // w fc p_k, w fc Re q_k, w fc Im q_k, w dfc rhat_k
    __shared__ cd sck[NI][2];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int nt = (ne + 15) / 16;
    const cd *zc = reinterpret_cast<const cd *>(A.zt) + (A.z_atom_major ? (size_t)c * A.nz
                                                                          : (size_t)(c >> 6) * A.nz * 64 + (c & 63));
    const int zs = A.z_atom_major ? 1 : 64;
    // per stage s: {first Z element, first coefficient pair, first level}
    __shared__ int stg[3 * (NL + 1)];
    if (tid < 3 * (A.nstage + 1)) stg[tid] = A.db_stage[tid];
    const int2 *zmap = reinterpret_cast<const int2 *>(A.db_zmap);
    // the centre's Z blocks and the coefficients of a stage are loaded one
    // stage ahead of their use, the places of its Z elements two
    int2 mp[ZP];
    cd zv[ZP];
    int zp[ZP];
    cd cv[CP];
    auto places = [&](int s) __attribute__((always_inline)) {
        const int z0 = stg[3 * s], z1 = stg[3 * s + 3];
#pragma unroll
        for (int u = 0; u < ZP; u++) mp[u] = z0 + u * T + tid < z1 ? zmap[z0 + u * T + tid] : make_int2(0, -1);
    };
    auto fetch = [&](int s) __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < ZP; u++) {
            zp[u] = mp[u].y;
            zv[u] = zc[(size_t)mp[u].x * zs];  // (places without an element read element 0)
        }
        const int c0 = stg[3 * s + 1], c1 = stg[3 * s + 4];
#pragma unroll
        for (int u = 0; u < CP; u++) {
            const int k = c0 + u * T + tid;
            cv[u] = reinterpret_cast<const cd *>(A.db_coef)[k < c1 ? k : c0];
        }
    };
    __syncthreads();
    places(0);
    // this image's record while the tables are on their way
    double x = 0, yy = 0, zz = 1.0, wn = 0.0;
    if (tid < ne) {
        const int64_t e = e0 + tid;
        x = A.img_r[3 * e];
        yy = A.img_r[3 * e + 1];
        zz = A.img_r[3 * e + 2];
        wn = A.atom_w[A.img_j[e]];
    }
    for (int k = tid; k < NL * NSLOT; k += T) {
        s_row[k] = A.db_row[k];
        s_fac[k] = A.db_fac[k];
    }
    // levels of this wavefront's tiles, and the component of every slot
    int tmask[TW];
    static_for<TW>([&](auto TT) __attribute__((always_inline)) {
        constexpr int t = decltype(TT)::value;
        tmask[t] = __builtin_amdgcn_readfirstlane(A.db_tile[wv * TW + t]);
    });
    for (int k = tid; k < NSLOT; k += T) s_b[k] = A.db_tile[D::NW * TW + k];
    for (int k = tid; k < (NI * KS + PAD) / 2; k += T) reinterpret_cast<double2 *>(Ul)[k] = make_double2(0.0, 0.0);
    for (int k = tid; k < ZLEN / 2; k += T) reinterpret_cast<double2 *>(Zl)[k] = make_double2(0.0, 0.0);
    for (int k = tid; k < (db_steps(TWOJ) + 5) * 16; k += T) Cl[k] = make_double2(0.0, 0.0);
    fetch(0);
    if (A.nstage > 1) places(1);
    // operand roles of the lane: A row (q, b) and k', B column = image
    const int q = (lane & 15) >> 2, bl = lane & 3, kp = lane >> 4, par = kp & 1;
    const int sw = par ? -1 : 1;  // the other part of the same element
    const int off1 = q == 0 ? 0 : (q == 1 ? sw : (q == 2 ? 2 : 2 + sw));
    const int off2 = q == 2 ? -2 : (q == 3 ? sw - 2 : 0);
    const int img = tid / G, mb = tid - img * G;  // W rows: one thread per (image, row)
    if (tid < NI) {
        double r = sqrt(x * x + yy * yy + zz * zz);
        if (r < 1e-8) {  // coincident atoms contribute nothing (SNAP.py:1487)
            x = 0;
            yy = 0;
            zz = 1.0;
            r = 1.0;
            wn = 0.0;
        }
        double fc, dfc;
        cutoff_fdf(A.cutoff_id, r, A.rcut, fc, dfc);
        CK ck;
        cayley_klein(x, yy, zz, r, A.rfac0 * M_PI * r / A.rcut, true, ck);
        double p[3];
        cd qq[3];
        su2_generators(ck, p, qq);
        sck[tid][0] = ck.ca;
        sck[tid][1] = ck.cb;
        const double wf = wn * fc, wd = wn * dfc / r;
#pragma unroll
        for (int k = 0; k < 3; k++) {
            sc[tid][k] = wf * p[k];
            sc[tid][3 + k] = wf * qq[k].re;
            sc[tid][6 + k] = wf * qq[k].im;
        }
        sc[tid][9] = wd * x;
        sc[tid][10] = wd * yy;
        sc[tid][11] = wd * zz;
    }
    __syncthreads();
    db_d4 acc[TW][NT];
#pragma unroll
    for (int t = 0; t < TW; t++)
#pragma unroll
        for (int n = 0; n < NT; n++) acc[t][n] = db_d4{0.0, 0.0, 0.0, 0.0};
    CK ck;
    ck.ca = img < NI ? sck[img][0] : cmake(1.0, 0.0);
    ck.cb = img < NI ? sck[img][1] : cmake(0.0, 0.0);
    cd w[TWOJ + 1];
#pragma unroll
    for (int m = 0; m <= TWOJ; m++) w[m] = cmake(m == 0 ? 1.0 : 0.0, 0.0);
    // rolled over stages and levels: unrolled, every wavefront would run once
    // through tens of KB of instructions
#pragma unroll 1
    for (int s = 0; s < A.nstage; s++) {
        const int l0 = stg[3 * s + 2], l1 = stg[3 * s + 5];
        if (s > 0) __syncthreads();  // the previous stage's operands have been read
        int uo = 0;  // values of the stage's earlier levels in a W row
#pragma unroll 1
        for (int l = l0; l < l1; l++) {
            if (l > 0) row_step_w<TWOJ>(l, mb, ck, w);
            if (img < NI && 2 * mb <= l) {
                double2 *ur = reinterpret_cast<double2 *>(Ul + img * KS + uo + 2 * mb * (l + 1));
#pragma unroll
                for (int m = 0; m <= TWOJ; m++)
                    if (m <= l) ur[m] = make_double2(w[m].re, w[m].im);
            }
            uo += 4 * ((2 * (l / 2 + 1) * (l + 1) + 3) / 4);
        }
#pragma unroll
        for (int u = 0; u < ZP; u++) {
            if (zp[u] < 0) continue;
            // place in the low half, twice the half weight above
            const double wt = 0.5 * (zp[u] >> 16);
            *reinterpret_cast<double2 *>(Zl + (zp[u] & 0xffff)) = make_double2(wt * zv[u].re, wt * zv[u].im);
        }
#pragma unroll
        for (int u = 0; u < CP; u++)
            if (u * T + tid < 4 * uo) Cl[u * T + tid] = make_double2(cv[u].re, cv[u].im);
        __syncthreads();
        if (s + 1 < A.nstage) fetch(s + 1);
        if (s + 2 < A.nstage) places(s + 2);
        // a (tile, level) at a time, two steps per turn, the operands of the
        // next turn on their way while the matrix cores work on this one
        // (two register sets in turn)
        struct Turn {
            double2 c[2];
            double x[2], y[2], b[2][NT];
        };
        static_for<TW>([&](auto TT) __attribute__((always_inline)) {
            constexpr int t = decltype(TT)::value;
            int ko = 0;
#pragma unroll 1
            for (int l = l0; l < l1; l++) {
                const int kq = (2 * (l / 2 + 1) * (l + 1) + 3) / 4;
                if ((tmask[t] >> l) & 1) {  // uniform
                    const int slot = l * NSLOT + (wv * TW + t) * 4 + bl;
                    const double *z = Zl + s_row[slot] + kp;
                    const double fac = s_fac[slot];
                    const double *ub = Ul + (lane & 15) * KS + kp + 4 * ko;
                    const double2 *cb = Cl + kp * 4 + q + 16 * ko;
                    auto load = [&](Turn &g, int kk) __attribute__((always_inline)) {
#pragma unroll
                        for (int h = 0; h < 2; h++) {
                            g.c[h] = cb[(kk + h) * 16];
                            g.x[h] = z[(kk + h) * 4 + off1];
                            g.y[h] = z[(kk + h) * 4 + off2];
#pragma unroll
                            for (int n = 0; n < NT; n++) g.b[h][n] = ub[n * 16 * KS + (kk + h) * 4];
                        }
                    };
                    auto mul = [&](const Turn &g, int kk) __attribute__((always_inline)) {
#pragma unroll
                        for (int h = 0; h < 2; h++) {
                            if (kk + h >= kq) return;  // uniform
                            const double av = fac * fma(g.c[h].x, g.x[h], g.c[h].y * g.y[h]);
#pragma unroll
                            for (int n = 0; n < NT; n++)
                                if (n < nt)
                                    acc[t][n] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, g.b[h][n], acc[t][n], 0, 0, 0);
                        }
                    };
                    Turn g0, g1;
                    load(g0, 0);
#pragma unroll 1
                    for (int kk = 0; kk < kq; kk += 4) {
                        load(g1, kk + 2);
                        mul(g0, kk);
                        load(g0, kk + 4);
                        mul(g1, kk + 2);
                    }
                }
                ko += kq;
            }
        });
    }
    // lane (image, b): combine the four sums, collect 16 images' rows in
    // LDS and write them out
    double *ob = Ul;
    static_for<NT>([&](auto NN) __attribute__((always_inline)) {
        constexpr int n = decltype(NN)::value;
        if (n >= nt) return;  // uniform
        __syncthreads();
        const double *S = sc[n * 16 + (lane & 15)];
        static_for<TW>([&](auto TT) __attribute__((always_inline)) {
            constexpr int t = decltype(TT)::value;
            const int b = s_b[(wv * TW + t) * 4 + kp];
            if (b < 0) return;
            double *o = ob + (lane & 15) * (3 * NB) + 3 * b;
#pragma unroll
            for (int k = 0; k < 3; k++)
                o[k] = S[k] * acc[t][n][1] + S[3 + k] * acc[t][n][2] + S[6 + k] * acc[t][n][3] + S[9 + k] * acc[t][n][0];
        });
        __syncthreads();
        const int cnt = (ne - 16 * n < 16 ? ne - 16 * n : 16) * 3 * NB;
        double *og = dbdr + (size_t)(e0 + 16 * n) * 3 * NB;
        for (int k = tid; k < cnt; k += T) og[k] = ob[k];
    });
}

// Centre of workgroup b: the 3-bit fields (b / 8) % 8 and b % 8 of the block
// index swapped (the XCD is b % 8), so that the eight centres whose Z
// entries share a 128-byte line run on one XCD.
__device__ __forceinline__ int64_t so4_db_centre(int64_t b) {
    return (b & ~(int64_t)63) | ((b & 7) << 3) | ((b >> 3) & 7);
}

// The first NI images of every centre, one workgroup each.  No loop over
// passes here: the constants of the cutoff and of the Cayley-Klein parameters
// are then held across it, which costs 144 spilled registers at 2J = 8
// (725 against 540 us for 4096 atoms when the two were compared).
template <int TWOJ>
__global__ __launch_bounds__(DbDim<TWOJ>::T) __attribute__((amdgpu_waves_per_eu(2))) void so4_dbdr_centre_kernel(
    DbArgs A, int64_t natoms, double *__restrict__ dbdr) {
    constexpr int NI = DbDim<TWOJ>::NI;
    const int64_t c = so4_db_centre(blockIdx.x);
    if (c >= natoms) return;
    const int64_t s0 = A.img_start[c], n = A.img_start[c + 1] - s0;
    if (n > 0) so4_dbdr_pass<TWOJ>(A, c, s0, (int)(n < NI ? n : NI), dbdr);
}

// The images past NI of the centres that have more (at 2J <= 8, NI = 48, none
// in a solid at the usual cutoffs; at 2J = 10, NI = 32, those of a dense one:
// 1728 atoms of 33 images take 735 us where 28 images take 375, which is still
// below the 1280 of the vector kernel), a persistent grid over the centres, strided so that the
// centres of a list whose every centre has more are shared out evenly.  The
// threads look at a centre each before the workgroup goes through them, and
// one workgroup per CU has the registers to itself: with two, the kernel's
// spills made even a launch that finds nothing to do cost 12 us (1728 atoms,
// 2J = 8; 5 us now), for 318 against 322 us where every centre has 60 to 90
// images (1200 atoms, all of dB/dr; 594 before the matrix cores).
template <int TWOJ>
__global__ __launch_bounds__(DbDim<TWOJ>::T) __attribute__((amdgpu_waves_per_eu(1))) void so4_dbdr_rest_kernel(
    DbArgs A, int64_t natoms, double *__restrict__ dbdr) {
    constexpr int NI = DbDim<TWOJ>::NI;
    constexpr int T = DbDim<TWOJ>::T;
#pragma unroll 1
    for (int64_t c0 = blockIdx.x; c0 < natoms; c0 += (int64_t)T * gridDim.x) {
        const int64_t ct = c0 + (int64_t)threadIdx.x * gridDim.x;
        if (!__syncthreads_or(ct < natoms && A.img_start[ct + 1] - A.img_start[ct] > NI)) continue;
#pragma unroll 1
        for (int k = 0; k < T; k++) {
            const int64_t c = c0 + (int64_t)k * gridDim.x;
            if (c >= natoms) break;
            const int64_t s1 = A.img_start[c + 1];
#pragma unroll 1
            for (int64_t e0 = A.img_start[c] + NI; e0 < s1; e0 += NI) {
                so4_dbdr_pass<TWOJ>(A, c, e0, (int)(s1 - e0 < NI ? s1 - e0 : NI), dbdr);
                __syncthreads();  // the next pass rewrites the LDS
            }
        }
    }
}

// -------------------------------------------------------------- row scatter
// Reference layout rows (SNAP.py:1458-1468).  One wavefront per (centre, 64
// of the 3 nb columns (b, c)), four to a workgroup: a lane goes once through
// the centre's images, eight loads in flight, and keeps the sums of the row
// it is in and those over the whole centre, so dB/dr is read once for all
// outputs; rows are owned by their centre, no atomics.  The images of a
// centre's rows follow each other in memory, so the row ends are only
// positions in that run: they come 64 at a time into a register and are
// picked by lane.  Bound by memory.
//   ROWS_DX    dxdr alone
//   ROWS_FULL  and -bstress/V per row, bstress[nsite] += Ri (x) dB,
//              bstress[row] -= Rj (x) dB
//   ROWS_VOIGT and its sum over the centre's rows, in which the absolute
//              positions cancel: 1/V sum_e r_e (x) dB, Voigt order
// 1728 atoms, 28 images each, 55 components: dxdr and the Voigt sums 30 us
// (130 MB read and written), before 92 us with the per-row rdxdr (a workgroup
// per centre, two passes over its images, one load in flight) and 49 us for
// its sum.  300 atoms, 48 images each, 147 components: dxdr and per-row rdxdr
// 149 -> 49 us (255 MB).
enum { ROWS_DX, ROWS_FULL, ROWS_VOIGT };

template <int MODE>
__global__ __launch_bounds__(256) void so4_rows_kernel(int64_t natoms, int nb, int nslice,
                                                        const int64_t *__restrict__ row_start,
                                                        const int64_t *__restrict__ row_img,
                                                        const int64_t *__restrict__ nsite,
                                                        const double *__restrict__ pos,
                                                        const double *__restrict__ img_r,
                                                        const double *__restrict__ dbdr,
                                                        const double *__restrict__ inv_vol, double *__restrict__ dxdr,
                                                        double *__restrict__ out) {
    constexpr int U = 8;
    const int lane = threadIdx.x & 63;
    const int64_t unit = (int64_t)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int64_t i = unit / nslice;
    if (i >= natoms) return;
    const int nbk = nb * 3, t = (int)(unit - i * nslice) * 64 + lane;
    const bool in = t < nbk;
    const int tc = in ? t : nbk - 1;
    const int b = tc / 3, c = tc - 3 * b;
    const int64_t r0 = row_start[i], r1 = row_start[i + 1], ns = nsite[i];
    const int64_t e0 = row_img[r0], e1 = row_img[r1];
    double iv = 0.0, Ri[3] = {0.0, 0.0, 0.0};
    if (MODE != ROWS_DX) iv = inv_vol[i];
    if (MODE == ROWS_FULL)
        for (int a = 0; a < 3; a++) Ri[a] = pos[3 * i + a];
    double self = 0.0, v = 0.0, site[3] = {0.0, 0.0, 0.0}, w[3] = {0.0, 0.0, 0.0};
    // ends of the rows rb .. rb + 63, relative to e0
    int64_t rw = r0, rb = r0;
    auto ends = [&](int64_t base) {
        const int64_t k = base + lane;
        return k < r1 ? (int)(row_img[k + 1] - e0) : 0x7fffffff;
    };
    int end = ends(rb);
    int next = __builtin_amdgcn_readlane(end, 0);
    const int n = (int)(e1 - e0);
    auto close = [&]() {  // the row rw is complete
        if (MODE == ROWS_FULL) {
            if (rw == ns) {
                for (int a = 0; a < 3; a++) site[a] += w[a];
            } else if (in) {
                for (int a = 0; a < 3; a++) out[(size_t)rw * 3 * nbk + 9 * b + 3 * a + c] = -w[a] * iv;
            }
            for (int a = 0; a < 3; a++) w[a] = 0.0;
        }
        if (rw != ns) {
            if (in) dxdr[(size_t)rw * nbk + tc] = v;
            self -= v;
        }
        v = 0.0;
        rw++;
        if (rw - rb == 64) {
            rb = rw;
            end = ends(rb);
        }
        next = __builtin_amdgcn_readlane(end, (int)(rw - rb));
    };
    const double *src = dbdr + (size_t)e0 * nbk + tc;
    const double *rr = img_r + 3 * e0;
    for (int e = 0; e < n; e += U) {
        double d[U], x[U][3];
#pragma unroll
        for (int k = 0; k < U; k++) {
            const int ek = e + k < n ? e + k : n - 1;
            d[k] = src[(size_t)ek * nbk];
            if (MODE != ROWS_DX)
                for (int a = 0; a < 3; a++) x[k][a] = rr[3 * ek + a];
        }
#pragma unroll
        for (int k = 0; k < U; k++) {
            if (e + k >= n) break;  // uniform, as the row ends
            while (e + k >= next) close();
            v += d[k];
            if (MODE == ROWS_VOIGT)
                for (int a = 0; a < 3; a++) site[a] += x[k][a] * d[k];
            if (MODE == ROWS_FULL)
                for (int a = 0; a < 3; a++) {
                    site[a] += Ri[a] * d[k];
                    w[a] -= (x[k][a] + Ri[a]) * d[k];
                }
        }
    }
    while (rw < r1) close();
    if (!in) return;
    dxdr[(size_t)ns * nbk + tc] = self;
    if (MODE == ROWS_FULL)
        for (int a = 0; a < 3; a++) out[(size_t)ns * 3 * nbk + 9 * b + 3 * a + c] = -site[a] * iv;
    if (MODE == ROWS_VOIGT) {
        // (a, c) of the Voigt order xx yy zz xy xz yz; without a volume the
        // rows are infinite with both signs and have no sum
        const bool fin = fabs(iv) < __builtin_huge_val();
        double *o = out + ((size_t)i * nb + b) * 6;
        for (int a = 0; a < 3; a++)
            if (a <= c) o[a == c ? a : a + c + 2] = fin ? site[a] * iv : __builtin_nan("");
    }
}

// ----------------------------------------------------- force contractions
// Plain path: dE/dR_m = sum over rows (i, m) of sum_b beta[i,b] dxdr[row,b,:]
// (neuralnetwork.py:484-497), gathered over centre m's rows through the
// reverse-row index.  One wavefront per atom.
__global__ __launch_bounds__(64) void dxdr_contract_kernel(int64_t natoms, int nb, const int64_t *__restrict__ row_start,
                                                            const int64_t *__restrict__ seq,
                                                            const int64_t *__restrict__ row_rev,
                                                            const double *__restrict__ beta,
                                                            const double *__restrict__ dxdr, double *__restrict__ grad) {
    const int64_t m = blockIdx.x;
    if (m >= natoms) return;
    const int lane = threadIdx.x;
    double a0 = 0, a1 = 0, a2 = 0;
    for (int64_t rw = row_start[m]; rw < row_start[m + 1]; rw++) {
        const int64_t i = seq[2 * rw + 1];
        const int64_t rr = row_rev[rw];
        const double *d = dxdr + (size_t)rr * nb * 3;
        for (int b = lane; b < nb; b += 64) {
            const double bt = beta[(size_t)i * nb + b];
            a0 += bt * d[3 * b];
            a1 += bt * d[3 * b + 1];
            a2 += bt * d[3 * b + 2];
        }
    }
    for (int off = 32; off > 0; off >>= 1) {
        a0 += __shfl_down(a0, off);
        a1 += __shfl_down(a1, off);
        a2 += __shfl_down(a2, off);
    }
    if (lane == 0) {
        grad[3 * m] = a0;
        grad[3 * m + 1] = a1;
        grad[3 * m + 2] = a2;
    }
}

// Transpose of the plain force contraction: for a gradient g [N, 3] with
// respect to dE/dR, grad_beta[i, b] = sum over rows (i, m) of
// dxdr[row, b, :] . g[m, :] -- the backward of dxdr_contract_kernel (the
// reference's loss differentiates its dxdr contraction this way,
// neuralnetwork.py:484-497).  One wavefront per centre over its own rows
// (no reverse index), lanes over b, four rows in flight.
__global__ __launch_bounds__(64) void dxdr_contract_t_kernel(int64_t natoms, int nb,
                                                              const int64_t *__restrict__ row_start,
                                                              const int64_t *__restrict__ seq,
                                                              const double *__restrict__ g,
                                                              const double *__restrict__ dxdr,
                                                              double *__restrict__ gbeta) {
    const int64_t i = blockIdx.x;
    if (i >= natoms) return;
    const int lane = threadIdx.x;
    const int64_t r0 = row_start[i], r1 = row_start[i + 1];
    for (int b = lane; b < nb; b += 64) {
        double a0 = 0, a1 = 0, a2 = 0, a3 = 0;
        int64_t rw = r0;
        for (; rw + 4 <= r1; rw += 4) {
            const double *d = dxdr + (size_t)rw * nb * 3 + 3 * b;
            const int64_t m0 = seq[2 * rw + 1], m1 = seq[2 * rw + 3], m2 = seq[2 * rw + 5], m3 = seq[2 * rw + 7];
            const size_t st = (size_t)nb * 3;
            a0 += d[0] * g[3 * m0] + d[1] * g[3 * m0 + 1] + d[2] * g[3 * m0 + 2];
            a1 += d[st] * g[3 * m1] + d[st + 1] * g[3 * m1 + 1] + d[st + 2] * g[3 * m1 + 2];
            a2 += d[2 * st] * g[3 * m2] + d[2 * st + 1] * g[3 * m2 + 1] + d[2 * st + 2] * g[3 * m2 + 2];
            a3 += d[3 * st] * g[3 * m3] + d[3 * st + 1] * g[3 * m3 + 1] + d[3 * st + 2] * g[3 * m3 + 2];
        }
        for (; rw < r1; rw++) {
            const double *d = dxdr + (size_t)rw * nb * 3 + 3 * b;
            const int64_t m = seq[2 * rw + 1];
            a0 += d[0] * g[3 * m] + d[1] * g[3 * m + 1] + d[2] * g[3 * m + 2];
        }
        gbeta[(size_t)i * nb + b] = (a0 + a1) + (a2 + a3);
    }
}

// One step of a sum over the wavefront's lanes: a lane and the lane `off`
// away from it each keep one half of the N values and add the other's.  Every sum
// is formed in the order of the xor butterfly, with half the exchanges of the
// step before instead of all N at every step.
template <int N>
__device__ __forceinline__ void wave_halve(double *v, int lane, int off) {
    const bool up = (lane & off) != 0;
#pragma unroll
    for (int k = 0; k < N / 2; k++) {
        const double send = up ? v[k] : v[k + N / 2], keep = up ? v[k + N / 2] : v[k];
        v[k] = keep + __shfl_xor(send, off);
    }
}

// Adjoint path: dE/dR_i = sum_{e of i} (dE/dr_rev(e) - dE/dr_e); virial of
// centre i = sum_e r_e (x) dE/dr_e.  One wavefront per atom (4 per
// workgroup), lanes over the centre's images, then sums over the lanes (fixed
// order: deterministic, no atomics).  With the virial the lane exchanges
// bound it: 135,245 atoms of 31 images 202 -> 87 us, 33,722 atoms 58 -> 25.
//
// NEG: the forces -dE/dR_i, summed as (dedr_e - dedr_rev(e)) -- the exact
// negation of the dE/dR sum, term by term in the same order.  With e_out the
// grid has one more workgroup, the last, which stores the sum of
// e_in[0, n_e) (the total energy) to e_out[0] by block_sum_1col: the same
// value as the one-column segment sum, with no launch of its own.
template <bool NEG>
__global__ __launch_bounds__(256) void so4_gather_kernel(int64_t natoms, const int64_t *__restrict__ img_start,
                                                          const int64_t *__restrict__ img_rev,
                                                          const double *__restrict__ img_r,
                                                          const double *__restrict__ dedr, double *__restrict__ grad,
                                                          double *__restrict__ virial,
                                                          const double *__restrict__ e_in = nullptr,
                                                          int64_t n_e = 0, double *__restrict__ e_out = nullptr) {
    static_assert(PXFF_SUM_THREADS == 256, "the energy workgroup is one gather workgroup");
    if (e_out != nullptr && blockIdx.x == gridDim.x - 1) {
        const double t = block_sum_1col(e_in, 0, n_e);
        if (threadIdx.x == 0) e_out[0] = t;
        return;
    }
    const int lane = threadIdx.x & 63;
    const int64_t i = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (i >= natoms) return;  // whole wavefront
    double g[3] = {0, 0, 0};
    double v[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    for (int64_t e = img_start[i] + lane; e < img_start[i + 1]; e += 64) {
        const int64_t q = img_rev[e];
        const double d[3] = {dedr[3 * e], dedr[3 * e + 1], dedr[3 * e + 2]};
#pragma unroll
        for (int k = 0; k < 3; k++) g[k] += NEG ? d[k] - dedr[3 * q + k] : dedr[3 * q + k] - d[k];
        if (virial) {
#pragma unroll
            for (int a = 0; a < 3; a++) {
                const double ra = img_r[3 * e + a];
#pragma unroll
                for (int c = 0; c < 3; c++) v[3 * a + c] += ra * d[c];
            }
        }
    }
    if (virial) {
        // 12 -> 6 -> 3 (4 with a zero) -> 2 -> 1 values per lane
        double t[12] = {g[0], g[1], g[2], v[0], v[1], v[2], v[3], v[4], v[5], v[6], v[7], v[8]};
        wave_halve<12>(t, lane, 32);
        wave_halve<6>(t, lane, 16);
        t[3] = 0.0;
        wave_halve<4>(t, lane, 8);
        wave_halve<2>(t, lane, 4);
        t[0] += __shfl_xor(t[0], 2);
        t[0] += __shfl_xor(t[0], 1);
        const int at = (lane >> 2) & 3;  // of the three values of a row of 16 lanes
        const int k = ((lane >> 5) & 1) * 6 + ((lane >> 4) & 1) * 3 + ((at >> 1) & 1) * 2 + (at & 1);
        if ((lane & 3) == 0 && at < 3) {
            if (k < 3)
                grad[3 * i + k] = t[0];
            else
                virial[9 * i + k - 3] = t[0];
        }
    } else {
        double t[4] = {g[0], g[1], g[2], 0.0};
        wave_halve<4>(t, lane, 32);
        wave_halve<2>(t, lane, 16);
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) t[0] += __shfl_xor(t[0], off);
        const int k = lane >> 4;
        if ((lane & 15) == 0 && k < 3) grad[3 * i + k] = t[0];
    }
}

// Per-atom rdxdr reduction (utilities/__init__.py:226-235).
__global__ void rdxdr_reduce_kernel(int64_t natoms, int nb, const int64_t *__restrict__ row_start,
                                    const double *__restrict__ rdxdr, double *__restrict__ out) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= natoms * nb) return;
    const int64_t i = t / nb;
    const int b = (int)(t - i * nb);
    double s[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
    for (int64_t rw = row_start[i]; rw < row_start[i + 1]; rw++)
        for (int k = 0; k < 9; k++) s[k] += rdxdr[((size_t)rw * nb + b) * 9 + k];
    const int vo[6] = {0, 4, 8, 1, 2, 5};
    for (int k = 0; k < 6; k++) out[((size_t)i * nb + b) * 6 + k] = s[vo[k]];
}

// Stress of centre i in the network's contraction (neuralnetwork.py:484-497):
// out[i, v] = -sum_b beta[i, b] rv[i, b, v] over the per-atom Voigt rdxdr.
// Bound by reading rv once.  One wavefront per atom, 60 lanes: lane = (ten b,
// component v), so that a lane keeps its component over the whole row and the
// loads are contiguous; then the ten lanes of a component in a fixed order.
// 1728 atoms, 55 components (4.6 MB): a few us, against 10.1 ms of a library
// matrix-vector product over the flattened (atom, b) with six columns.
__global__ __launch_bounds__(256) void voigt_contract_kernel(int64_t natoms, int nb, const double *__restrict__ beta,
                                                              const double *__restrict__ rv,
                                                              double *__restrict__ out) {
    __shared__ double red[4][60];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int64_t i = (int64_t)blockIdx.x * 4 + wv;
    const bool in = i < natoms && lane < 60;
    if (in) {
        const double *be = beta + (size_t)i * nb, *r = rv + (size_t)i * nb * 6 + lane;
        double s0 = 0.0, s1 = 0.0;
        int b = lane / 6;
        for (; b + 10 < nb; b += 20) {
            s0 += be[b] * r[60 * (b / 10)];
            s1 += be[b + 10] * r[60 * (b / 10 + 1)];
        }
        if (b < nb) s0 += be[b] * r[60 * (b / 10)];
        red[wv][lane] = s0 + s1;
    }
    __syncthreads();
    if (in && lane < 6) {
        double s = 0.0;
#pragma unroll
        for (int k = 0; k < 10; k++) s += red[wv][6 * k + lane];
        out[6 * i + lane] = -s;
    }
}

// ----------------------------------------------------------- tangent of B
// dB_b = sum over the (block k, factor f) pairs targeting b of f p_k with
// p_k = 2 Re sum_loc hw(loc) conj(dU^l[loc]) Z_k[loc] and dU = dU_tot (u_norm
// already applied by the accumulation kernel).  A wavefront takes one b of a
// 64-atom tile, one atom per lane: it sums the (at most three) blocks of b,
// which no other b has, so every Z element is read once.  dU and Z are both
// tile-major, every load is a coalesced 1 KB row, four sums per block and
// eight rows of each in flight.  Bound by the Z stream.  The workgroups of a
// tile have the same index modulo 8, so that one XCD's L2 serves the tile's
// dU to all of them and gathers the 8-byte stores of its dB rows; the larger
// b, with the longer blocks, start first.  33,722 atoms (2J = 8, 1.29 GB of Z):
// 306 us, 4.2 TB/s; a workgroup per tile with the blocks' sums in LDS took 356,
// its 534 workgroups being a round of 512 and a rest.
constexpr int TANB_WAVES = 4;
constexpr int TANB_XCDS = 8;
__global__ __launch_bounds__(TANB_WAVES * 64) void so4_tangent_b_kernel(
    int64_t natoms, int nhalf, int nz, int nb, int ldim, const double *__restrict__ dutile,
    const double *__restrict__ z, const double *__restrict__ h_weight, const int *__restrict__ hoff,
    const int *__restrict__ blk_level_start, const int *__restrict__ blk_zoff, const int *__restrict__ b_src,
    const double *__restrict__ b_srcf, double *__restrict__ db) {
    const int tg = (nb + TANB_WAVES - 1) / TANB_WAVES;
    const int64_t q = blockIdx.x / TANB_XCDS;
    const int64_t tile = q / tg * TANB_XCDS + blockIdx.x % TANB_XCDS;
    const int b = nb - 1 - __builtin_amdgcn_readfirstlane((int)(q % tg) * TANB_WAVES + (threadIdx.x >> 6));
    if (tile * 64 >= natoms || b < 0) return;  // whole wavefront
    const int lane = threadIdx.x & 63;
    const cd *dut = reinterpret_cast<const cd *>(dutile) + (size_t)tile * nhalf * 64 + lane;
    const cd *zt = reinterpret_cast<const cd *>(z) + (size_t)tile * nz * 64 + lane;
    double acc = 0.0;
    for (int s = 0; s < 3; s++) {
        const int k = b_src[3 * b + s];
        if (k < 0) continue;
        int l = 0;
        while (l + 1 < ldim && k >= blk_level_start[l + 1]) l++;
        const int nloc = (l / 2 + 1) * (l + 1);
        const cd *u = dut + (size_t)hoff[l] * 64, *v = zt + (size_t)blk_zoff[k] * 64;
        const double *hw = h_weight + hoff[l];
        double p[4] = {0.0, 0.0, 0.0, 0.0};
        int t = 0;
        for (; t + 8 <= nloc; t += 8) {
            cd uu[8], vv[8];
#pragma unroll
            for (int c = 0; c < 8; c++) vv[c] = v[(size_t)(t + c) * 64], uu[c] = u[(size_t)(t + c) * 64];
#pragma unroll
            for (int c = 0; c < 8; c++) p[c & 3] += hw[t + c] * cdotre(uu[c], vv[c]);
        }
        if (t + 4 <= nloc) {
#pragma unroll
            for (int c = 0; c < 4; c++) p[c] += hw[t + c] * cdotre(u[(size_t)(t + c) * 64], v[(size_t)(t + c) * 64]);
            t += 4;
        }
        for (; t < nloc; t++) p[0] += hw[t] * cdotre(u[(size_t)t * 64], v[(size_t)t * 64]);
        acc += b_srcf[3 * b + s] * (2.0 * ((p[0] + p[1]) + (p[2] + p[3])));
    }
    const int64_t i = tile * 64 + lane;
    if (i < natoms) db[(size_t)i * nb + b] = acc;
}

// Atom-major copy of the tile-major Z: za[i][e] = Z[i/64][e][i%64].  A
// workgroup moves 32 rows of one tile through LDS: coalesced 1 KB row loads,
// 512 B contiguous stores per atom.
__global__ __launch_bounds__(256) void so4_z_atom_major_kernel(int64_t natoms, int nz, const double *__restrict__ zt,
                                                                double *__restrict__ za) {
    __shared__ cd buf[32][65];
    const int64_t tile = blockIdx.x;
    const int e0 = blockIdx.y * 32;
    const int lane = threadIdx.x & 63;
    const cd *src = reinterpret_cast<const cd *>(zt) + (size_t)tile * nz * 64;
    for (int r = threadIdx.x >> 6; r < 32; r += 4)
        if (e0 + r < nz) buf[r][lane] = src[(size_t)(e0 + r) * 64 + lane];
    __syncthreads();
    cd *dst = reinterpret_cast<cd *>(za);
    for (int idx = threadIdx.x; idx < 64 * 32; idx += blockDim.x) {
        const int a = idx >> 5, r = idx & 31;
        const int64_t i = tile * 64 + a;
        if (i < natoms && e0 + r < nz) dst[(size_t)i * nz + e0 + r] = buf[r][a];
    }
}

}  // namespace pxff

// =================================================================== C ABI
using namespace pxff;

namespace pxff {
// Process-wide launch parameters set by the autotuner (pxff_tune_set).
// Atomic: a call reads each knob once when it launches, so calls from
// several host threads and streams never race with a concurrent set (a set
// affects the launches that start after it).
static std::atomic<int> g_tune[PXFF_TUNE_COUNT] = {0, 16, 4, 4};
static const int g_tune_lo[PXFF_TUNE_COUNT] = {0, 1, 1, 0};
static const int g_tune_hi[PXFF_TUNE_COUNT] = {256, 256, 4, 4};
int tune_value(int knob) { return g_tune[knob].load(std::memory_order_relaxed); }

int so4_check_params(const pxff_so4_params *p) {
    PXFF_REQUIRE(p != nullptr, "null params");
    if (p->twol < 0 || p->twol > 10 || (p->twol & 1)) {
        set_error("unsupported 2J=" + std::to_string(p->twol) + " (even 2J in 0..10 supported)");
        return PXFF_ENOTIMPL;
    }
    PXFF_REQUIRE(p->rcut > 0, "rcut must be > 0");
    PXFF_REQUIRE(p->cutoff_id >= 1 && p->cutoff_id <= 7, "cutoff id must be 1..7");
    return 0;
}

// queried once; concurrent first calls store the same value
static std::atomic<int> g_num_cus{0};
int num_cus() {
    int n = g_num_cus.load(std::memory_order_relaxed);
    if (n == 0) {
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess) return 256;
        hipDeviceProp_t prop;
        if (hipGetDeviceProperties(&prop, dev) != hipSuccess) return 256;
        n = prop.multiProcessorCount;
        g_num_cus.store(n, std::memory_order_relaxed);
    }
    return n;
}
}  // namespace pxff

extern "C" int pxff_so4_sizes(int twol, int *nu, int *nhalf, int *nz, int *nb) {
    So4HostTables t;
    if (!build_so4_tables(twol, 0, t)) {
        set_error("unsupported 2J=" + std::to_string(twol));
        return PXFF_ENOTIMPL;
    }
    if (nu) *nu = t.nu;
    if (nhalf) *nhalf = t.nhalf;
    if (nz) *nz = t.nz;
    if (nb) *nb = t.nb;
    return 0;
}

extern "C" int pxff_so4_ui(const pxff_so4_params *p, int64_t natoms, const int64_t *d_img_start,
                           const int64_t *d_img_j, const double *d_img_r, const double *d_atom_w,
                           const double *d_site_w, const int64_t *d_work_order, double *d_utot, void *stream) {
    int rc = so4_check_params(p);
    if (rc) return rc;
    if (natoms <= 0) return 0;
    const So4Dev *T = nullptr;
    if ((rc = get_so4_tables(p->twol, p->normalize_u, &T))) return rc;
    hipStream_t s = (hipStream_t)stream;
    const int grid = (int)std::min<int64_t>(natoms, (int64_t)num_cus() * tune_value(PXFF_TUNE_ACCUM_WAVES_PER_CU));
    const double fcut0 = cutoff_f0_host(p->cutoff_id);
#define PXFF_ACCUM_UI(MODE)                                                                              \
    PXFF_DISPATCH_TWOJ(p->twol, (so4_accum_kernel<TJ, false, true, MODE><<<grid, 64, 0, s>>>(               \
                                    natoms, d_img_start, d_img_j, d_img_r, d_atom_w, d_site_w, nullptr,       \
                                    d_work_order, T->rootpq, T->lnorm, p->rcut, p->rfac0, p->cutoff_id, fcut0, \
                                    d_utot)))
    const int mode = tune_value(PXFF_TUNE_ACCUM_LDSADD);
    if (mode == 4 && p->twol <= 8) {
        PXFF_DISPATCH_TWOJ(p->twol, if constexpr (TJ <= 8) {
            so4_utot_kernel<TJ, false><<<grid, 64, 0, s>>>(natoms, d_img_start, d_img_j, d_img_r, d_atom_w, d_site_w,
                                                          nullptr, d_work_order, T->rootpq, T->lnorm, p->rcut,
                                                          p->rfac0, p->cutoff_id, fcut0, d_utot);
        });
    } else {
        switch (mode) {
        case 1: PXFF_ACCUM_UI(1); break;
        case 2: PXFF_ACCUM_UI(2); break;
        case 3: PXFF_ACCUM_UI(3); break;
        default: PXFF_ACCUM_UI(0); break;
        }
    }
#undef PXFF_ACCUM_UI
    PXFF_LAUNCH_CHECK();
    return 0;
}

extern "C" int pxff_so4_ui_staged(const pxff_so4_params *p, int64_t natoms, const int64_t *d_img_start,
                                  const int64_t *d_img_j, const double *d_img_r, const double *d_atom_w,
                                  const double *d_site_w, const int64_t *d_work_order, int64_t cap, double *d_stage,
                                  double *d_utot, void *stream) {
    int rc = so4_check_params(p);
    if (rc) return rc;
    PXFF_REQUIRE(cap >= 0 && (cap == 0 || d_stage != nullptr), "stage workspace missing");
    if (natoms <= 0) return 0;
    // the register-sum kernel is the one with a staged form (2J <= 8);
    // the other summation modes stage in LDS themselves
    if (tune_value(PXFF_TUNE_ACCUM_LDSADD) != 4 || p->twol > 8)
        return pxff_so4_ui(p, natoms, d_img_start, d_img_j, d_img_r, d_atom_w, d_site_w, d_work_order, d_utot,
                           stream);
    const So4Dev *T = nullptr;
    if ((rc = get_so4_tables(p->twol, p->normalize_u, &T))) return rc;
    hipStream_t s = (hipStream_t)stream;
    const double fcut0 = cutoff_f0_host(p->cutoff_id);
    const int sgrid = (int)std::max<int64_t>(1, std::min<int64_t>(div_up(cap, 256), (int64_t)num_cus() * 8));
    so4_stage_kernel<false><<<sgrid, 256, 0, s>>>(natoms, cap, d_img_start, d_img_j, d_img_r, d_atom_w, nullptr,
                                                  p->rcut, p->rfac0, p->cutoff_id, d_stage);
    PXFF_LAUNCH_CHECK();
    PXFF_DISPATCH_TWOJ(p->twol, if constexpr (TJ <= 8) {
        constexpr int NG = 64 / (TJ / 2 + 1);
        // centres per wavefront: as many as leave a wavefront per SIMD; below
        // four the sum over a centre's groups costs what it did (4095 atoms
        // of 32 images, three centres to a wavefront: 39 against 38 us; 1728
        // atoms, one: 31 against 21)
        const int64_t want = natoms / ((int64_t)num_cus() * 4);
        if (want >= 4) {
            const int split = NG / (int)std::min<int64_t>(NG, want);
            const int64_t grid = div_up(natoms, NG / split);
            PXFF_REQUIRE(grid <= 0x7fffffff, "too many atoms for one launch");
            so4_utot_group_kernel<TJ, false><<<(unsigned)grid, 64, 0, s>>>(natoms, split, d_img_start, d_site_w,
                                                                           T->lnorm, fcut0, cap, d_stage, d_utot);
        } else {
            const int grid =
                (int)std::min<int64_t>(natoms, (int64_t)num_cus() * tune_value(PXFF_TUNE_ACCUM_WAVES_PER_CU));
            so4_utot_staged_kernel<TJ><<<grid, 64, 0, s>>>(natoms, d_img_start, d_site_w, d_work_order, T->lnorm,
                                                          fcut0, d_stage, d_utot);
        }
    });
    PXFF_LAUNCH_CHECK();
    return 0;
}

extern "C" int pxff_so4_b(const pxff_so4_params *p, int64_t natoms, const double *d_utot, const double *d_z,
                          double *d_b, void *stream) {
    int rc = so4_check_params(p);
    if (rc) return rc;
    if (natoms <= 0) return 0;
    PXFF_REQUIRE(d_b != nullptr, "null B output");
    const So4Dev *T = nullptr;
    if ((rc = get_so4_tables(p->twol, p->normalize_u, &T))) return rc;
    hipStream_t s = (hipStream_t)stream;
    const dim3 grid((unsigned)div_up(natoms, 64), (unsigned)div_up(T->nb, 16));
    PXFF_DISPATCH_TWOJ(p->twol, (so4_b_kernel<TJ><<<grid, 256, 0, s>>>(natoms, d_utot, d_z, T->nz, T->nb, T->b_zoff,
                                                                       T->b_level, d_b)));
    PXFF_LAUNCH_CHECK();
    return 0;
}

extern "C" int pxff_so4_yi(const pxff_so4_params *p, int64_t natoms, const double *d_z, const double *d_beta,
                           double *d_y, void *stream) {
    int rc = so4_check_params(p);
    if (rc) return rc;
    if (natoms <= 0) return 0;
    const So4Dev *T = nullptr;
    if ((rc = get_so4_tables(p->twol, p->normalize_u, &T))) return rc;
    hipStream_t s = (hipStream_t)stream;
    const size_t lds = sizeof(double) * 64 * (size_t)T->nb;
    const int64_t ntiles = (natoms + 63) / 64;
    const int64_t grid = ntiles * ((T->nytask + 3) / 4);
    PXFF_REQUIRE(grid <= 0x7fffffff, "too many atoms for one launch");
    if (lds > 65536)
        PXFF_HIP_CHECK(hipFuncSetAttribute((const void *)so4_yi_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           (int)lds));
    so4_yi_kernel<<<(unsigned)grid, 256, lds, s>>>(natoms, T->nytask, T->nz, T->nb, T->nhalf, T->ytask, d_z, d_beta,
                                                   T->blk_zoff, T->blk_tb, T->blk_tf, T->hscale, d_y);
    PXFF_LAUNCH_CHECK();
    return 0;
}

static int so4_deidrj_launch(const pxff_so4_params *p, int64_t nimg, const int64_t *d_count,
                             const int64_t *d_img_atom, const int64_t *d_img_j, const double *d_img_r,
                             const double *d_atom_w, const double *d_y, double *d_dedr, void *stream) {
    int rc = so4_check_params(p);
    if (rc) return rc;
    if (nimg <= 0) return 0;
    const So4Dev *T = nullptr;
    if ((rc = get_so4_tables(p->twol, p->normalize_u, &T))) return rc;
    hipStream_t s = (hipStream_t)stream;
    const int ng = 64 / (p->twol / 2 + 1);
    // rounds per wavefront: at most 64 / ng (one staged lane per image), and
    // few enough that the grid has about 16 wavefronts per CU
    const int nr = (int)std::max<int64_t>(1, std::min<int64_t>(64 / ng, nimg / ((int64_t)num_cus() * 16 * ng)));
    const int nb = ng * nr;  // images per wavefront (staged batch)
    const int wpb = tune_value(PXFF_TUNE_IMAGE_WAVES_PER_BLOCK);
    const int grid = div_up(div_up(nimg, nb), wpb);
    const size_t lds = sizeof(double) * (size_t)wpb * (DEIDRJ_NST + 5) * 64;  // per-wavefront stage
    PXFF_DISPATCH_TWOJ(p->twol, (so4_deidrj_kernel<TJ><<<grid, 64 * wpb, lds, s>>>(nimg, d_img_atom, d_img_j, d_img_r, d_atom_w,
                                                                           d_y, T->rootpq, p->rcut, p->rfac0,
                                                                           p->cutoff_id, d_dedr, d_count, nr)));
    PXFF_LAUNCH_CHECK();
    return 0;
}

extern "C" int pxff_so4_deidrj(const pxff_so4_params *p, int64_t nimg, const int64_t *d_img_atom,
                               const int64_t *d_img_j, const double *d_img_r, const double *d_atom_w,
                               const double *d_y, double *d_dedr, void *stream) {
    return so4_deidrj_launch(p, nimg, nullptr, d_img_atom, d_img_j, d_img_r, d_atom_w, d_y, d_dedr, stream);
}

extern "C" int pxff_so4_deidrj_counted(const pxff_so4_params *p, int64_t cap, const int64_t *d_count,
                                       const int64_t *d_img_atom, const int64_t *d_img_j, const double *d_img_r,
                                       const double *d_atom_w, const double *d_y, double *d_dedr, void *stream) {
    PXFF_REQUIRE(d_count != nullptr, "null image count");
    return so4_deidrj_launch(p, cap, d_count, d_img_atom, d_img_j, d_img_r, d_atom_w, d_y, d_dedr, stream);
}

extern "C" int pxff_so4_gather(int64_t natoms, const int64_t *d_img_start, const int64_t *d_img_rev,
                               const double *d_img_r, const double *d_dedr, double *d_grad, double *d_virial,
                               void *stream) {
    if (natoms <= 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    so4_gather_kernel<false><<<div_up(natoms, 4), 256, 0, s>>>(natoms, d_img_start, d_img_rev, d_img_r, d_dedr,
                                                               d_grad, d_virial);
    PXFF_LAUNCH_CHECK();
    return 0;
}

extern "C" int pxff_so4_forces(int64_t natoms, const int64_t *d_img_start, const int64_t *d_img_rev,
                               const double *d_img_r, const double *d_dedr, double *d_forces, double *d_virial,
                               void *stream) {
    if (natoms <= 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    so4_gather_kernel<true><<<div_up(natoms, 4), 256, 0, s>>>(natoms, d_img_start, d_img_rev, d_img_r, d_dedr,
                                                              d_forces, d_virial);
    PXFF_LAUNCH_CHECK();
    return 0;
}

extern "C" int pxff_so4_forces_energy(int64_t natoms, const int64_t *d_img_start, const int64_t *d_img_rev,
                                      const double *d_img_r, const double *d_dedr, double *d_forces, double *d_virial,
                                      const double *d_e_atom, int64_t n_e, double *d_energy, void *stream) {
    PXFF_REQUIRE(d_energy != nullptr, "null energy output");
    PXFF_REQUIRE(n_e >= 0 && (n_e == 0 || d_e_atom != nullptr), "bad atom energies");
    PXFF_REQUIRE(natoms >= 0, "natoms must be >= 0");
    hipStream_t s = (hipStream_t)stream;
    // workgroups 0 .. div_up(natoms, 4) - 1 gather forces; the last one sums the energies
    so4_gather_kernel<true><<<div_up(natoms, 4) + 1, 256, 0, s>>>(natoms, d_img_start, d_img_rev, d_img_r, d_dedr,
                                                                  d_forces, d_virial, d_e_atom, n_e, d_energy);
    PXFF_LAUNCH_CHECK();
    return 0;
}

static int so4_tangent_launch(const pxff_so4_params *p, const So4Dev *T, int64_t natoms, const int64_t *d_img_start,
                              const int64_t *d_img_j, const double *d_img_r, const double *d_atom_w,
                              const double *d_dr, const double *d_z, double *d_dutot, double *d_db, void *stream, int64_t cap = 0,
                              double *d_stage = nullptr) {
    hipStream_t s = (hipStream_t)stream;
    const int grid = (int)std::min<int64_t>(natoms, (int64_t)num_cus() * tune_value(PXFF_TUNE_ACCUM_WAVES_PER_CU));
#define PXFF_ACCUM_TAN(MODE)                                                                      \
    PXFF_DISPATCH_TWOJ(p->twol, (so4_accum_kernel<TJ, true, true, MODE><<<grid, 64, 0, s>>>(         \
                                    natoms, d_img_start, d_img_j, d_img_r, d_atom_w, nullptr, d_dr, nullptr, \
                                    T->rootpq, T->lnorm, p->rcut, p->rfac0, p->cutoff_id, 0.0, d_dutot)))
    // the tangent sums in registers whenever they fit (2J <= 8): 0.53 ms
    // against 0.75 ms for the LDS modes on the 33.7k-atom training batch,
    // whatever mode the forward's tuning chose
    const int mode = p->twol <= 8 ? 4 : tune_value(PXFF_TUNE_ACCUM_LDSADD);
    // centres per wavefront as in pxff_so4_ui_staged
    const int64_t want = natoms / ((int64_t)num_cus() * 4);
    if (p->twol <= 8 && d_stage != nullptr && want >= 4) {
        const int sgrid = (int)std::max<int64_t>(1, std::min<int64_t>(div_up(cap, 256), (int64_t)num_cus() * 8));
        so4_stage_kernel<true><<<sgrid, 256, 0, s>>>(natoms, cap, d_img_start, d_img_j, d_img_r, d_atom_w, d_dr,
                                                     p->rcut, p->rfac0, p->cutoff_id, d_stage);
        PXFF_LAUNCH_CHECK();
        PXFF_DISPATCH_TWOJ(p->twol, if constexpr (TJ <= 8) {
            constexpr int NG = 64 / (TJ / 2 + 1);
            const int split = NG / (int)std::min<int64_t>(NG, want);
            const int64_t ngrid = div_up(natoms, NG / split);
            PXFF_REQUIRE(ngrid <= 0x7fffffff, "too many atoms for one launch");
            so4_utot_group_kernel<TJ, true><<<(unsigned)ngrid, 64, 0, s>>>(natoms, split, d_img_start, nullptr,
                                                                          T->lnorm, 0.0, cap, d_stage, d_dutot);
        });
    } else if (mode == 4 && p->twol <= 8) {
        PXFF_DISPATCH_TWOJ(p->twol, if constexpr (TJ <= 8) {
            so4_utot_kernel<TJ, true><<<grid, 64, 0, s>>>(natoms, d_img_start, d_img_j, d_img_r, d_atom_w, nullptr,
                                                         d_dr, nullptr, T->rootpq, T->lnorm, p->rcut, p->rfac0,
                                                         p->cutoff_id, 0.0, d_dutot);
        });
    } else {
        switch (mode) {
        case 1: PXFF_ACCUM_TAN(1); break;
        case 2: PXFF_ACCUM_TAN(2); break;
        case 3: PXFF_ACCUM_TAN(3); break;
        default: PXFF_ACCUM_TAN(0); break;
        }
    }
#undef PXFF_ACCUM_TAN
    PXFF_LAUNCH_CHECK();
    const int64_t tgrid = div_up(div_up(natoms, 64), TANB_XCDS) * (int64_t)TANB_XCDS * div_up(T->nb, TANB_WAVES);
    PXFF_REQUIRE(tgrid <= 0x7fffffff, "too many atoms for one launch");
    so4_tangent_b_kernel<<<(unsigned)tgrid, TANB_WAVES * 64, 0, s>>>(
        natoms, T->nhalf, T->nz, T->nb, p->twol + 1, d_dutot, d_z, T->h_weight, T->hoff, T->blk_level_start,
        T->blk_zoff, T->b_src, T->b_srcf, d_db);
    PXFF_LAUNCH_CHECK();
    return 0;
}

extern "C" int pxff_so4_tangent(const pxff_so4_params *p, int64_t natoms, const int64_t *d_img_start,
                                const int64_t *d_img_j, const double *d_img_r, const double *d_atom_w,
                                const double *d_dr, const double *d_z, double *d_dutot, double *d_db, void *stream) {
    int rc = so4_check_params(p);
    if (rc) return rc;
    if (natoms <= 0) return 0;
    const So4Dev *T = nullptr;
    if ((rc = get_so4_tables(p->twol, p->normalize_u, &T))) return rc;
    return so4_tangent_launch(p, T, natoms, d_img_start, d_img_j, d_img_r, d_atom_w, d_dr, d_z, d_dutot, d_db, stream);
}

extern "C" int pxff_so4_tangent_staged(const pxff_so4_params *p, int64_t natoms, const int64_t *d_img_start,
                                       const int64_t *d_img_j, const double *d_img_r, const double *d_atom_w,
                                       const double *d_dr, const double *d_z, int64_t cap, double *d_stage,
                                       double *d_dutot, double *d_db, void *stream) {
    int rc = so4_check_params(p);
    if (rc) return rc;
    PXFF_REQUIRE(cap >= 0 && (cap == 0 || d_stage != nullptr), "stage workspace missing");
    if (natoms <= 0) return 0;
    const So4Dev *T = nullptr;
    if ((rc = get_so4_tables(p->twol, p->normalize_u, &T))) return rc;
    return so4_tangent_launch(p, T, natoms, d_img_start, d_img_j, d_img_r, d_atom_w, d_dr, d_z, d_dutot, d_db, stream,
                              cap, d_stage);
}

// ------------------------------------------------- no-allocation tangent
// The dU_tot . dr workspace of pxff_so4_tangent in a file-scope device array
// (one copy per GPU, held until the process ends), for callers that cannot
// allocate device memory (HIP graph capture, tight loops).  Host code must
// not use the array's name as a device address: its address on the current
// device comes from hipGetSymbolAddress, resolved once per device.
constexpr size_t NOALLOC_SCRATCH_BYTES = (size_t)32 << 20;
static __device__ __align__(256) double scratch[NOALLOC_SCRATCH_BYTES / sizeof(double)];
static std::mutex g_scratch_mutex;
static std::map<int, double *> g_scratch_ptr;  // device -> address of scratch there

static int scratch_on_device(double **out) {
    int dev = 0;
    PXFF_HIP_CHECK(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lk(g_scratch_mutex);
    auto it = g_scratch_ptr.find(dev);
    if (it == g_scratch_ptr.end()) {
        double *ptr = nullptr;
        PXFF_HIP_CHECK(hipGetSymbolAddress((void **)&ptr, HIP_SYMBOL(scratch)));
        PXFF_REQUIRE(ptr != nullptr, "no device address for the no-allocation scratch array");
        it = g_scratch_ptr.emplace(dev, ptr).first;
    }
    *out = it->second;
    return 0;
}

extern "C" int pxff_so4_tangent_noalloc(const pxff_so4_params *p, int64_t natoms, const int64_t *d_img_start,
                                        const int64_t *d_img_j, const double *d_img_r, const double *d_atom_w,
                                        const double *d_dr, const double *d_z, double *d_db, void *stream) {
    int rc = so4_check_params(p);
    if (rc) return rc;
    if (natoms <= 0) return 0;
    const So4Dev *T = nullptr;
    if ((rc = find_so4_tables(p->twol, p->normalize_u, &T))) return rc;
    const size_t need = (size_t)((natoms + 63) / 64) * 64 * (size_t)T->nhalf * 2 * sizeof(double);
    if (need > NOALLOC_SCRATCH_BYTES) {
        set_error("pxff_so4_tangent_noalloc: " + std::to_string(natoms) + " atoms at 2J=" + std::to_string(p->twol) +
                  " need " + std::to_string(need) + " bytes of workspace, more than the " +
                  std::to_string(NOALLOC_SCRATCH_BYTES) + " of the static array (use pxff_so4_tangent)");
        return PXFF_EINVAL;
    }
    double *du = nullptr;
    if ((rc = scratch_on_device(&du))) return rc;
    return so4_tangent_launch(p, T, natoms, d_img_start, d_img_j, d_img_r, d_atom_w, d_dr, d_z, du, d_db, stream);
}

extern "C" int pxff_so4_z_atom_major(const pxff_so4_params *p, int64_t natoms, const double *d_z, double *d_za,
                                     void *stream) {
    int rc = so4_check_params(p);
    if (rc) return rc;
    if (natoms <= 0) return 0;
    const So4Dev *T = nullptr;
    if ((rc = get_so4_tables(p->twol, p->normalize_u, &T))) return rc;
    const dim3 grid((unsigned)div_up(natoms, 64), (unsigned)div_up(T->nz, 32));
    so4_z_atom_major_kernel<<<grid, 256, 0, (hipStream_t)stream>>>(natoms, T->nz, d_z, d_za);
    PXFF_LAUNCH_CHECK();
    return 0;
}

extern "C" int pxff_so4_dbdr(const pxff_so4_params *p, int64_t nimg, const int64_t *d_img_atom,
                             const int64_t *d_img_j, const double *d_img_r, const double *d_atom_w, const double *d_z,
                             double *d_dbdr, void *stream) {
    int rc = so4_check_params(p);
    if (rc) return rc;
    if (nimg <= 0) return 0;
    const So4Dev *T = nullptr;
    if ((rc = get_so4_tables(p->twol, p->normalize_u, &T))) return rc;
    hipStream_t s = (hipStream_t)stream;
    const int ng = 64 / (p->twol / 2 + 1);
    const int grid = div_up(nimg, ng);
    PXFF_DISPATCH_TWOJ(p->twol, (so4_dbdr_kernel<TJ><<<grid, 64, 0, s>>>(
                                    nimg, d_img_atom, d_img_j, d_img_r, d_atom_w, d_z, T->nz, T->nb, T->rootpq,
                                    T->lnorm, T->blk_level_start, T->blk_zoff, T->blk_tb, T->blk_tf, p->rcut,
                                    p->rfac0, p->cutoff_id, d_dbdr)));
    PXFF_LAUNCH_CHECK();
    return 0;
}

extern "C" int pxff_so4_dbdr_centres(const pxff_so4_params *p, int64_t natoms, const int64_t *d_img_start,
                                     const int64_t *d_img_j, const double *d_img_r, const double *d_atom_w,
                                     const double *d_z, int z_atom_major, double *d_dbdr, void *stream) {
    int rc = so4_check_params(p);
    if (rc) return rc;
    if (natoms <= 0) return 0;
    const So4Dev *T = nullptr;
    if ((rc = get_so4_tables(p->twol, p->normalize_u, &T))) return rc;
    PXFF_REQUIRE(natoms <= ((int64_t)1 << 31) - 64, "too many atoms for one launch");
    hipStream_t s = (hipStream_t)stream;
    // one workgroup per centre, rounded up to whole 64-centre tiles (the
    // centre map permutes within a tile; centres >= natoms exit)
    const unsigned grid = (unsigned)((natoms + 63) / 64 * 64);
    const DbArgs A{d_img_start, d_img_j,   d_img_r,   d_atom_w,  d_z,        T->nz,       p->cutoff_id,
                   z_atom_major ? 1 : 0, T->db_nstage, T->db_tile, T->db_row, T->db_fac, T->db_coef, T->db_zmap,
                   T->db_stage, p->rcut,   p->rfac0};
    const unsigned rest = (unsigned)std::min<int64_t>(natoms, (int64_t)num_cus());
    PXFF_DISPATCH_TWOJ(p->twol, (so4_dbdr_centre_kernel<TJ><<<grid, DbDim<TJ>::T, 0, s>>>(A, natoms, d_dbdr)));
    PXFF_LAUNCH_CHECK();
    PXFF_DISPATCH_TWOJ(p->twol, (so4_dbdr_rest_kernel<TJ><<<rest, DbDim<TJ>::T, 0, s>>>(A, natoms, d_dbdr)));
    PXFF_LAUNCH_CHECK();
    return 0;
}

static int so4_rows_grid(int64_t natoms, int nb, int &nslice, unsigned &grid) {
    PXFF_REQUIRE(nb > 0, "nb must be > 0");
    nslice = (3 * nb + 63) / 64;
    const int64_t g = (natoms * nslice + 3) / 4;
    PXFF_REQUIRE(g <= 0x7fffffff, "too many rows for one launch");
    grid = (unsigned)g;
    return 0;
}

extern "C" int pxff_so4_rows(int64_t natoms, int nb, const int64_t *d_row_start, const int64_t *d_row_img,
                             const int64_t *d_seq, const int64_t *d_nsite, const double *d_pos, const double *d_img_r,
                             const double *d_dbdr, const double *d_inv_vol, double *d_dxdr, double *d_rdxdr,
                             void *stream) {
    (void)d_seq;
    if (natoms <= 0) return 0;
    int nslice = 0, rc = 0;
    unsigned grid = 0;
    if ((rc = so4_rows_grid(natoms, nb, nslice, grid))) return rc;
    hipStream_t s = (hipStream_t)stream;
    if (d_rdxdr)
        so4_rows_kernel<ROWS_FULL><<<grid, 256, 0, s>>>(natoms, nb, nslice, d_row_start, d_row_img, d_nsite, d_pos,
                                                         d_img_r, d_dbdr, d_inv_vol, d_dxdr, d_rdxdr);
    else
        so4_rows_kernel<ROWS_DX><<<grid, 256, 0, s>>>(natoms, nb, nslice, d_row_start, d_row_img, d_nsite, d_pos,
                                                       d_img_r, d_dbdr, d_inv_vol, d_dxdr, nullptr);
    PXFF_LAUNCH_CHECK();
    return 0;
}

extern "C" int pxff_rows_voigt(int64_t natoms, int nb, const int64_t *d_row_start, const int64_t *d_row_img,
                               const int64_t *d_nsite, const double *d_img_r, const double *d_dbdr,
                               const double *d_inv_vol, double *d_dxdr, double *d_rv, void *stream) {
    if (natoms <= 0) return 0;
    int nslice = 0, rc = 0;
    unsigned grid = 0;
    if ((rc = so4_rows_grid(natoms, nb, nslice, grid))) return rc;
    so4_rows_kernel<ROWS_VOIGT><<<grid, 256, 0, (hipStream_t)stream>>>(
        natoms, nb, nslice, d_row_start, d_row_img, d_nsite, nullptr, d_img_r, d_dbdr, d_inv_vol, d_dxdr, d_rv);
    PXFF_LAUNCH_CHECK();
    return 0;
}

extern "C" int pxff_dxdr_contract_t(int64_t natoms, int nb, const int64_t *d_row_start, const int64_t *d_seq,
                                    const double *d_g, const double *d_dxdr, double *d_gbeta, void *stream) {
    if (natoms <= 0) return 0;
    PXFF_REQUIRE(nb > 0, "nb must be > 0");
    PXFF_REQUIRE(natoms <= 0x7fffffff, "too many atoms for one launch");
    dxdr_contract_t_kernel<<<(unsigned)natoms, 64, 0, (hipStream_t)stream>>>(natoms, nb, d_row_start, d_seq, d_g,
                                                                            d_dxdr, d_gbeta);
    PXFF_LAUNCH_CHECK();
    return 0;
}

extern "C" int pxff_dxdr_contract(int64_t natoms, int nb, const int64_t *d_row_start, const int64_t *d_seq,
                                  const int64_t *d_row_rev, const double *d_beta, const double *d_dxdr, double *d_grad,
                                  void *stream) {
    if (natoms <= 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    dxdr_contract_kernel<<<(int)natoms, 64, 0, s>>>(natoms, nb, d_row_start, d_seq, d_row_rev, d_beta, d_dxdr, d_grad);
    PXFF_LAUNCH_CHECK();
    return 0;
}

extern "C" int pxff_rdxdr_reduce(int64_t natoms, int nb, const int64_t *d_row_start, const double *d_rdxdr,
                                 double *d_out, void *stream) {
    if (natoms <= 0) return 0;
    hipStream_t s = (hipStream_t)stream;
    rdxdr_reduce_kernel<<<div_up(natoms * nb, 256), 256, 0, s>>>(natoms, nb, d_row_start, d_rdxdr, d_out);
    PXFF_LAUNCH_CHECK();
    return 0;
}

extern "C" int pxff_voigt_contract(int64_t natoms, int nb, const double *d_beta, const double *d_rv, double *d_out,
                                   void *stream) {
    if (natoms <= 0) return 0;
    PXFF_REQUIRE(nb > 0, "nb must be > 0");
    PXFF_REQUIRE(natoms <= 0x7fffffff, "too many atoms for one launch");
    hipStream_t s = (hipStream_t)stream;
    voigt_contract_kernel<<<div_up(natoms, 4), 256, 0, s>>>(natoms, nb, d_beta, d_rv, d_out);
    PXFF_LAUNCH_CHECK();
    return 0;
}

extern "C" int pxff_tune_set(int knob, int value) {
    PXFF_REQUIRE(knob >= 0 && knob < PXFF_TUNE_COUNT, "unknown tuning knob");
    PXFF_REQUIRE(value >= g_tune_lo[knob] && value <= g_tune_hi[knob], "tuning value out of range");
    if (knob == PXFF_TUNE_IMAGE_WAVES_PER_BLOCK) PXFF_REQUIRE(value == 1 || value == 2 || value == 4, "waves per block must be 1, 2 or 4");
    g_tune[knob].store(value, std::memory_order_relaxed);
    return 0;
}

extern "C" int pxff_tune_get(int knob) {
    if (knob < 0 || knob >= PXFF_TUNE_COUNT) return -1;
    return tune_value(knob);
}
