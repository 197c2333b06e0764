// Device-side constant tables and shared launch helpers of the SO(4)/SNAP
// kernels (host declarations; definitions in so4_kernels.hip).
#pragma once
#include <utility>

#include "pxff_common.h"

namespace pxff {

// Per-(device, 2J, normalisation) constant tables in device memory, built
// once from So4HostTables and kept until process exit.
struct So4Dev {
    int twol, nu, nhalf, nz, nb, ncg, nblk;
    double *cg;
    int *blk_level_start, *blk_zoff, *blk_tb;
    double *blk_tf;
    int *b_zoff, *b_level;
    int *b_src;       // [nb*3] blocks targeting b (-1 = none)
    double *b_srcf;   // [nb*3] their factors
    int *zh;          // [nz] half-U element paired with each Z element
    double *hscale;   // [nhalf] 2 hw(h) u_norm(l(h)): Y scale per half element
    double *rootpq, *lnorm;
    int *hoff, *h_level, *h_diag;
    double *h_weight;
    int *idxu_block;
    int nzgroups;
    int *zgroups;
    int nbrow;        // B row partials per atom
    int *b_brow0;     // [nb] first B row partial of b
    // matrix-core dB/dr: levels of each tile and component of each slot
    // (tile * 4 + row), LDS row and factor per (level,
    // slot), generator coefficients, Z elements in level order, first Z
    // element, coefficient pair and level of each stage
    int db_nstage;
    int *db_tile, *db_row, *db_zmap, *db_stage;
    double *db_fac, *db_coef;
    int nytask;       // Y tasks: (level, run of half elements) per wavefront
    int *ytask;       // [nytask * YTASK_STRIDE]
};

// A Y task is {l, loc0, count <= YTASK_ROWS, first block, end block, h0}: the
// half elements h0 .. h0 + count - 1 (locations loc0.. of level l) summed
// over the blocks [first, end) of level l.
constexpr int YTASK_ROWS = 4;
constexpr int YTASK_STRIDE = 6;

int get_so4_tables(int twol, int norm, const So4Dev **out);
int so4_check_params(const pxff_so4_params *p);
int num_cus();
int tune_value(int knob);

__host__ __device__ constexpr int nhalf_of(int twoj) {
    int s = 0;
    for (int l = 0; l <= twoj; l++) s += (l / 2 + 1) * (l + 1);
    return s;
}
// Compile-time loop: f(std::integral_constant<int, 0>) ... f(<N-1>).
template <typename F, int... I>
__device__ inline void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ inline void static_for(F &&f) {
    static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// Blocks (l1, l2, l) of level l.
__host__ __device__ constexpr int nblk_level(int twoj, int l) {
    int nbl = 0;
    for (int l1 = 0; l1 <= twoj; l1++)
        for (int l2 = 0; l2 <= l1; l2++)
            if (l >= l1 - l2 && l <= l1 + l2 && ((l1 + l2 - l) & 1) == 0) nbl++;
    return nbl;
}
// Matrix-core dB/dr.  Wavefronts per workgroup: four, so that two workgroups
// share a CU; eight at 2J = 10, where six tiles per wavefront would not fit
// its registers.
__host__ __device__ constexpr int db_waves(int twoj) { return twoj >= 10 ? 8 : 4; }
// Steps of four values (half element, re / im) of a level, and the LDS stride
// of n values: at least 4 of padding, 2 modulo 4 (the 16 rows that an
// operand load walks down fall in distinct banks).
__host__ __device__ constexpr int db_steps(int l) { return (2 * (l / 2 + 1) * (l + 1) + 3) / 4; }
__host__ __device__ constexpr int db_pad(int n) { return (n + 5) / 4 * 4 + 2; }
__host__ __device__ constexpr int db_stride(int twoj) { return db_pad(4 * db_steps(twoj)); }
__host__ __device__ constexpr int db_level_stride(int l) { return db_pad(2 * (l / 2 + 1) * (l + 1)); }
// Stages: runs of levels whose values fit one W row together (a barrier pair
// and the loads of a stage cost as much as the products of a low level);
// the first level of l's stage.
__host__ __device__ constexpr int db_stage_first(int twoj, int l) {
    int first = 0, used = 0;
    for (int k = 0; k <= l; k++) {
        if (used + db_steps(k) > db_steps(twoj)) {
            first = k;
            used = 0;
        }
        used += db_steps(k);
    }
    return first;
}
// LDS place of the first Z row of level l (4 doubles of guard in front), the
// doubles of the largest stage with a zero row behind it, and the most Z
// elements of a stage.
__host__ __device__ constexpr int db_level_zbase(int twoj, int l) {
    int n = 4;
    for (int k = db_stage_first(twoj, l); k < l; k++) n += nblk_level(twoj, k) * db_level_stride(k);
    return n;
}
__host__ __device__ constexpr int db_stage_zlds(int twoj) {
    int best = 0;
    for (int l = 0; l <= twoj; l++) {
        const int n = db_level_zbase(twoj, l) + nblk_level(twoj, l) * db_level_stride(l);
        best = n > best ? n : best;
    }
    return best + db_stride(twoj);
}
__host__ __device__ constexpr int db_stage_zmax(int twoj) {
    int best = 0;
    for (int l = 0; l <= twoj; l++) {
        int n = 0;
        for (int k = db_stage_first(twoj, l); k <= l; k++) n += nblk_level(twoj, k) * (k / 2 + 1) * (k + 1);
        best = n > best ? n : best;
    }
    return best;
}
__host__ __device__ constexpr int nb_of(int twoj) {
    int s = 0;
    for (int l1 = 0; l1 <= twoj; l1++)
        for (int l2 = 0; l2 <= l1; l2++)
            for (int l = l1 - l2; l <= (twoj < l1 + l2 ? twoj : l1 + l2); l += 2)
                if (l >= l1) s++;
    return s;
}
__host__ __device__ constexpr int hoff_of(int l) {
    int s = 0;
    for (int k = 0; k < l; k++) s += (k / 2 + 1) * (k + 1);
    return s;
}

#define PXFF_DISPATCH_TWOJ(twol, ...)                                             \
    switch (twol) {                                                               \
    case 0: { constexpr int TJ = 0; __VA_ARGS__; } break;                         \
    case 2: { constexpr int TJ = 2; __VA_ARGS__; } break;                         \
    case 4: { constexpr int TJ = 4; __VA_ARGS__; } break;                         \
    case 6: { constexpr int TJ = 6; __VA_ARGS__; } break;                         \
    case 8: { constexpr int TJ = 8; __VA_ARGS__; } break;                         \
    case 10: { constexpr int TJ = 10; __VA_ARGS__; } break;                       \
    default: ::pxff::set_error("unsupported 2J"); return PXFF_ENOTIMPL;           \
    }

}  // namespace pxff
