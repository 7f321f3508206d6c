// elem_general.hpp -- interface of the run-time-degree element kernel (elem_general.hip).
#pragma once

#include "common.hpp"

namespace yeti {

constexpr int GEN_MAXN = 64, GEN_MAXP = 4;   // nodes per element, degree per direction

struct GenArgs {
    const double *coords;      // (3, nb_cp)
    const int32_t *ien;        // (nnode, nelem), 1-based
    const double *weight;      // (nnode, nelem)
    const int32_t *nijk;       // (3, nelem), 1-based spans
    const double *tab[3];      // 1D basis tables per knot span: [B | dB][g][i], half length; see basis_table
    const int32_t *elems;      // active elements (patch-local)
    const int64_t *offs;       // COO offset per active element
    int32_t n_active;
    int32_t n[3];              // nodes per direction
    int32_t tab_n, ng;         // functions per table row, Gauss points per direction
    double lam, mu, rho;
    GaussRule g;
    const double *geo = nullptr;   // p = 4: geometry records of the elements (elem_geo_kernel), geo_rec apart
    int64_t geo_rec = 0;
};

// COO values (and rows / columns, when Kr is given) of the active elements: stiffness, or with
// `mass` the consistent mass matrix. At most GEN_MAXN nodes and MAX_NG points per direction, or 125
// nodes and 5 points with geometry records (stiffness).
int launch_elem_general(const GenArgs &ga, bool mass, double *Kd, int32_t *Kr, int32_t *Kc, hipStream_t st);

}  // namespace yeti
