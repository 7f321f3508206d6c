// assembly.hip -- FP64 stiffness / RHS assembly of 3D NURBS solid elements (YETI type U1) on
// MI355X (gfx950), behind the C ABI of include/yeti_amd.h.
//
// Reference path (paths relative to YETI's src/yeti_iga/):
//   sys_linmat_lindef_static         main/build_system_elemStorage.f90:24-315
//   sys_linmat_lindef_static_omp     main/build_system_elemStorage_OMP.f90:26-289
//   UELMAT_byCP / uelmat_byCP_omp    main/UELMAT.f90:22-225 / main/uelmat_solid_omp.f90:1-200
//   shap, dersbasisfuns              main/shap.f90:21-180, main/dersbasisfuns.f90:30-131
//   stiffmatrix_byCP, material_lib   main/stiffmatrix.F90:130-225, main/material_lib.f90:28-98
//   shapPress                        main/shapPress.f:18-265
//
// Here: the handle, its tables and the launches; right-hand sides and their gradients; the p = 3 and
// 4 mass. Element stiffness: elem_p3.hip (p = 3, 4 points per direction) and elem_general.hip (all
// else); shape gradients: shape_grad.hpp. An element's COO slice is in YETI's order (nodj-major,
// then nodi, then the 3x3 block column-major; diagonal blocks: the 6 upper entries, diagonal halved).
#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "common.hpp"
#include "coo_entries.hpp"
#include "elem_general.hpp"
#include "elem_p3.hpp"

namespace yeti {

std::string &last_error() {
    static thread_local std::string s;
    return s;
}

AllocCtx &alloc_ctx() {
    static thread_local AllocCtx c;
    return c;
}

int set_error(int code, const char *fmt, ...) {
    char buf[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    last_error() = buf;
    return code;
}

// ------------------------------------------------------------------------------------------
// Gauss-Legendre rule (same nodes/weights as main/GaussLegendre.f90:27-160, computed by Newton
// iteration on P_n; agrees with the 30-digit table to ~1 ulp).
static void gauss_legendre(int n, double *x, double *w) {
    for (int i = 0; i < n; ++i) {
        double z = -std::cos(M_PI * (i + 0.75) / (n + 0.5));
        for (int it = 0; it < 100; ++it) {
            double p0 = 1.0, p1 = z;
            for (int k = 2; k <= n; ++k) {
                double pk = ((2.0 * k - 1.0) * z * p1 - (k - 1.0) * p0) / k;
                p0 = p1;
                p1 = pk;
            }
            double dp = (n == 1) ? 1.0 : n * (z * p1 - p0) / (z * z - 1.0);
            double dz = p1 / dp;
            z -= dz;
            if (std::fabs(dz) < 1e-17) break;
        }
        double p0 = 1.0, p1 = z;
        for (int k = 2; k <= n; ++k) {
            double pk = ((2.0 * k - 1.0) * z * p1 - (k - 1.0) * p0) / k;
            p0 = p1;
            p1 = pk;
        }
        double dp = (n == 1) ? 1.0 : n * (z * p1 - p0) / (z * z - 1.0);
        x[i] = z;
        w[i] = 2.0 / ((1.0 - z * z) * dp * dp);
    }
    if (n % 2 == 1) x[n / 2] = 0.0;
    for (int i = 0; i < n / 2; ++i) {
        double xs = 0.5 * (x[n - 1 - i] - x[i]);
        double ws = 0.5 * (w[i] + w[n - 1 - i]);
        x[i] = -xs;
        x[n - 1 - i] = xs;
        w[i] = ws;
        w[n - 1 - i] = ws;
    }
}

void gauss_rule_host(int n, double *x, double *w) { gauss_legendre(n, x, w); }


// ------------------------------------------------------------------------------------------
// Device: non-zero B-splines of degree P and first derivatives at u for 0-based span i
// (Cox-de Boor triangle + closed-form derivative; the contract of dersbasisfuns.f90:30-131).
template <int P>
__host__ __device__ inline void bspline_ders(int i, double u, const double *__restrict__ U, double *N,
                                             double *dN) {
    double left[P + 1], right[P + 1], cur[P + 1], low[P + 1];
    cur[0] = 1.0;
    low[0] = 1.0;
#pragma unroll
    for (int j = 1; j <= P; ++j) {
        left[j] = u - U[i + 1 - j];
        right[j] = U[i + j] - u;
        double saved = 0.0;
#pragma unroll
        for (int r = 0; r < j; ++r) {
            double tmp = cur[r] / (right[r + 1] + left[j - r]);
            cur[r] = saved + right[r + 1] * tmp;
            saved = left[j - r] * tmp;
        }
        cur[j] = saved;
        if (j == P - 1) {
#pragma unroll
            for (int r = 0; r < P; ++r) low[r] = cur[r];
        }
    }
#pragma unroll
    for (int r = 0; r <= P; ++r) {
        N[r] = cur[r];
        int k = i - P + r;
        double d = 0.0;
        if (r >= 1) {
            double den = U[k + P] - U[k];
            if (den != 0.0) d += P * low[r - 1] / den;
        }
        if (r <= P - 1) {
            double den = U[k + P + 1] - U[k + 1];
            if (den != 0.0) d -= P * low[r] / den;
        }
        dN[r] = d;
    }
}

#include "elem_geo.hpp"
#include "shape_grad.hpp"

// ------------------------------------------------------------------------------------------
// Right-hand side of loaded elements (UELMAT.f90:121-223): body loads 101/102 at the volume
// Gauss points, surface loads 10..99 at the face Gauss points.
struct LoadTable {
    const int32_t *jdltype;        // [nb_load]
    const double *adlmag;          // [nb_load]
    const int32_t *add_off;        // [nb_load] offset into add_infos
    const double *add_infos;
    const int32_t *elem_loads;     // CSR: loads acting on each loaded element
    const int32_t *elem_loads_ptr; // [n_loaded + 1]
    const double *nodal_dist;      // (nb_n_dist, nb_cp)
    int32_t nb_n_dist;
    int32_t only_type = 0;         // load-gradient runs: 0 = every load, else only this JDLType
};

struct RhsPatch {
    const double *coords;
    const int32_t *ien;
    const double *weight;
    const int32_t *nijk;
    const double *U[3];
    const int32_t *elems;          // loaded elements of the patch (patch-local)
    int32_t n_loaded;
    int32_t slot0;                 // index of this patch's first loaded element in the RHS buffer
    int32_t p[3];
    int32_t ng;
    double rho;
    GaussRule g;
};

template <int MAXN>
__device__ void rhs_basis(const RhsPatch &rp, int e, const double *pt, int nn, const double *sW,
                          const double (*sX)[3], double *R, double (*dR)[3], double AJ[3][3], double *detJ) {
    // R[c] (and, if dR is given, dR[c][m] = dR/d(parent coordinate m)) for the nodes a = lane + 64 c
    // parametric point and 1D bases (loaded elements' degrees, up to 4)
    const int lane = threadIdx.x;
    __shared__ double sb[3][10], sdb[3][10], shalf[3];
    if (lane < 3) {
        int d = lane;
        int span1 = rp.nijk[3 * (int64_t)e + d];
        const double *U = rp.U[d];
        double u0 = U[span1 - 1], u1 = U[span1];
        double u = ((u1 - u0) * pt[d] + (u1 + u0)) * 0.5;
        shalf[d] = 0.5 * (u1 - u0);
        int p = rp.p[d];
        int i = span1 - 1;
        double left[10], right[10], cur[10], low[10];
        cur[0] = 1.0;
        low[0] = 1.0;
        for (int j = 1; j <= p; ++j) {
            left[j] = u - U[i + 1 - j];
            right[j] = U[i + j] - u;
            double saved = 0.0;
            for (int r = 0; r < j; ++r) {
                double tmp = cur[r] / (right[r + 1] + left[j - r]);
                cur[r] = saved + right[r + 1] * tmp;
                saved = left[j - r] * tmp;
            }
            cur[j] = saved;
            if (j == p - 1)
                for (int r = 0; r < p; ++r) low[r] = cur[r];
        }
        for (int r = 0; r <= p; ++r) {
            int k = i - p + r;
            double dd = 0.0;
            if (r >= 1) {
                double den = U[k + p] - U[k];
                if (den != 0.0) dd += p * low[r - 1] / den;
            }
            if (r <= p - 1) {
                double den = U[k + p + 1] - U[k + 1];
                if (den != 0.0) dd -= p * low[r] / den;
            }
            sb[d][p - r] = cur[r];   // reversed local index
            sdb[d][p - r] = dd;
        }
    }
    __syncthreads();
    const int n0 = rp.p[0] + 1, n1 = rp.p[1] + 1;
    double s[16];
    for (int m = 0; m < 16; ++m) s[m] = 0.0;
    double Nl[MAXN / 64 + 1], dNl[MAXN / 64 + 1][3];
    int c = 0;
    for (int a = lane; a < nn; a += 64, ++c) {
        int i = a % n0, j = (a / n0) % n1, k = a / (n0 * n1);
        double w = sW[a];
        double Na = sb[0][i] * sb[1][j] * sb[2][k] * w;
        double d0 = sdb[0][i] * sb[1][j] * sb[2][k] * w;
        double d1 = sb[0][i] * sdb[1][j] * sb[2][k] * w;
        double d2 = sb[0][i] * sb[1][j] * sdb[2][k] * w;
        Nl[c] = Na;
        dNl[c][0] = d0; dNl[c][1] = d1; dNl[c][2] = d2;
        s[0] += Na; s[1] += d0; s[2] += d1; s[3] += d2;
        for (int r = 0; r < 3; ++r) {
            s[4 + r] += sX[a][r] * Na;
            s[7 + 3 * r] += sX[a][r] * d0;
            s[8 + 3 * r] += sX[a][r] * d1;
            s[9 + 3 * r] += sX[a][r] * d2;
        }
    }
    for (int m = 0; m < 16; ++m) {
        double v = s[m];
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        s[m] = v;
    }
    double Wi = 1.0 / s[0];
    double dw[3] = {s[1] * Wi, s[2] * Wi, s[3] * Wi};
    double J[3][3];
    for (int r = 0; r < 3; ++r)
        for (int cc = 0; cc < 3; ++cc) J[r][cc] = (s[7 + 3 * r + cc] - s[4 + r] * dw[cc]) * Wi;
    for (int r = 0; r < 3; ++r)
        for (int cc = 0; cc < 3; ++cc) AJ[r][cc] = J[r][cc] * shalf[cc];
    *detJ = AJ[0][0] * (AJ[1][1] * AJ[2][2] - AJ[1][2] * AJ[2][1])
          - AJ[0][1] * (AJ[1][0] * AJ[2][2] - AJ[1][2] * AJ[2][0])
          + AJ[0][2] * (AJ[1][0] * AJ[2][1] - AJ[1][1] * AJ[2][0]);
    c = 0;
    for (int a = lane; a < nn; a += 64, ++c) {
        R[c] = Nl[c] * Wi;
        if (dR)
            for (int m = 0; m < 3; ++m) dR[c][m] = (dNl[c][m] - Nl[c] * dw[m]) * Wi * shalf[m];
    }
    __syncthreads();
}

static __device__ inline void cross3(const double *a, const double *b, double *c) {
    c[0] = a[1] * b[2] - a[2] * b[1];
    c[1] = a[2] * b[0] - a[0] * b[2];
    c[2] = a[0] * b[1] - a[1] * b[0];
}

constexpr int RHS_MAXN = 125;   // (4 + 1)^3: nodes of a loaded element, whose degrees kernel_available admits
constexpr int PATCH_MAXN = 729; // (8 + 1)^3: nodes of a solid patch, with or without active elements

// Dynamic LDS of elem_rhs_kernel: the element's node coordinates, weights, local indices and CP
// ids (sized by the patch's node count, so that many elements share a CU).
static size_t rhs_smem_bytes(const RhsPatch &rp) {
    const size_t nn = (size_t)(rp.p[0] + 1) * (rp.p[1] + 1) * (rp.p[2] + 1);
    return nn * (4 * sizeof(double) + 2 * sizeof(int32_t));
}

constexpr int RHS_MAXP = 4;     // highest degree per direction
constexpr int RHS_PC = 64;      // quadrature points per chunk
constexpr int RHS_PT = MAX_NG + 2;   // 1D points: the Gauss points, -1 and +1

// bspline_ders for a run-time degree, into node order (reversed local index, shap.f90:94-119)
static __device__ inline void rhs_basis_1d(int p, int i, double u, const double *U, double *B, double *D) {
    auto put = [&](auto N, auto dN, int n) {
        for (int r = 0; r < n; ++r) {
            B[n - 1 - r] = N[r];
            D[n - 1 - r] = dN[r];
        }
    };
    double N[RHS_MAXP + 1], dN[RHS_MAXP + 1];
    switch (p) {
    case 1: bspline_ders<1>(i, u, U, N, dN); put(N, dN, 2); break;
    case 2: bspline_ders<2>(i, u, U, N, dN); put(N, dN, 3); break;
    case 3: bspline_ders<3>(i, u, U, N, dN); put(N, dN, 4); break;
    default: bspline_ders<4>(i, u, U, N, dN); put(N, dN, 5); break;
    }
}

// One 256-thread block per loaded element. The element's points are few (ng^2 per face load,
// ng^3 for its body loads) and each needs 16 sums over the nodes, so the work is latency: the 1D
// bases of every point a load can use (Gauss points, -1, +1) are built once, one thread each;
// then in chunks of RHS_PC points
//   1. `parts` adjacent lanes per point split the nodes' sums (W, dW, x, dx/du, the load field)
//      and add them by shuffles; the first lane turns them into the point's load f_q / W;
//   2. every thread owns a node (groups of threads split the chunk's points) and adds
//      N_a(q) w_a f_q in registers.
// 16x4x4 p=2 (16 elements, 9 points each) 41.8 -> 6.8 us, 64^3 p=3 (4096 elements) 233 -> 46 us, body
// loads on all of 24^3 p=3 3752 -> 230 us, against one wave per element that walked the points one
// after the other with its node sums in scratch memory.
__global__ void __launch_bounds__(256) elem_rhs_kernel(RhsPatch rp, LoadTable lt, double *rhs_buf) {
    const int le = blockIdx.x;
    if (le >= rp.n_loaded) return;
    const int e = rp.elems[le];
    const int t = threadIdx.x;
    const int n0 = rp.p[0] + 1, n1 = rp.p[1] + 1, nn = n0 * n1 * (rp.p[2] + 1);
    const int ng = rp.ng;
    extern __shared__ double rhs_smem[];
    double (*sX)[3] = reinterpret_cast<double (*)[3]>(rhs_smem);
    double *sW = rhs_smem + 3 * nn;
    int32_t *sIen = reinterpret_cast<int32_t *>(rhs_smem + 4 * nn);
    int32_t *sLoc = sIen + nn;      // i | j << 8 | k << 16
    __shared__ double tB[3][RHS_PT][RHS_MAXP + 1], tD[3][RHS_PT][RHS_MAXP + 1], hel[3];
    __shared__ double fq[RHS_PC][3];
    __shared__ int32_t qpt[RHS_PC];  // 1D points of the chunk's points, packed as sLoc
    __shared__ double red[256][3];
    for (int a = t; a < nn; a += 256) {
        const int cp = rp.ien[(int64_t)nn * e + a];
        sIen[a] = cp;
        for (int d = 0; d < 3; ++d) sX[a][d] = rp.coords[3 * (int64_t)(cp - 1) + d];
        sW[a] = rp.weight[(int64_t)nn * e + a];
        sLoc[a] = (a % n0) | ((a / n0) % n1) << 8 | (a / (n0 * n1)) << 16;
    }
    // waves 0..2 take a direction each: the switch on its degree is uniform in a wave
    if ((t >> 6) < 3 && (t & 63) < ng + 2) {
        const int d = t >> 6, g = t & 63;
        const int span1 = rp.nijk[3 * (int64_t)e + d];
        const double *U = rp.U[d];
        const double u0 = U[span1 - 1], u1 = U[span1];
        const double x = g < ng ? rp.g.x[g] : g == ng ? -1.0 : 1.0;
        rhs_basis_1d(rp.p[d], span1 - 1, ((u1 - u0) * x + (u1 + u0)) * 0.5, U, tB[d][g], tD[d][g]);
        if (g == 0) hel[d] = 0.5 * (u1 - u0);
    }
    const int gle = rp.slot0 + le;
    const int l0 = lt.elem_loads_ptr[gle], l1 = lt.elem_loads_ptr[gle + 1];
    bool any_body = false;
    for (int li = l0; li < l1; ++li) {
        const int ty = lt.jdltype[lt.elem_loads[li]];
        any_body |= (ty == 101 || ty == 102);
    }
    // phase 2: thread t owns node an, the points split over the ngrp groups
    const int nnr = nn <= 32 ? 32 : nn <= 64 ? 64 : 128;
    const int ngrp = 256 / nnr, an = t % nnr, grp = t / nnr;
    double acc[3] = {0.0, 0.0, 0.0};
    __syncthreads();
    // pass l0 - 1: the body loads together; then one pass per face load
    for (int li = any_body ? l0 - 1 : l0; li < l1; ++li) {
        const bool body = li < l0;
        int il = -1, ty = 0;
        if (!body) {
            il = lt.elem_loads[li];
            ty = lt.jdltype[il];
            if (!(ty > 9 && ty < 100)) continue;
        }
        const int face = ty / 10, typ = ty % 10;
        const double *dist = !body && typ == 4 ? lt.nodal_dist + ((int)lt.add_infos[lt.add_off[il]] - 1) : nullptr;
        const int npt = body ? ng * ng * ng : ng * ng;
        const int parts = npt <= 16 ? 16 : npt <= 32 ? 8 : 4;
        for (int q0 = 0; q0 < npt; q0 += RHS_PC) {
            const int nq = min(npt - q0, RHS_PC);
            const int qq = t / parts, part = t % parts;
            double s[17];
#pragma unroll
            for (int m = 0; m < 17; ++m) s[m] = 0.0;
            int g0 = 0, g1 = 0, g2 = 0;
            double wq = 0.0;
            if (qq < nq) {
                const int q = q0 + qq;
                if (body) {
                    g0 = q / (ng * ng);
                    g1 = (q / ng) % ng;
                    g2 = q % ng;
                    wq = rp.g.w[g0] * rp.g.w[g1] * rp.g.w[g2];
                } else {
                    // the first face coordinate runs fastest
                    const int fi = q % ng, fj = q / ng;
                    wq = rp.g.w[fi] * rp.g.w[fj];
                    switch (face) {
                    case 1: g0 = ng; g1 = fi; g2 = fj; break;
                    case 2: g0 = ng + 1; g1 = fi; g2 = fj; break;
                    case 3: g0 = fi; g1 = ng; g2 = fj; break;
                    case 4: g0 = fi; g1 = ng + 1; g2 = fj; break;
                    case 5: g0 = fj; g1 = fi; g2 = ng; break;
                    default: g0 = fj; g1 = fi; g2 = ng + 1; break;
                    }
                }
                for (int a = part; a < nn; a += parts) {
                    const int l = sLoc[a], i = l & 255, j = (l >> 8) & 255, k = l >> 16;
                    const double w = sW[a], B0 = tB[0][g0][i], B1 = tB[1][g1][j], B2 = tB[2][g2][k];
                    const double Na = B0 * B1 * B2 * w;
                    const double d0 = tD[0][g0][i] * B1 * B2 * w;
                    const double d1 = B0 * tD[1][g1][j] * B2 * w;
                    const double d2 = B0 * B1 * tD[2][g2][k] * w;
                    s[0] += Na; s[1] += d0; s[2] += d1; s[3] += d2;
#pragma unroll
                    for (int r = 0; r < 3; ++r) {
                        const double x = sX[a][r];
                        s[4 + r] += x * Na;
                        s[7 + 3 * r] += x * d0;
                        s[8 + 3 * r] += x * d1;
                        s[9 + 3 * r] += x * d2;
                    }
                    if (dist) s[16] += dist[(int64_t)lt.nb_n_dist * (sIen[a] - 1)] * Na;
                }
            }
            for (int o = 1; o < parts; o <<= 1)
#pragma unroll
                for (int m = 0; m < 17; ++m) s[m] += __shfl_xor(s[m], o, 64);
            if (part == 0 && qq < nq) {
                const double Wi = 1.0 / s[0];
                double c[3][3];   // c[m] = dx / d(parent coordinate m)
#pragma unroll
                for (int m = 0; m < 3; ++m)
#pragma unroll
                    for (int r = 0; r < 3; ++r)
                        c[m][r] = (s[7 + 3 * r + m] - s[4 + r] * (s[1 + m] * Wi)) * Wi * hel[m];
                double f[3] = {0.0, 0.0, 0.0};
                if (body) {
                    double n[3];
                    cross3(c[1], c[2], n);
                    const double det = c[0][0] * n[0] + c[0][1] * n[1] + c[0][2] * n[2];
                    for (int lj = l0; lj < l1; ++lj) {
                        const int jl = lt.elem_loads[lj], tj = lt.jdltype[jl];
                        if (tj != 101 && tj != 102) continue;
                        const double *A = lt.add_infos + lt.add_off[jl];
                        if (tj == 101) {
                            double vd[3] = {A[3] - A[0], A[4] - A[1], A[5] - A[2]};
                            const double nd = sqrt(vd[0] * vd[0] + vd[1] * vd[1] + vd[2] * vd[2]);
                            for (int d = 0; d < 3; ++d) vd[d] /= nd;
                            const double ag[3] = {s[4] * Wi - A[0], s[5] * Wi - A[1], s[6] * Wi - A[2]};
                            const double sc = ag[0] * vd[0] + ag[1] * vd[1] + ag[2] * vd[2];
                            const double mag = rp.rho * lt.adlmag[jl] * lt.adlmag[jl];
                            for (int d = 0; d < 3; ++d) f[d] += mag * (ag[d] - sc * vd[d]);
                        } else {
                            for (int d = 0; d < 3; ++d) f[d] += lt.adlmag[jl] * A[d];
                        }
                    }
                    for (int d = 0; d < 3; ++d) f[d] *= wq * fabs(det);
                } else {
                    const double fmag = typ == 4 ? s[16] * Wi : lt.adlmag[il];
                    double n[3];
                    if (face <= 2) cross3(c[1], c[2], n);
                    else if (face <= 4) cross3(c[2], c[0], n);
                    else cross3(c[0], c[1], n);
                    if (typ >= 1 && typ <= 3) {
                        const double dS = sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]);
                        for (int d = 0; d < 3; ++d) f[d] = typ == d + 1 ? wq * dS * fmag : 0.0;
                    } else if (typ == 0 || typ == 4) {
                        // normal load: the cross product of the face tangents, pointing inwards;
                        // codes above face 6 are face 6, as for the points above
                        const double sg = (face == 1 || face == 3 || face == 5) ? wq * fmag : -wq * fmag;
                        for (int d = 0; d < 3; ++d) f[d] = sg * n[d];
                    }
                }
                for (int d = 0; d < 3; ++d) fq[qq][d] = f[d] * Wi;
                qpt[qq] = g0 | g1 << 8 | g2 << 16;
            }
            __syncthreads();
            if (an < nn) {
                const int l = sLoc[an], i = l & 255, j = (l >> 8) & 255, k = l >> 16;
                for (int q = grp; q < nq; q += ngrp) {
                    const int g = qpt[q];
                    const double N = tB[0][g & 255][i] * tB[1][(g >> 8) & 255][j] * tB[2][g >> 16][k];
#pragma unroll
                    for (int d = 0; d < 3; ++d) acc[d] += N * fq[q][d];
                }
            }
            __syncthreads();
        }
    }
    for (int d = 0; d < 3; ++d) red[t][d] = acc[d];
    __syncthreads();
    double *out = rhs_buf + (int64_t)gle * 3 * RHS_MAXN;
    for (int x = t; x < 3 * nn; x += 256) {
        const int a = x / 3, d = x % 3;
        double v = 0.0;
        for (int g = 0; g < ngrp; ++g) v += red[a + g * nnr][d];
        out[x] = v * sW[a];
    }
}

// Shape derivative of the surface-load work, per loaded element and node: g_cj = 2 u^T dF/dX_cj
// for the face loads of elem_rhs_kernel (same faces, quadrature and load types). With the face
// tangents c_m = dx/dxi_m (columns of AJ), dc_m/dX_cj = e_j dR_c/dxi_m, so
//   fixed direction v (types 1-3), F_a = R_a v w dS f, dS = |cA x cB|:
//     d dS/dX_cj = dR_c/dxi_A (cB x n)_j + dR_c/dxi_B (n x cA)_j,  n = (cA x cB)/dS
//   normal load (types 0 and 4), F_a = R_a (A x B) w f:
//     u . d(A x B)/dX_cj = dR_c/dxi_A (B x u)_j + dR_c/dxi_B (u x A)_j
// with u = u(xi_q) = sum_a R_a u_a. Body loads (101 centrifugal, 102 constant) at the volume
// Gauss points as elem_rhs_kernel, derivative below.
__global__ void __launch_bounds__(64) elem_load_grad_kernel(RhsPatch rp, LoadTable lt, const double *__restrict__ u,
                                                            double *grad_buf) {
    const int le = blockIdx.x;
    if (le >= rp.n_loaded) return;
    const int e = rp.elems[le];
    const int lane = threadIdx.x;
    const int nn = (rp.p[0] + 1) * (rp.p[1] + 1) * (rp.p[2] + 1);
    __shared__ double sX[RHS_MAXN][3];
    __shared__ double sW[RHS_MAXN];
    __shared__ double sU[RHS_MAXN][3];
    __shared__ int32_t sIen[RHS_MAXN];
    for (int a = lane; a < nn; a += 64) {
        int cp = rp.ien[(int64_t)nn * e + a];
        sIen[a] = cp;
        for (int d = 0; d < 3; ++d) {
            sX[a][d] = rp.coords[3 * (int64_t)(cp - 1) + d];
            sU[a][d] = u[3 * (int64_t)(cp - 1) + d];
        }
        sW[a] = rp.weight[(int64_t)nn * e + a];
    }
    __syncthreads();
    constexpr int NPL = (RHS_MAXN + 63) / 64;
    double g[NPL][3];
    for (int c = 0; c < NPL; ++c) g[c][0] = g[c][1] = g[c][2] = 0.0;
    double R[NPL], dR[NPL][3];
    const int ng = rp.ng;
    const int gle = rp.slot0 + le;
    const int l0 = lt.elem_loads_ptr[gle], l1 = lt.elem_loads_ptr[gle + 1];
    bool any_body = false;
    for (int li = l0; li < l1; ++li) {
        int t = lt.jdltype[lt.elem_loads[li]];
        any_body |= (t == 101 || t == 102);
    }
    // body loads, u . F = sum_q w |J| u(x_q) . f(x_q):
    //   d/dX_cj = w |J| [ (u . f) dR_c/dx_j + R_c (u . df/dx)_j ],
    // d|J|/dX_cj = |J| dR_c/dx_j; f = rho omega^2 (I - d d^T)(x - A) for 101 (so
    // u . df/dx = rho omega^2 (I - d d^T) u), a constant vector for 102.
    if (any_body) {
        for (int gi = 0; gi < ng; ++gi)
            for (int gj = 0; gj < ng; ++gj)
                for (int gk = 0; gk < ng; ++gk) {
                    double pt[3] = {rp.g.x[gi], rp.g.x[gj], rp.g.x[gk]};
                    double AJ[3][3], detJ;
                    rhs_basis<RHS_MAXN>(rp, e, pt, nn, sW, sX, R, dR, AJ, &detJ);
                    const double dvol = rp.g.w[gi] * rp.g.w[gj] * rp.g.w[gk] * fabs(detJ);
                    // rows of the inverse Jacobian: dxi_m/dx = (col_{m+1} x col_{m+2}) / detJ
                    double col[3][3], cof[3][3];
                    for (int m = 0; m < 3; ++m)
                        for (int d = 0; d < 3; ++d) col[m][d] = AJ[d][m];
                    for (int m = 0; m < 3; ++m) cross3(col[(m + 1) % 3], col[(m + 2) % 3], cof[m]);
                    double uq[3] = {0.0, 0.0, 0.0}, xq[3] = {0.0, 0.0, 0.0};
                    int c = 0;
                    for (int a = lane; a < nn; a += 64, ++c)
                        for (int d = 0; d < 3; ++d) {
                            uq[d] += R[c] * sU[a][d];
                            xq[d] += R[c] * sX[a][d];
                        }
                    for (int o = 32; o > 0; o >>= 1)
                        for (int d = 0; d < 3; ++d) {
                            uq[d] += __shfl_xor(uq[d], o, 64);
                            xq[d] += __shfl_xor(xq[d], o, 64);
                        }
                    double uf = 0.0, hv[3] = {0.0, 0.0, 0.0};
                    for (int li = l0; li < l1; ++li) {
                        const int il = lt.elem_loads[li];
                        const int t = lt.jdltype[il];
                        if (lt.only_type && t != lt.only_type) continue;
                        const double *A = lt.add_infos + lt.add_off[il];
                        if (t == 101) {
                            double vd[3] = {A[3] - A[0], A[4] - A[1], A[5] - A[2]};
                            const double nd = sqrt(vd[0] * vd[0] + vd[1] * vd[1] + vd[2] * vd[2]);
                            for (int d = 0; d < 3; ++d) vd[d] /= nd;
                            const double ag[3] = {xq[0] - A[0], xq[1] - A[1], xq[2] - A[2]};
                            const double sc = ag[0] * vd[0] + ag[1] * vd[1] + ag[2] * vd[2];
                            const double ud = uq[0] * vd[0] + uq[1] * vd[1] + uq[2] * vd[2];
                            const double mag = rp.rho * lt.adlmag[il] * lt.adlmag[il];
                            for (int d = 0; d < 3; ++d) {
                                uf += mag * (ag[d] - sc * vd[d]) * uq[d];
                                hv[d] += mag * (uq[d] - ud * vd[d]);
                            }
                        } else if (t == 102) {
                            uf += lt.adlmag[il] * (A[0] * uq[0] + A[1] * uq[1] + A[2] * uq[2]);
                        }
                    }
                    const double wq = 2.0 * dvol;
                    c = 0;
                    for (int a = lane; a < nn; a += 64, ++c)
                        for (int d = 0; d < 3; ++d) {
                            const double dRdx =
                                (dR[c][0] * cof[0][d] + dR[c][1] * cof[1][d] + dR[c][2] * cof[2][d]) / detJ;
                            g[c][d] += wq * (uf * dRdx + R[c] * hv[d]);
                        }
                }
    }
    for (int li = l0; li < l1; ++li) {
        int il = lt.elem_loads[li];
        int t = lt.jdltype[il];
        if (!(t > 9 && t < 100) || (lt.only_type && t != lt.only_type)) continue;
        int face = t / 10, typ = t % 10;
        int field = typ == 4 ? (int)lt.add_infos[lt.add_off[il]] : 0;
        // columns spanning the face, in the order of elem_rhs_kernel's normal
        const int nA = face <= 2 ? 1 : face <= 4 ? 2 : 0, nB = face <= 2 ? 2 : face <= 4 ? 0 : 1;
        // (A, B) of the normal load per face
        int mA, mB;
        switch (face) {
        case 1: mA = 1; mB = 2; break;
        case 2: mA = 2; mB = 1; break;
        case 3: mA = 2; mB = 0; break;
        case 4: mA = 0; mB = 2; break;
        case 5: mA = 0; mB = 1; break;
        default: mA = 1; mB = 0; break;
        }
        for (int fj = 0; fj < ng; ++fj)
            for (int fi = 0; fi < ng; ++fi) {
                double xi_i = rp.g.x[fi], xi_j = rp.g.x[fj];
                double pt[3];
                switch (face) {
                case 1: pt[0] = -1.0; pt[1] = xi_i; pt[2] = xi_j; break;
                case 2: pt[0] = 1.0; pt[1] = xi_i; pt[2] = xi_j; break;
                case 3: pt[0] = xi_i; pt[1] = -1.0; pt[2] = xi_j; break;
                case 4: pt[0] = xi_i; pt[1] = 1.0; pt[2] = xi_j; break;
                case 5: pt[0] = xi_j; pt[1] = xi_i; pt[2] = -1.0; break;
                default: pt[0] = xi_j; pt[1] = xi_i; pt[2] = 1.0; break;
                }
                double AJ[3][3], detJ;
                rhs_basis<RHS_MAXN>(rp, e, pt, nn, sW, sX, R, dR, AJ, &detJ);
                double col[3][3];
                for (int m = 0; m < 3; ++m)
                    for (int d = 0; d < 3; ++d) col[m][d] = AJ[d][m];
                double nrm[3];
                cross3(col[nA], col[nB], nrm);
                const double dS = sqrt(nrm[0] * nrm[0] + nrm[1] * nrm[1] + nrm[2] * nrm[2]);
                // u and the load field at the face point
                double uq[3] = {0.0, 0.0, 0.0}, fm = 0.0;
                int c = 0;
                for (int a = lane; a < nn; a += 64, ++c) {
                    for (int d = 0; d < 3; ++d) uq[d] += R[c] * sU[a][d];
                    if (typ == 4) fm += lt.nodal_dist[(int64_t)lt.nb_n_dist * (sIen[a] - 1) + (field - 1)] * R[c];
                }
                for (int o = 32; o > 0; o >>= 1) {
                    for (int d = 0; d < 3; ++d) uq[d] += __shfl_xor(uq[d], o, 64);
                    fm += __shfl_xor(fm, o, 64);
                }
                const double fmag = typ == 4 ? fm : lt.adlmag[il];
                const double wq = 2.0 * rp.g.w[fi] * rp.g.w[fj] * fmag;
                double tA[3], tB[3];   // g_c = wq (dR_c/dxi_A tA + dR_c/dxi_B tB)
                int cA, cB;
                if (typ >= 1 && typ <= 3) {
                    const double un = uq[typ - 1];   // u . v
                    double n[3] = {nrm[0] / dS, nrm[1] / dS, nrm[2] / dS};
                    cross3(col[nB], n, tA);
                    cross3(n, col[nA], tB);
                    for (int d = 0; d < 3; ++d) {
                        tA[d] *= un;
                        tB[d] *= un;
                    }
                    cA = nA;
                    cB = nB;
                } else {
                    cross3(col[mB], uq, tA);
                    cross3(uq, col[mA], tB);
                    cA = mA;
                    cB = mB;
                }
                c = 0;
                for (int a = lane; a < nn; a += 64, ++c)
                    for (int d = 0; d < 3; ++d) g[c][d] += wq * (dR[c][cA] * tA[d] + dR[c][cB] * tB[d]);
            }
    }
    int c = 0;
    for (int a = lane; a < nn; a += 64, ++c)
        for (int d = 0; d < 3; ++d) grad_buf[(int64_t)gle * 3 * RHS_MAXN + 3 * a + d] = g[c][d];
}

// F = F_conc + sum over loaded elements (in element order) of their RHS (build_system_elemStorage.f90:295-303);
// F_conc may be null (then F starts from zero).
__global__ void rhs_gather_kernel(int32_t nb_cp, const double *__restrict__ F_conc,
                                  const int32_t *__restrict__ cp_ptr,
                                  const int32_t *__restrict__ cp_ent,
                                  const double *__restrict__ rhs_buf, double *__restrict__ F) {
    int cp = blockIdx.x * blockDim.x + threadIdx.x;
    if (cp >= nb_cp) return;
    double f0 = 0.0, f1 = 0.0, f2 = 0.0;
    if (F_conc) {
        f0 = F_conc[3 * (int64_t)cp];
        f1 = F_conc[3 * (int64_t)cp + 1];
        f2 = F_conc[3 * (int64_t)cp + 2];
    }
    // ent = slot * RHS_MAXN + local node; GU entries in flight at once, added in order (one at a
    // time each entry waits for two memory round trips: 16.4 -> 7.9 us at 23x18x13 p=4)
    constexpr int GU = 8;
    const int k1 = cp_ptr[cp + 1];
    for (int k = cp_ptr[cp]; k < k1; k += GU) {
        double r[GU][3];
#pragma unroll
        for (int u = 0; u < GU; ++u) {
            const double *p = rhs_buf + 3 * (int64_t)cp_ent[min(k + u, k1 - 1)];
            r[u][0] = p[0];
            r[u][1] = p[1];
            r[u][2] = p[2];
        }
#pragma unroll
        for (int u = 0; u < GU; ++u)
            if (k + u < k1) {
                f0 += r[u][0];
                f1 += r[u][1];
                f2 += r[u][2];
            }
    }
    F[3 * (int64_t)cp] = f0;
    F[3 * (int64_t)cp + 1] = f1;
    F[3 * (int64_t)cp + 2] = f2;
}

// Zero a range of a COO buffer (slots of inactive elements in the SLOTTED layout).
__global__ void fill_zero_kernel(double *Kd, int32_t *Kr, int32_t *Kc, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (; i < n; i += stride) {
        Kd[i] = 0.0;
        if (Kr) Kr[i] = 0;
        if (Kc) Kc[i] = 0;
    }
}

// ------------------------------------------------------------------------------------------
// Host side
struct PatchDev {
    int p[3];
    int ng;
    int nnode;
    int nelem;
    double lam, mu, rho;
    bool u1;
    // knot vectors, and 1D basis tables per knot span, padded to tab_n = max degree + 1 functions
    // (basis_table; tab_n = 0: no active element), in one buffer
    DevBuf<double> knots;
    const double *U[3] = {nullptr, nullptr, nullptr}, *tab[3] = {nullptr, nullptr, nullptr};
    int tab_n = 0;
    DevBuf<int32_t> ien, nijk, elems;
    DevBuf<double> weight;
    DevBuf<int64_t> offs;
    int32_t n_active = 0;
    DevBuf<int32_t> loaded;
    int32_t n_loaded = 0;
    int32_t slot0 = 0;
    DevBuf<double> geo;     // per-Gauss-point geometry of one element batch (allocated on first run)
};

}  // namespace yeti

struct yeti_asm {
    // host copies of the per-patch device pointers (for the CSR builder)
    std::vector<const int32_t *> v_ien, v_elems;
    std::vector<const int64_t *> v_offs;
    std::vector<int32_t> v_nnode, v_nactive;
    int layout;
    int64_t nb_data;        // entries the layout uses
    int64_t nb_data_cap;    // nb_data requested by the caller
    int32_t nb_cp, nb_dof_tot;
    std::vector<yeti::PatchDev *> patches;
    yeti::DevBuf<double> coords;
    // zero ranges (slotted layout, inactive elements)
    std::vector<std::pair<int64_t, int64_t>> zero_ranges;
    // loads
    yeti::DevBuf<double> F_conc;
    yeti::DevBuf<int32_t> jdl, add_off, elem_loads, elem_loads_ptr, cp_ptr, cp_ent;
    yeti::DevBuf<double> adlmag, add_infos, nodal_dist, rhs_buf, grad_buf;
    int32_t nb_n_dist = 1;
    // optional per-launch timing of the element kernel (HIP events on the launch stream)
    bool timing = false;
    std::vector<hipEvent_t> ev;
    int32_t ev_used = 0;
    int32_t n_loaded_total = 0;
    // shape gradients (built on first use): CP -> element-node entries of the active U1 elements
    // in CSR form, the per-entry partials, the masses per workgroup and per pair
    yeti::DevBuf<int32_t> vib_ptr;
    yeti::DevBuf<int32_t> vib_ent;
    yeti::DevBuf<double> vib_eg, vib_em, vib_mass;
    // gradLinElastWork_AN: offsets of the centrifugal loads' axis points in load_additionalInfos
    // as the reference reads them (the k-th load of type 101 at 6k), and the work buffers
    yeti::DevBuf<int32_t> add_off_ref;
    bool ref_infos_ok = true;
    bool any_centrifugal = false;   // a load of type 101
    yeti::DevBuf<double> gw_vec, gw_vec2;
    int64_t vib_nent = -1, vib_nslot = 0;
    ~yeti_asm() {
        for (auto *p : patches) delete p;
        for (auto e : ev) (void)hipEventDestroy(e);
    }
};

namespace yeti {

static int parse_elt_types(const yeti_system_inputs *in, std::vector<std::string> &out) {
    out.clear();
    std::string s(in->ELT_TYPE, in->ELT_TYPE + in->len_ELT_TYPE);
    size_t k = 0;
    while (k < s.size()) {
        if (s[k] == 'U') {
            size_t j = k + 1;
            while (j < s.size() && s[j] != 'U' && s[j] != ' ' && s[j] != '\0') ++j;
            out.push_back(s.substr(k, j - k));
            k = j;
        } else {
            ++k;
        }
    }
    if ((int)out.size() < in->nb_patch)
        return set_error(YETI_ERR_INVALID_ARGUMENT, "ELT_TYPE lists %d types for %d patches",
                         (int)out.size(), in->nb_patch);
    return 0;
}

static int gauss_per_dir(int nbint) {
    int n = (int)std::pow((double)nbint, 1.0 / 3.0);
    if (n * n * n < nbint) n += 1;
    return n;
}

// elem_p3_kernel and elem_general_kernel<8, 0> (p = 4) take p + 1 Gauss points per direction
static bool fixed_kernel_available(int p0, int p1, int p2, int ng) {
    return p0 == p1 && p1 == p2 && (p0 == 3 || p0 == 4) && ng == p0 + 1;
}

// every other case goes to elem_general.hip: up to 64 nodes, degrees up to 4, up to 9 points. (p = 1
// and 2 as well: one wave per 16-node tile pair and several workgroups per CU against one persistent
// workgroup, 64^3 p = 1 1.39 -> 1.19 ms, p = 2 6.23 -> 5.07 ms with indices; at 32^3 p = 3 it takes 5.23
// ms, elem_p3_kernel 1.95.)
static bool kernel_available(int p0, int p1, int p2, int ng) {
    if (fixed_kernel_available(p0, p1, p2, ng)) return true;
    return p0 >= 1 && p1 >= 1 && p2 >= 1 && p0 <= 4 && p1 <= 4 && p2 <= 4 && (p0 + 1) * (p1 + 1) * (p2 + 1) <= 64 &&
           ng >= 1 && ng <= MAX_NG;
}

// 1D basis table of one direction: for each knot span with elements the degree + 1 functions,
// padded with zeros to N, and their derivatives at ng Gauss points, [B | dB][g][i] in reversed local
// index (shap.f90:94-119), and half the span's length; 2 ng N + 2 values per span.
template <int P>
static void basis_table_p(const double *U, int nkv, int N, int ng, const double *gx, std::vector<double> &tab) {
    const int rec = 2 * ng * N + 2;
    double B[P + 1], dB[P + 1];
    tab.assign((size_t)rec * std::max(nkv - 1, 1), 0.0);
    for (int i = P; i + P + 1 < nkv; ++i) {
        const double u0 = U[i], u1 = U[i + 1];
        if (!(u1 > u0)) continue;
        double *t = tab.data() + (size_t)rec * i;
        for (int g = 0; g < ng; ++g) {
            bspline_ders<P>(i, ((u1 - u0) * gx[g] + (u1 + u0)) * 0.5, U, B, dB);
            for (int r = 0; r <= P; ++r) {
                t[g * N + P - r] = B[r];
                t[(ng + g) * N + P - r] = dB[r];
            }
        }
        t[2 * ng * N] = 0.5 * (u1 - u0);
    }
}

static void basis_table(int p, const double *U, int nkv, int N, int ng, const double *gx, std::vector<double> &tab) {
    switch (p) {
    case 1: basis_table_p<1>(U, nkv, N, ng, gx, tab); break;
    case 2: basis_table_p<2>(U, nkv, N, ng, gx, tab); break;
    case 3: basis_table_p<3>(U, nkv, N, ng, gx, tab); break;
    default: basis_table_p<4>(U, nkv, N, ng, gx, tab); break;
    }
}

static int device_cu_count() {
    static thread_local int cached_dev = -1, cached_n = 0;
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    if (dev != cached_dev) {
        int n = 0;
        if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) n = 256;
        cached_dev = dev;
        cached_n = n;
    }
    return cached_n;
}

// Elements per launch pair (geometry pass + element kernel): bounds the geometry buffer
// (12 doubles per Gauss point: 400 MB at p = 3) while keeping every CU busy.
constexpr int32_t ELEM_BATCH = 65536;

// event pair k of the handle's timing record (created on first use)
static int timing_events(yeti_asm *h, int k, hipEvent_t *a, hipEvent_t *b) {
    while ((int)h->ev.size() < 2 * (k + 1)) {
        hipEvent_t e;
        YETI_HIP(hipEventCreate(&e));
        h->ev.push_back(e);
    }
    *a = h->ev[2 * k];
    *b = h->ev[2 * k + 1];
    return 0;
}

static GenArgs general_args(yeti_asm *h, PatchDev &pd) {
    GenArgs ga{};
    ga.coords = h->coords.p;
    ga.ien = pd.ien.p;
    ga.weight = pd.weight.p;
    ga.nijk = pd.nijk.p;
    for (int d = 0; d < 3; ++d) {
        ga.tab[d] = pd.tab[d];
        ga.n[d] = pd.p[d] + 1;
    }
    ga.elems = pd.elems.p;
    ga.offs = pd.offs.p;
    ga.n_active = pd.n_active;
    ga.tab_n = pd.tab_n;
    ga.ng = pd.ng;
    ga.lam = pd.lam;
    ga.mu = pd.mu;
    ga.rho = pd.rho;
    gauss_legendre(pd.ng, ga.g.x, ga.g.w);
    return ga;
}

template <int P, int NG>
static int launch_elem(yeti_asm *h, PatchDev &pd, const double *coords, double *Kd, int32_t *Kr, int32_t *Kc,
                       hipStream_t st) {
    using C = ElemCfg<P, NG>;
    if (pd.n_active == 0) return 0;
    const int32_t batch = std::min(pd.n_active, ELEM_BATCH);
    const size_t geo_n = (size_t)batch * C::REC;
    if (pd.geo.n < geo_n) YETI_HIP(pd.geo.alloc(geo_n));
    PatchArgs pa;
    pa.coords = coords;
    pa.ien = pd.ien.p;
    pa.weight = pd.weight.p;
    pa.nijk = pd.nijk.p;
    pa.U0 = pd.U[0];
    pa.U1 = pd.U[1];
    pa.U2 = pd.U[2];
    pa.lam = pd.lam;
    pa.mu = pd.mu;
    gauss_legendre(NG, pa.g.x, pa.g.w);
    const int cus = device_cu_count();
    for (int32_t e0 = 0; e0 < pd.n_active; e0 += batch) {
        pa.elems = pd.elems.p + e0;
        pa.offs = pd.offs.p + e0;
        pa.n_active = std::min(batch, pd.n_active - e0);
        constexpr int GEO_EPB = 4;   // elements per workgroup, one wave each
        hipLaunchKernelGGL((elem_geo_kernel<P, NG>), dim3((unsigned)((pa.n_active + GEO_EPB - 1) / GEO_EPB)), dim3(256), 0,
                           st, pa, pd.geo.p);
        hipEvent_t ea = nullptr, eb = nullptr;
        if (h->timing) {
            int rc = timing_events(h, h->ev_used++, &ea, &eb);
            if (rc) return rc;
            YETI_HIP(hipEventRecord(ea, st));
        }
        if constexpr (P == 3) {
            int rc = launch_elem_p3(pd.geo.p, pa.offs, pa.n_active, pa.lam, pa.mu, cus, Kd, Kr, Kc, st);
            if (rc) return rc;
        } else {
            GenArgs ga = general_args(h, pd);
            ga.elems = pa.elems;
            ga.offs = pa.offs;
            ga.n_active = pa.n_active;
            ga.geo = pd.geo.p;
            ga.geo_rec = C::REC;
            int rc = launch_elem_general(ga, false, Kd, Kr, Kc, st);
            if (rc) return rc;
        }
        if (h->timing) YETI_HIP(hipEventRecord(eb, st));
    }
    return 0;
}

// Degree triples and Gauss orders the fixed-degree kernels are not built for (elem_general.hip).
static int launch_generic(yeti_asm *h, PatchDev &pd, double *Kd, int32_t *Kr, int32_t *Kc, hipStream_t st,
                          bool mass = false) {
    const GenArgs ga = general_args(h, pd);
    hipEvent_t ea = nullptr, eb = nullptr;
    if (h->timing && !mass) {
        int rc = timing_events(h, h->ev_used++, &ea, &eb);
        if (rc) return rc;
        YETI_HIP(hipEventRecord(ea, st));
    }
    int rc = launch_elem_general(ga, mass, Kd, Kr, Kc, st);
    if (rc == 0 && eb) YETI_HIP(hipEventRecord(eb, st));
    return rc;
}

static int run_elements(yeti_asm *h, double *Kd, int32_t *Kr, int32_t *Kc, hipStream_t st) {
    h->ev_used = 0;
    for (auto &zr : h->zero_ranges) {
        int64_t n = zr.second;
        int blocks = (int)std::min<int64_t>((n + 255) / 256, 65536);
        hipLaunchKernelGGL(fill_zero_kernel, dim3(blocks), dim3(256), 0, st, Kd + zr.first,
                           Kr ? Kr + zr.first : nullptr, Kc ? Kc + zr.first : nullptr, n);
        YETI_HIP(hipGetLastError());
    }
    for (auto *pd : h->patches) {
        if (!pd->u1 || pd->n_active == 0) continue;
        int rc = 0;
        if (!fixed_kernel_available(pd->p[0], pd->p[1], pd->p[2], pd->ng)) {
            rc = launch_generic(h, *pd, Kd, Kr, Kc, st);
            if (rc) return rc;
            continue;
        }
        int key = pd->p[0] * 16 + pd->ng;
        switch (key) {
        case 3 * 16 + 4: rc = launch_elem<3, 4>(h, *pd, h->coords.p, Kd, Kr, Kc, st); break;
        case 4 * 16 + 5: rc = launch_elem<4, 5>(h, *pd, h->coords.p, Kd, Kr, Kc, st); break;
        default: return set_error(YETI_ERR_UNSUPPORTED_DEGREE, "no kernel for p=%d ng=%d", pd->p[0], pd->ng);
        }
        if (rc) return rc;
    }
    return 0;
}

// ---------------------------------------------------------------------------------------
// Consistent mass matrix (compute_CMASSMatrix.f:22-215 with UMASSMAT_byCP, UMASSMAT.f:220-330,
// solid branch): M_ab[k][k] = sum_q rho w_q DetJac_q R_a(q) R_b(q) (DetJac signed, parent ->
// physical), off-diagonal k != l entries 0, emitted in the stiffness COO layout (a < b: 3 x 3
// block, kk fastest; a = b: the upper 6 with the diagonal halved) at the same element offsets.
// One 256-thread workgroup per element (grid-stride over the active elements), Gauss points in
// chunks of MQC:
//   1. the 1D bases of the chunk's points, one thread per (point, direction);
//   2. W, dW and the Jacobian of each point from G = 256 / MQC threads that split its nodes and
//      add their sums with lane shuffles;
//   3. R_a(q) = N_a w_a / W for the chunk in LDS (node-major, points contiguous);
//   4. the node-pair sums as 16 x 16 tiles (a tile, b tile) of (dv R)^T R on
//      v_mfma_f64_16x16x4f64, upper tiles spread over the four waves, accumulated over chunks;
// then the upper triangle of M goes to LDS (packed by column, b (b + 1) / 2 + a) and all threads
// write the element's COO range front to back, so every store of a wave is one contiguous run.
template <int P, int NG>
struct MassCfg {
    static constexpr int NP1 = P + 1, NN = NP1 * NP1 * NP1, NQ = NG * NG * NG;
    static constexpr int NNP = (NN + 15) / 16 * 16, NT = NNP / 16, NTILE = NT * (NT + 1) / 2;
    static constexpr int MAXT = (NTILE + 3) / 4;                       // tiles per wave
    // points per chunk: 32, so that at p = 3 the LDS (26 KB) and registers (compiled for
    // 4 waves per SIMD) allow 4 workgroups per CU (64-point chunks: 49 KB, 3 per CU, 16.6 ms
    // against 15.5 ms at 64^3)
    static constexpr int MQC = 32;
    static constexpr int G = 256 / MQC;                                // threads per point
    static constexpr int RS = MQC + 2;                                 // R row stride (doubles)
    static constexpr int NPAIR = NN * (NN + 1) / 2;
    // LDS (doubles): xw, dvq, then R + bases, which the packed M reuses after the last chunk
    static constexpr int O_DV = 4 * NN, O_U = O_DV + MQC;
    static constexpr int O_B = O_U + NNP * RS, O_DB = O_B + MQC * 3 * NP1;
    static constexpr int N_U = NNP * RS + 2 * MQC * 3 * NP1;
    static constexpr int NDBL = O_U + (N_U > NPAIR ? N_U : NPAIR);
    static constexpr int NCOO = coo_start(NN);
};

template <int P, int NG, bool WRITE_IDX>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(P == 3 ? 4 : 1)))
mass_kernel(PatchArgs pa, double rho, double *__restrict__ Md,
                                                   int32_t *__restrict__ Mr, int32_t *__restrict__ Mc) {
    using C = MassCfg<P, NG>;
    constexpr int NP1 = C::NP1, NN = C::NN, NQ = C::NQ, MQC = C::MQC, G = C::G, RS = C::RS;
    __shared__ __attribute__((aligned(16))) double sm[C::NDBL];
    __shared__ double hel[3], wiq[MQC];
    __shared__ int32_t dof[NN];
    double(*xw)[4] = reinterpret_cast<double(*)[4]>(sm);
    double *dvq = sm + C::O_DV;
    double *Rq = sm + C::O_U;                                              // [NNP][RS]
    double(*Bq)[3][NP1] = reinterpret_cast<double(*)[3][NP1]>(sm + C::O_B);
    double(*dBq)[3][NP1] = reinterpret_cast<double(*)[3][NP1]>(sm + C::O_DB);
    double *mp = sm + C::O_U;                                              // packed upper M
    const int t = threadIdx.x, lane = t & 63, wv = t >> 6;
    const int nl = lane & 15, kg = lane >> 4;
    const int qq = t / G, part = t % G;
    // this wave's tiles u = wv + 4 s, numbered column by column: u = tb (tb + 1) / 2 + ta
    int ta[C::MAXT], tb[C::MAXT];
#pragma unroll
    for (int s = 0; s < C::MAXT; ++s) {
        const int u = wv + 4 * s;
        int j = 0;
        while ((j + 1) * (j + 2) / 2 <= u) ++j;
        tb[s] = j;
        ta[s] = u - j * (j + 1) / 2;
    }
    for (int64_t gi = blockIdx.x; gi < pa.n_active; gi += gridDim.x) {
        const int e = pa.elems[gi];
        __syncthreads();   // the previous element is done with the LDS arrays
        for (int a = t; a < NN; a += 256) {
            const int32_t cp = pa.ien[(int64_t)NN * e + a] - 1;
            xw[a][0] = pa.coords[3 * (int64_t)cp];
            xw[a][1] = pa.coords[3 * (int64_t)cp + 1];
            xw[a][2] = pa.coords[3 * (int64_t)cp + 2];
            xw[a][3] = pa.weight[(int64_t)NN * e + a];
            dof[a] = 3 * cp;
        }
        f64x4 acc[C::MAXT];
#pragma unroll
        for (int s = 0; s < C::MAXT; ++s) acc[s] = f64x4{0.0, 0.0, 0.0, 0.0};
        for (int q0 = 0; q0 < NQ; q0 += MQC) {
            const int nq = NQ - q0 < MQC ? NQ - q0 : MQC;
            __syncthreads();
            // 1. bases: direction `part` of point qq (shap.f90:75-178); the reference's 3D rule
            // runs i (xi) slowest and k (zeta) fastest (GaussLegendre.f90:175-186)
            if (part < 3 && qq < nq) {
                const int q = q0 + qq, d = part;
                const int gd = d == 0 ? q / (NG * NG) : d == 1 ? (q / NG) % NG : q % NG;
                const double *U = d == 0 ? pa.U0 : d == 1 ? pa.U1 : pa.U2;
                const int span1 = pa.nijk[3 * (int64_t)e + d];
                const double u0 = U[span1 - 1], u1 = U[span1];
                const double u = ((u1 - u0) * pa.g.x[gd] + (u1 + u0)) * 0.5;
                double N[NP1], dN[NP1];
                bspline_ders<P>(span1 - 1, u, U, N, dN);
#pragma unroll
                for (int i = 0; i < NP1; ++i) {
                    Bq[qq][d][i] = N[P - i];
                    dBq[qq][d][i] = dN[P - i];
                }
                if (qq == 0) hel[d] = 0.5 * (u1 - u0);
            }
            __syncthreads();
            // 2. W, dW/dxi and dX/dxi of point qq: nodes part, part + G, ... then a shuffle sum
            {
                double s[16];
#pragma unroll
                for (int k = 0; k < 16; ++k) s[k] = 0.0;
                if (qq < nq) {
#pragma unroll 1
                    for (int a = part; a < NN; a += G) {
                        const int i = a % NP1, j = (a / NP1) % NP1, k = a / (NP1 * NP1);
                        const double w = xw[a][3], x0 = xw[a][0], x1 = xw[a][1], x2 = xw[a][2];
                        const double B0 = Bq[qq][0][i], B1 = Bq[qq][1][j], B2 = Bq[qq][2][k];
                        const double b12 = B1 * B2 * w;
                        const double Na = B0 * b12;
                        const double d0 = dBq[qq][0][i] * b12;
                        const double d1 = B0 * dBq[qq][1][j] * B2 * w;
                        const double d2 = B0 * B1 * dBq[qq][2][k] * w;
                        s[0] += Na;
                        s[1] += d0; s[2] += d1; s[3] += d2;
                        s[4] += x0 * Na; s[5] += x1 * Na; s[6] += x2 * Na;
                        s[7] += x0 * d0; s[8] += x0 * d1; s[9] += x0 * d2;
                        s[10] += x1 * d0; s[11] += x1 * d1; s[12] += x1 * d2;
                        s[13] += x2 * d0; s[14] += x2 * d1; s[15] += x2 * d2;
                    }
                }
#pragma unroll
                for (int o = 1; o < G; o <<= 1)   // the G threads of a point are adjacent lanes
#pragma unroll
                    for (int k = 0; k < 16; ++k) s[k] += __shfl_xor(s[k], o, 64);
                if (part == 0) {
                    double dv = 0.0, Wi = 0.0;
                    if (qq < nq) {
                        const int q = q0 + qq;
                        Wi = 1.0 / s[0];
                        const double dw[3] = {s[1] * Wi, s[2] * Wi, s[3] * Wi};
                        double J[3][3];
#pragma unroll
                        for (int r = 0; r < 3; ++r)
#pragma unroll
                            for (int c = 0; c < 3; ++c) J[r][c] = (s[7 + 3 * r + c] - s[4 + r] * dw[c]) * Wi;
                        const double det = J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) +
                                           J[0][1] * (J[1][2] * J[2][0] - J[1][0] * J[2][2]) +
                                           J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
                        const int g0 = q / (NG * NG), g1 = (q / NG) % NG, g2 = q % NG;
                        dv = rho * (pa.g.w[g0] * pa.g.w[g1] * pa.g.w[g2]) * (det * hel[0] * hel[1] * hel[2]);
                    }
                    dvq[qq] = dv;   // 0 at the padding points of the last chunk
                    wiq[qq] = Wi;
                }
            }
            __syncthreads();
            // 3. R_a(q) = N_a w_a / W; zero rows past NN and columns past nq
            for (int x = t; x < C::NNP * MQC; x += 256) {
                const int a = x / MQC, c = x % MQC;
                double r = 0.0;
                if (a < NN && c < nq) {
                    const int i = a % NP1, j = (a / NP1) % NP1, k = a / (NP1 * NP1);
                    r = Bq[c][0][i] * Bq[c][1][j] * Bq[c][2][k] * xw[a][3] * wiq[c];
                }
                Rq[a * RS + c] = r;
            }
            __syncthreads();
            // 4. tile sums; K step 2v uses point 8v + 2 kg, step 2v + 1 point 8v + 2 kg + 1 (A and
            // B with the same permutation of the K sum)
#pragma unroll 1
            for (int v = 0; v < MQC / 8; ++v) {
                const int qo = 8 * v + 2 * kg;
                const f64x2 dv2 = *reinterpret_cast<const f64x2 *>(dvq + qo);
#pragma unroll
                for (int s = 0; s < C::MAXT; ++s) {
                    if (wv + 4 * s < C::NTILE) {
                        f64x2 A = *reinterpret_cast<const f64x2 *>(Rq + (16 * ta[s] + nl) * RS + qo);
                        const f64x2 B = *reinterpret_cast<const f64x2 *>(Rq + (16 * tb[s] + nl) * RS + qo);
                        A.x *= dv2.x;
                        A.y *= dv2.y;
                        acc[s] = __builtin_amdgcn_mfma_f64_16x16x4f64(A.x, B.x, acc[s], 0, 0, 0);
                        acc[s] = __builtin_amdgcn_mfma_f64_16x16x4f64(A.y, B.y, acc[s], 0, 0, 0);
                    }
                }
            }
        }
        __syncthreads();   // every wave is done with R before M overwrites it
        // accumulator lane layout: register r of lane l holds row (l >> 4) + 4 r, column l & 15
#pragma unroll
        for (int s = 0; s < C::MAXT; ++s) {
            if (wv + 4 * s < C::NTILE) {
                const int b = 16 * tb[s] + nl;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int a = 16 * ta[s] + kg + 4 * r;
                    if (a <= b && b < NN) mp[b * (b + 1) / 2 + a] = acc[s][r];
                }
            }
        }
        __syncthreads();
        // emission: entry x of the element's range lies in column b with start(b) <= x < start(b+1)
        const int64_t base = pa.offs[gi];
        int b = 0;
        for (int x = t; x < C::NCOO; x += 256) {
            while (b + 1 < NN && coo_start(b + 1) <= x) ++b;
            const unsigned r = (unsigned)(x - coo_start(b));
            const int mb = b * (b + 1) / 2;
            double v;
            int32_t row, col;
            if (r < 9u * (unsigned)b) {
                const unsigned a = r / 9u, y = r - 9u * a, kk = y % 3u, ll = y / 3u;
                v = kk == ll ? mp[mb + (int)a] : 0.0;
                row = dof[a] + (int)kk;
                col = dof[b] + (int)ll;
            } else {
                const unsigned y = r - 9u * (unsigned)b;   // (0,0) (0,1) (1,1) (0,2) (1,2) (2,2)
                const int kk = (0x210100 >> (4 * y)) & 15, ll = (0x222110 >> (4 * y)) & 15;
                v = kk == ll ? 0.5 * mp[mb + b] : 0.0;
                row = dof[b] + kk;
                col = dof[b] + ll;
            }
            // streaming output, read back by no kernel of this launch
            __builtin_nontemporal_store(v, Md + base + x);
            if (WRITE_IDX) {
                __builtin_nontemporal_store(row, Mr + base + x);
                __builtin_nontemporal_store(col, Mc + base + x);
            }
        }
    }
}

template <int P, int NG>
static int launch_mass(yeti_asm *h, PatchDev &pd, double *Md, int32_t *Mr, int32_t *Mc, hipStream_t st) {
    PatchArgs pa{};
    pa.coords = h->coords.p;
    pa.ien = pd.ien.p;
    pa.weight = pd.weight.p;
    pa.nijk = pd.nijk.p;
    pa.U0 = pd.U[0];
    pa.U1 = pd.U[1];
    pa.U2 = pd.U[2];
    pa.elems = pd.elems.p;
    pa.offs = pd.offs.p;
    pa.n_active = pd.n_active;
    gauss_legendre(NG, pa.g.x, pa.g.w);
    const unsigned grid = (unsigned)std::min<int64_t>(pd.n_active, 1 << 20);
    if (Mr)
        hipLaunchKernelGGL((mass_kernel<P, NG, true>), dim3(grid), dim3(256), 0, st, pa, pd.rho, Md, Mr, Mc);
    else
        hipLaunchKernelGGL((mass_kernel<P, NG, false>), dim3(grid), dim3(256), 0, st, pa, pd.rho, Md, Mr, Mc);
    YETI_HIP(hipGetLastError());
    return 0;
}

// p = 3 and 4 take mass_kernel, whose waves share an element's tiles (32^3 p = 3: 2.04 ms against 3.57 ms
// of elem_general.hip), the rest elem_general.hip
static int run_mass(yeti_asm *h, double *Md, int32_t *Mr, int32_t *Mc, hipStream_t st) {
    for (auto &zr : h->zero_ranges) {
        int64_t n = zr.second;
        int blocks = (int)std::min<int64_t>((n + 255) / 256, 65536);
        hipLaunchKernelGGL(fill_zero_kernel, dim3(blocks), dim3(256), 0, st, Md + zr.first,
                           Mr ? Mr + zr.first : nullptr, Mc ? Mc + zr.first : nullptr, n);
        YETI_HIP(hipGetLastError());
    }
    for (auto *pd : h->patches) {
        if (!pd->u1 || pd->n_active == 0) continue;
        int rc = 0;
        if (!fixed_kernel_available(pd->p[0], pd->p[1], pd->p[2], pd->ng)) {   // other degree triples / orders
            rc = launch_generic(h, *pd, Md, Mr, Mc, st, true);
            if (rc) return rc;
            continue;
        }
        switch (pd->p[0] * 16 + pd->ng) {
        case 3 * 16 + 4: rc = launch_mass<3, 4>(h, *pd, Md, Mr, Mc, st); break;
        case 4 * 16 + 5: rc = launch_mass<4, 5>(h, *pd, Md, Mr, Mc, st); break;
        default: return set_error(YETI_ERR_UNSUPPORTED_DEGREE, "mass: no kernel for p=%d ng=%d", pd->p[0], pd->ng);
        }
        if (rc) return rc;
    }
    return 0;
}

// B-spline values and first derivatives at u for a run-time degree p <= PMAX, span i (0-based):
// the triangular recurrence with the degree p - 1 values kept for the derivatives (the contract
// of dersbasisfuns.f90:30-131, first derivative only)
template <int PMAX>
__device__ inline void bspline_ders_rt(int i, int p, double u, const double *__restrict__ U, double *N, double *dN) {
    double lf[PMAX + 1], rt[PMAX + 1], lo[PMAX + 1];
    N[0] = 1.0;
    lo[0] = 1.0;
    for (int j = 1; j <= p; ++j) {
        lf[j] = u - U[i + 1 - j];
        rt[j] = U[i + j] - u;
        double saved = 0.0;
        for (int r = 0; r < j; ++r) {
            const double tmp = N[r] / (rt[r + 1] + lf[j - r]);
            N[r] = saved + rt[r + 1] * tmp;
            saved = lf[j - r] * tmp;
        }
        N[j] = saved;
        if (j == p - 1)
            for (int r = 0; r < p; ++r) lo[r] = N[r];
    }
    for (int r = 0; r <= p; ++r) {
        const int k = i - p + r;
        double dd = 0.0;
        if (r >= 1 && U[k + p] != U[k]) dd += p * lo[r - 1] / (U[k + p] - U[k]);
        if (r <= p - 1 && U[k + p + 1] != U[k + 1]) dd -= p * lo[r] / (U[k + p + 1] - U[k + 1]);
        dN[r] = dd;
    }
}

// Shape gradients of models with other than max(p) + 1 Gauss points per direction: run-time
// degrees and order, one 256-thread workgroup per active element, Gauss points in chunks of VQC:
//   1. bases, one thread per (point, direction);
//   2. W, dW and dx/du of a point by 256 / VQC threads and a shuffle sum, then du/dx and dv;
//   3. R and dR/dx of every (node, point) of the chunk in LDS;
//   4. per (point, pair): the tensor T[m][k] and the mass;
//   5. per (node, pair): g += tensor . dR/dx, accumulated over the chunks in the registers of the
//      (node, pair)'s thread.
constexpr int VQC = 16;

struct GradDegrees {
    int p[3];
    int ng;
};

template <int KIND>
__global__ void __launch_bounds__(256) shape_grad_rt_kernel(PatchArgs pa, GradFields gf, GradDegrees dg,
                                                            int64_t ebase, double *__restrict__ eg,
                                                            double *__restrict__ em) {
    constexpr int P = GEN_MAXP, NP1 = P + 1, NN = GEN_MAXN, G = 256 / VQC;
    const int p0 = dg.p[0], p1 = dg.p[1], p2 = dg.p[2];
    const int n0 = p0 + 1, n1 = p1 + 1, nn = n0 * n1 * (p2 + 1);
    const int ng = dg.ng, NQ = ng * ng * ng;
    constexpr int NFLD = KIND == GRAD_VOLUME ? 1 : KIND == GRAD_PAIRS ? VIB_MAXF + 1 : VIB_MAXF;
    __shared__ double xw[NN][4];
    __shared__ double uf[NFLD][NN][3];
    __shared__ double Bq[VQC][3][NP1], dBq[VQC][3][NP1];
    __shared__ double gq[VQC][14];     // du/dx (9, [c][k] = du_c/dx_k), dv, 1/W, dW/du / W (3)
    __shared__ double Rx[NN][VQC][4];  // R, dR/dx
    __shared__ double Tq[VQC][VIB_MAXF][9];
    __shared__ double mpart[VQC][VIB_MAXF];
    __shared__ double hel[3];
    const int t = threadIdx.x;
    const int nf = KIND == GRAD_VOLUME ? 1 : gf.nf;
    const int qq = t / G, part = t % G;
    for (int64_t gi = blockIdx.x; gi < pa.n_active; gi += gridDim.x) {
        const int e = pa.elems[gi];
        __syncthreads();   // the previous element is done with the LDS arrays
        for (int a = t; a < nn; a += 256) {
            const int64_t cp = (int64_t)pa.ien[(int64_t)nn * e + a] - 1;
            xw[a][0] = pa.coords[3 * cp];
            xw[a][1] = pa.coords[3 * cp + 1];
            xw[a][2] = pa.coords[3 * cp + 2];
            xw[a][3] = pa.weight[(int64_t)nn * e + a];
            if (KIND != GRAD_VOLUME)
                for (int c = 0; c < 3; ++c) {
                    for (int f = 0; f < nf; ++f) uf[f][a][c] = gf.fk[(gf.k0 + f) + (int64_t)gf.nk * (c + 3 * cp)];
                    if (KIND == GRAD_PAIRS) uf[NFLD - 1][a][c] = gf.f0[c + 3 * cp];
                }
        }
        // this thread's node sums: (node, pair) x = t + 256 s, a = x mod nn, f = x / nn
        constexpr int GSL = (NN * VIB_MAXF + 255) / 256;
        double gr[GSL][3];
#pragma unroll
        for (int s = 0; s < GSL; ++s) gr[s][0] = gr[s][1] = gr[s][2] = 0.0;
        double macc = 0.0;   // this thread's (point, pair) share of the element mass
        for (int q0 = 0; q0 < NQ; q0 += VQC) {
            const int nq = NQ - q0 < VQC ? NQ - q0 : VQC;
            __syncthreads();
            // 1. bases of direction `part` at point qq (shap.f90:75-178 for the parametric form)
            if (part < 3 && qq < nq) {
                const int q = q0 + qq, d = part;
                const int gd = d == 0 ? q / (ng * ng) : d == 1 ? (q / ng) % ng : q % ng;
                const double *U = d == 0 ? pa.U0 : d == 1 ? pa.U1 : pa.U2;
                const int span1 = pa.nijk[3 * (int64_t)e + d];
                const double u0 = U[span1 - 1], u1 = U[span1];
                const double u = ((u1 - u0) * pa.g.x[gd] + (u1 + u0)) * 0.5;
                double N[NP1], dN[NP1];
                const int pd = d == 0 ? p0 : d == 1 ? p1 : p2;
                bspline_ders_rt<P>(span1 - 1, pd, u, U, N, dN);
                for (int i = 0; i <= pd; ++i) {
                    Bq[qq][d][i] = N[pd - i];
                    dBq[qq][d][i] = dN[pd - i];
                }
                if (qq == 0) hel[d] = 0.5 * (u1 - u0);
            }
            __syncthreads();
            // 2. W, dW/du and dx/du of point qq: nodes part, part + G, ... then a shuffle sum
            {
                double s[16];
#pragma unroll
                for (int k = 0; k < 16; ++k) s[k] = 0.0;
                if (qq < nq) {
#pragma unroll 1
                    for (int a = part; a < nn; a += G) {
                        const int i = a % n0, j = (a / n0) % n1, k = a / (n0 * n1);
                        const double w = xw[a][3], x0 = xw[a][0], x1 = xw[a][1], x2 = xw[a][2];
                        const double B0 = Bq[qq][0][i], B1 = Bq[qq][1][j], B2 = Bq[qq][2][k];
                        const double b12 = B1 * B2 * w;
                        const double Na = B0 * b12;
                        const double d0 = dBq[qq][0][i] * b12;
                        const double d1 = B0 * dBq[qq][1][j] * B2 * w;
                        const double d2 = B0 * B1 * dBq[qq][2][k] * w;
                        s[0] += Na;
                        s[1] += d0; s[2] += d1; s[3] += d2;
                        s[4] += x0 * Na; s[5] += x1 * Na; s[6] += x2 * Na;
                        s[7] += x0 * d0; s[8] += x0 * d1; s[9] += x0 * d2;
                        s[10] += x1 * d0; s[11] += x1 * d1; s[12] += x1 * d2;
                        s[13] += x2 * d0; s[14] += x2 * d1; s[15] += x2 * d2;
                    }
                }
#pragma unroll
                for (int o = 1; o < G; o <<= 1)   // the G threads of a point are adjacent lanes
#pragma unroll
                    for (int k = 0; k < 16; ++k) s[k] += __shfl_xor(s[k], o, 64);
                if (part == 0) {
                    double *gp = gq[qq];
                    if (qq < nq) {
                        const int q = q0 + qq;
                        const double Wi = 1.0 / s[0];
                        const double dw[3] = {s[1] * Wi, s[2] * Wi, s[3] * Wi};
                        double J[3][3];   // dx_r / du_c
#pragma unroll
                        for (int r = 0; r < 3; ++r)
#pragma unroll
                            for (int c = 0; c < 3; ++c) J[r][c] = (s[7 + 3 * r + c] - s[4 + r] * dw[c]) * Wi;
                        const double det = J[0][0] * (J[1][1] * J[2][2] - J[1][2] * J[2][1]) +
                                           J[0][1] * (J[1][2] * J[2][0] - J[1][0] * J[2][2]) +
                                           J[0][2] * (J[1][0] * J[2][1] - J[1][1] * J[2][0]);
                        const double di = 1.0 / det;
                        gp[0] = (J[1][1] * J[2][2] - J[1][2] * J[2][1]) * di;
                        gp[1] = (J[0][2] * J[2][1] - J[0][1] * J[2][2]) * di;
                        gp[2] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]) * di;
                        gp[3] = (J[1][2] * J[2][0] - J[1][0] * J[2][2]) * di;
                        gp[4] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) * di;
                        gp[5] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) * di;
                        gp[6] = (J[1][0] * J[2][1] - J[1][1] * J[2][0]) * di;
                        gp[7] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) * di;
                        gp[8] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * di;
                        const int g0 = q / (ng * ng), g1 = (q / ng) % ng, g2 = q % ng;
                        gp[9] = (pa.g.w[g0] * pa.g.w[g1] * pa.g.w[g2]) * (det * hel[0] * hel[1] * hel[2]);
                        gp[10] = Wi;
                        gp[11] = dw[0];
                        gp[12] = dw[1];
                        gp[13] = dw[2];
                    } else {
                        for (int k = 0; k < 14; ++k) gp[k] = 0.0;
                    }
                }
            }
            __syncthreads();
            // 3. R = N w / W and dR/dx = (dN w / W - R dW / W) du/dx
            for (int x = t; x < nn * VQC; x += 256) {
                const int a = x / VQC, c = x % VQC;
                double r4[4] = {0.0, 0.0, 0.0, 0.0};
                if (c < nq) {
                    const int i = a % n0, j = (a / n0) % n1, k = a / (n0 * n1);
                    const double w = xw[a][3], Wi = gq[c][10];
                    const double B0 = Bq[c][0][i], B1 = Bq[c][1][j], B2 = Bq[c][2][k];
                    const double R = B0 * B1 * B2 * w * Wi;
                    const double du[3] = {dBq[c][0][i] * B1 * B2 * w * Wi - R * gq[c][11],
                                          B0 * dBq[c][1][j] * B2 * w * Wi - R * gq[c][12],
                                          B0 * B1 * dBq[c][2][k] * w * Wi - R * gq[c][13]};
                    r4[0] = R;
                    for (int kk = 0; kk < 3; ++kk)
                        r4[1 + kk] = du[0] * gq[c][kk] + du[1] * gq[c][3 + kk] + du[2] * gq[c][6 + kk];
                }
                for (int kk = 0; kk < 4; ++kk) Rx[a][c][kk] = r4[kk];
            }
            __syncthreads();
            // 4. per (point, pair): the fields, stresses, the tensor and the mass; the nodes of a
            // (point, pair) are split over 4 adjacent lanes and their sums added by shuffles
            {
                const int pr = t >> 2, part4 = t & 3, c = pr % VQC, f = pr / VQC;
                const bool act = f < nf && c < nq;
                double u[3] = {0.0, 0.0, 0.0}, D[3][3] = {}, H[3][3] = {};   // D[i][k] = dv_i/dx_k, H: field 0
                if (KIND != GRAD_VOLUME && act) {
#pragma unroll 1
                    for (int a = part4; a < nn; a += 4) {
                        const double R = Rx[a][c][0], g0 = Rx[a][c][1], g1 = Rx[a][c][2], g2 = Rx[a][c][3];
#pragma unroll
                        for (int i = 0; i < 3; ++i) {
                            const double ua = uf[f][a][i];
                            u[i] += R * ua;
                            D[i][0] += ua * g0;
                            D[i][1] += ua * g1;
                            D[i][2] += ua * g2;
                            if (KIND == GRAD_PAIRS) {
                                const double u0 = uf[NFLD - 1][a][i];
                                H[i][0] += u0 * g0;
                                H[i][1] += u0 * g1;
                                H[i][2] += u0 * g2;
                            }
                        }
                    }
                }
#pragma unroll
                for (int o = 1; o < 4; o <<= 1) {
#pragma unroll
                    for (int i = 0; i < 3; ++i) {
                        u[i] += __shfl_xor(u[i], o, 64);
#pragma unroll
                        for (int k = 0; k < 3; ++k) {
                            D[i][k] += __shfl_xor(D[i][k], o, 64);
                            if (KIND == GRAD_PAIRS) H[i][k] += __shfl_xor(H[i][k], o, 64);
                        }
                    }
                }
                if (KIND == GRAD_MODES)
#pragma unroll
                    for (int i = 0; i < 3; ++i)
#pragma unroll
                        for (int k = 0; k < 3; ++k) H[i][k] = D[i][k];
                if (part4 == 0 && f < nf) {
                    double T[9] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
                    if (c < nq) {
                        const double lam = pa.lam, mu = pa.mu, dv = gq[c][9];
                        const double td = lam * (D[0][0] + D[1][1] + D[2][2]), th = lam * (H[0][0] + H[1][1] + H[2][2]);
                        double sd[3][3], sh[3][3], W = 0.0;
#pragma unroll
                        for (int i = 0; i < 3; ++i)
#pragma unroll
                            for (int k = 0; k < 3; ++k) {
                                sd[i][k] = mu * (D[i][k] + D[k][i]) + (i == k ? td : 0.0);
                                sh[i][k] = mu * (H[i][k] + H[k][i]) + (i == k ? th : 0.0);
                                W += sh[i][k] * D[i][k];
                            }
                        const double uu = KIND == GRAD_MODES ? gf.rho * (u[0] * u[0] + u[1] * u[1] + u[2] * u[2])
                                                             : KIND == GRAD_VOLUME ? 1.0 : 0.0;
                        const double Wp = KIND == GRAD_VOLUME ? 1.0 : KIND == GRAD_MODES ? W - gf.vals[f] * uu : W;
#pragma unroll
                        for (int m = 0; m < 3; ++m)
#pragma unroll
                            for (int k = 0; k < 3; ++k) {
                                double v = m == k ? Wp : 0.0;
#pragma unroll
                                for (int i = 0; i < 3; ++i)
                                    v -= KIND == GRAD_MODES ? 2.0 * (D[i][m] * sd[i][k]) : D[i][m] * sh[i][k] + H[i][m] * sd[i][k];
                                T[3 * m + k] = dv * v;
                            }
                        macc += uu * dv;
                    }
                    for (int k = 0; k < 9; ++k) Tq[c][f][k] = T[k];
                }
            }
            __syncthreads();
            // 5. per (node, pair): g[m] += sum_q T[m][k] dR/dx_k
#pragma unroll
            for (int s = 0; s < GSL; ++s) {
                const int x = t + 256 * s;
                if (x >= nn * nf) continue;
                const int a = x % nn, f = x / nn;
                double g[3] = {0.0, 0.0, 0.0};
                for (int c = 0; c < nq; ++c) {
                    const double g0 = Rx[a][c][1], g1 = Rx[a][c][2], g2 = Rx[a][c][3];
#pragma unroll
                    for (int m = 0; m < 3; ++m)
                        g[m] += Tq[c][f][3 * m] * g0 + Tq[c][f][3 * m + 1] * g1 + Tq[c][f][3 * m + 2] * g2;
                }
#pragma unroll
                for (int m = 0; m < 3; ++m) gr[s][m] += g[m];
            }
        }
        if ((t & 3) == 0) mpart[(t >> 2) % VQC][(t >> 2) / VQC] = (t >> 2) / VQC < nf ? macc : 0.0;
        __syncthreads();
#pragma unroll
        for (int s = 0; s < GSL; ++s) {
            const int x = t + 256 * s;
            if (x >= nn * nf) continue;
            const int a = x % nn, f = x / nn;
#pragma unroll
            for (int m = 0; m < 3; ++m) eg[3 * (nf * (ebase + gi * nn + a) + f) + m] = gr[s][m];
        }
        if (t < VIB_MAXF) {
            double ms = 0.0;
            for (int c = 0; c < VQC; ++c) ms += mpart[c][t];
            em[gi * VIB_MAXF + t] = ms;
        }
    }
}

// Total mass of pair f over the slots, in a fixed order (one block per pair).
__global__ void __launch_bounds__(256) grad_mass_kernel(const double *em, int64_t nslot, double *mass) {
    __shared__ double sh[256];
    const int f = blockIdx.x;
    double v = 0.0;
#pragma unroll 4
    for (int64_t i = threadIdx.x; i < nslot; i += 256) v += em[i * VIB_MAXF + f];
    sh[threadIdx.x] = v;
    __syncthreads();
    for (int o = 128; o > 0; o >>= 1) {
        if ((int)threadIdx.x < o) sh[threadIdx.x] += sh[threadIdx.x + o];
        __syncthreads();
    }
    if (threadIdx.x == 0) mass[f] = sh[0];
}

// out[k0 + f, m, cp] = scale times the sum over the element-node entries of cp, in entry order,
// divided by mass[f] when mass is given; one thread per (cp, f, m), so that neighbouring threads
// read an entry's pairs as one run (33x29x26 p=3, 4 modes: 62 us with the pairs in separate arrays
// -> 28 us; the element kernel's stores, then in 24-byte runs, take 13 us more). GU entries are in
// flight at once.
__global__ void __launch_bounds__(256) grad_gather_kernel(int32_t nb_cp, const int32_t *__restrict__ ptr,
                                                          const int32_t *__restrict__ ent,
                                                          const double *__restrict__ eg, int32_t nf,
                                                          const double *__restrict__ mass, double scale, int32_t k0,
                                                          int32_t nk, double *__restrict__ out) {
    constexpr int GU = 8;
    const int row = 3 * nf;
    for (int64_t x = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; x < row * (int64_t)nb_cp;
         x += (int64_t)gridDim.x * blockDim.x) {
        const int32_t cp = (int32_t)(x / row);
        const int fm = (int)(x - row * (int64_t)cp), f = fm / 3, m = fm - 3 * f;
        const double *g = eg + fm;
        double s = 0.0;
        const int64_t j1 = ptr[cp + 1];
        for (int64_t j = ptr[cp]; j < j1; j += GU) {
            double v[GU];
#pragma unroll
            for (int u = 0; u < GU; ++u) v[u] = g[row * (int64_t)ent[min(j + u, j1 - 1)]];
#pragma unroll
            for (int u = 0; u < GU; ++u) s += j + u < j1 ? v[u] : 0.0;
        }
        s *= scale;
        out[(k0 + f) + (int64_t)nk * (m + 3 * (int64_t)cp)] = mass ? s / mass[f] : s;
    }
}

// the sum-factorised kernel takes max(p) + 1 Gauss points (all degrees the stiffness accepts);
// other orders go to shape_grad_rt_kernel
static bool grad_factorised(const PatchDev &pd) { return pd.tab_n >= 2 && pd.tab_n <= 5 && pd.ng == pd.tab_n; }

// workgroups of the factorised kernel: a function of the element count only (each adds its
// elements' masses), enough for several per CU
template <int N, int Q>
static unsigned grad_grid(int32_t n_active) {
    constexpr int EPB = Grad<N, Q>::WPB * Grad<N, Q>::EPW;
    return (unsigned)std::min<int64_t>((n_active + EPB - 1) / EPB, 3072);
}

static unsigned grad_slots(const PatchDev &pd) {
    if (!grad_factorised(pd)) return (unsigned)pd.n_active;
    switch (pd.tab_n) {
    case 2: return grad_grid<2, 2>(pd.n_active);
    case 3: return grad_grid<3, 3>(pd.n_active);
    case 4: return grad_grid<4, 4>(pd.n_active);
    default: return grad_grid<5, 5>(pd.n_active);
    }
}

template <int N, int KIND>
static void launch_grad(yeti_asm *h, PatchDev &pd, const GradFields &gf, int64_t ebase, int64_t mbase, hipStream_t st) {
    GradArgs ga{};
    ga.coords = h->coords.p;
    ga.ien = pd.ien.p;
    ga.weight = pd.weight.p;
    ga.nijk = pd.nijk.p;
    for (int d = 0; d < 3; ++d) {
        ga.tab[d] = pd.tab[d];
        ga.n[d] = pd.p[d] + 1;
    }
    ga.elems = pd.elems.p;
    ga.n_active = pd.n_active;
    ga.lam = pd.lam;
    ga.mu = pd.mu;
    gauss_legendre(N, ga.g.x, ga.g.w);
    ga.f = gf;
    ga.eg = h->vib_eg.p;
    ga.ebase = ebase;
    ga.em = h->vib_em.p + mbase * VIB_MAXF;
    hipLaunchKernelGGL((shape_grad_kernel<N, N, KIND>), dim3(grad_grid<N, N>(pd.n_active)), dim3(64 * Grad<N, N>::WPB), 0,
                       st, ga);
}

template <int KIND>
static int launch_grad_kind(yeti_asm *h, PatchDev &pd, const GradFields &gf, int64_t ebase, int64_t mbase,
                            hipStream_t st) {
    if (grad_factorised(pd)) {
        switch (pd.tab_n) {
        case 2: launch_grad<2, KIND>(h, pd, gf, ebase, mbase, st); break;
        case 3: launch_grad<3, KIND>(h, pd, gf, ebase, mbase, st); break;
        case 4: launch_grad<4, KIND>(h, pd, gf, ebase, mbase, st); break;
        default: launch_grad<5, KIND>(h, pd, gf, ebase, mbase, st); break;
        }
    } else {
        PatchArgs pa{};
        pa.coords = h->coords.p;
        pa.ien = pd.ien.p;
        pa.weight = pd.weight.p;
        pa.nijk = pd.nijk.p;
        pa.U0 = pd.U[0];
        pa.U1 = pd.U[1];
        pa.U2 = pd.U[2];
        pa.elems = pd.elems.p;
        pa.n_active = pd.n_active;
        pa.lam = pd.lam;
        pa.mu = pd.mu;
        gauss_legendre(pd.ng, pa.g.x, pa.g.w);
        GradDegrees dg{{pd.p[0], pd.p[1], pd.p[2]}, pd.ng};
        const unsigned grid = (unsigned)std::min<int64_t>(pd.n_active, 1 << 20);
        hipLaunchKernelGGL((shape_grad_rt_kernel<KIND>), dim3(grid), dim3(256), 0, st, pa, gf, dg, ebase, h->vib_eg.p,
                           h->vib_em.p + mbase * VIB_MAXF);
    }
    YETI_HIP(hipGetLastError());
    return 0;
}

// CP -> element-node entries of the active U1 elements (entry = patch base + gi nnode + a), in
// patch, element and node order; buffers for the per-entry partials and the masses.
static int vib_setup(yeti_asm *h) {
    if (h->vib_nent >= 0) return 0;
    std::vector<int32_t> cnt(h->nb_cp + 1, 0);
    std::vector<std::vector<int32_t>> ien_h(h->patches.size()), el_h(h->patches.size());
    int64_t nent = 0, nslot = 0;
    for (size_t k = 0; k < h->patches.size(); ++k) {
        PatchDev &pd = *h->patches[k];
        if (!pd.u1 || pd.n_active == 0) continue;
        ien_h[k].resize((size_t)pd.nnode * pd.nelem);
        el_h[k].resize(pd.n_active);
        YETI_HIP(hipMemcpy(ien_h[k].data(), pd.ien.p, ien_h[k].size() * sizeof(int32_t), hipMemcpyDeviceToHost));
        YETI_HIP(hipMemcpy(el_h[k].data(), pd.elems.p, el_h[k].size() * sizeof(int32_t), hipMemcpyDeviceToHost));
        for (int32_t gi = 0; gi < pd.n_active; ++gi)
            for (int a = 0; a < pd.nnode; ++a) {
                const int32_t id = ien_h[k][(size_t)pd.nnode * el_h[k][gi] + a];   // 1-based
                if (id < 1 || id > h->nb_cp)
                    return set_error(YETI_ERR_INVALID_ARGUMENT, "vibration gradient: IEN entry %d out of range", id);
                ++cnt[id];
            }
        nent += (int64_t)pd.n_active * pd.nnode;
        nslot += grad_slots(pd);
    }
    if (nent > INT32_MAX) return set_error(YETI_ERR_SIZE_OVERFLOW, "vibration gradient: %lld element nodes", (long long)nent);
    std::vector<int32_t> ptr(h->nb_cp + 1, 0);
    for (int32_t c = 0; c < h->nb_cp; ++c) ptr[c + 1] = ptr[c] + cnt[c + 1];
    std::vector<int32_t> pos(ptr.begin(), ptr.end() - 1);
    std::vector<int32_t> ent(std::max<int64_t>(nent, 1));
    int64_t base = 0;
    for (size_t k = 0; k < h->patches.size(); ++k) {
        PatchDev &pd = *h->patches[k];
        if (!pd.u1 || pd.n_active == 0) continue;
        for (int32_t gi = 0; gi < pd.n_active; ++gi)
            for (int a = 0; a < pd.nnode; ++a) {
                const int32_t cp = ien_h[k][(size_t)pd.nnode * el_h[k][gi] + a] - 1;
                ent[pos[cp]++] = (int32_t)(base + (int64_t)gi * pd.nnode + a);
            }
        base += (int64_t)pd.n_active * pd.nnode;
    }
    YETI_HIP(h->vib_ptr.upload(ptr.data(), ptr.size()));
    YETI_HIP(h->vib_ent.upload(ent.data(), ent.size()));
    YETI_HIP(h->vib_eg.alloc((size_t)std::max<int64_t>(nent, 1) * VIB_MAXF * 3));
    YETI_HIP(h->vib_em.alloc((size_t)std::max<int64_t>(nslot, 1) * VIB_MAXF));
    YETI_HIP(h->vib_mass.alloc(VIB_MAXF));
    h->vib_nent = nent;
    h->vib_nslot = nslot;
    return 0;
}

// Gradients of npair pairs (kind: shape_grad.hpp) over the active solid elements:
// out[k, m, cp], (npair, 3, nb_cp) column-major, times scale, divided by the pair's mass when
// normalize. f0: field 0 of GRAD_PAIRS; fk: the npair fields (npair, 3, nb_cp) column-major; vals
// (host): eigenvalues, or null for 0. mass_out (device, one value per pair of the last launch), or
// null.
static int run_shape_grad(yeti_asm *h, GradKind kind, const double *f0, const double *fk, const double *vals,
                          int32_t npair, double *out, double scale, bool normalize, double *mass_out, hipStream_t st) {
    for (auto *pd : h->patches) {
        if (!pd->u1 || pd->n_active == 0) continue;
        const bool general = pd->p[0] >= 1 && pd->p[1] >= 1 && pd->p[2] >= 1 && pd->p[0] <= GEN_MAXP &&
                             pd->p[1] <= GEN_MAXP && pd->p[2] <= GEN_MAXP && pd->nnode <= GEN_MAXN && pd->ng >= 1 &&
                             pd->ng <= MAX_NG;
        if (!fixed_kernel_available(pd->p[0], pd->p[1], pd->p[2], pd->ng) && !general)
            return set_error(YETI_ERR_UNSUPPORTED_DEGREE, "shape gradient: no kernel for degrees (%d,%d,%d), ng=%d",
                             pd->p[0], pd->p[1], pd->p[2], pd->ng);
    }
    int rc = vib_setup(h);
    if (rc) return rc;
    for (int32_t k0 = 0; k0 < npair; k0 += VIB_MAXF) {
        GradFields gf{};
        gf.f0 = f0;
        gf.fk = fk;
        gf.nk = npair;
        gf.k0 = k0;
        gf.nf = std::min<int32_t>(VIB_MAXF, npair - k0);
        for (int f = 0; f < gf.nf && vals; ++f) gf.vals[f] = vals[k0 + f];
        int64_t ebase = 0, mbase = 0;
        for (auto *pd : h->patches) {
            if (!pd->u1 || pd->n_active == 0) continue;
            gf.rho = pd->rho;
            rc = kind == GRAD_MODES   ? launch_grad_kind<GRAD_MODES>(h, *pd, gf, ebase, mbase, st)
                 : kind == GRAD_PAIRS ? launch_grad_kind<GRAD_PAIRS>(h, *pd, gf, ebase, mbase, st)
                                      : launch_grad_kind<GRAD_VOLUME>(h, *pd, gf, ebase, mbase, st);
            if (rc) return rc;
            ebase += (int64_t)pd->n_active * pd->nnode;
            mbase += grad_slots(*pd);
        }
        double *mass = mass_out ? mass_out : h->vib_mass.p;
        if (normalize || mass_out) {   // no active element: zero mass, as the reference's empty sum
            hipLaunchKernelGGL(grad_mass_kernel, dim3(gf.nf), dim3(256), 0, st, (const double *)h->vib_em.p, h->vib_nslot,
                               mass);
            YETI_HIP(hipGetLastError());
        }
        // a bounded grid: one of 2^32 threads or more would drop all but the remainder
        const unsigned blocks = (unsigned)std::min<int64_t>((3 * gf.nf * (int64_t)h->nb_cp + 255) / 256, 65536);
        hipLaunchKernelGGL(grad_gather_kernel, dim3(blocks), dim3(256), 0, st, h->nb_cp, (const int32_t *)h->vib_ptr.p,
                           (const int32_t *)h->vib_ent.p, (const double *)h->vib_eg.p, gf.nf,
                           normalize ? (const double *)mass : (const double *)nullptr, scale, k0, npair, out);
        YETI_HIP(hipGetLastError());
    }
    return 0;
}

// -d(u^T K u)/dX (3 per CP, COORDS3D order): eigenvalue 0, the sums scaled by -1 and not
// normalised. u is dof-interleaved (3 cp + c), the (1, 3, nb_cp) column-major layout of one field.
static int run_strain_energy_grad(yeti_asm *h, const double *u, double *g, hipStream_t st) {
    return run_shape_grad(h, GRAD_MODES, nullptr, u, nullptr, 1, g, -1.0, false, nullptr, st);
}

// u^T F shape derivative of the face and body loads: g = 2 u^T dF/dX (3 per CP), gathered like F.
// reference_terms: only the terms gradLinElastWork_AN computes (centrifugal loads, their axis
// points read as it reads them; its face-load term is a stub, optim/gradUELMAT_solid.f90:463-477).
static int run_load_grad(yeti_asm *h, const double *u, double *g, hipStream_t st, bool reference_terms = false) {
    if (h->n_loaded_total > 0 && !h->grad_buf.p) YETI_HIP(h->grad_buf.alloc((size_t)h->n_loaded_total * 3 * RHS_MAXN));
    LoadTable lt;
    lt.jdltype = h->jdl.p;
    lt.adlmag = h->adlmag.p;
    lt.add_off = reference_terms ? h->add_off_ref.p : h->add_off.p;
    lt.only_type = reference_terms ? 101 : 0;
    lt.add_infos = h->add_infos.p;
    lt.elem_loads = h->elem_loads.p;
    lt.elem_loads_ptr = h->elem_loads_ptr.p;
    lt.nodal_dist = h->nodal_dist.p;
    lt.nb_n_dist = h->nb_n_dist;
    for (auto *pd : h->patches) {
        if (pd->n_loaded == 0) continue;
        RhsPatch rp;
        rp.coords = h->coords.p;
        rp.ien = pd->ien.p;
        rp.weight = pd->weight.p;
        rp.nijk = pd->nijk.p;
        for (int d = 0; d < 3; ++d) {
            rp.U[d] = pd->U[d];
            rp.p[d] = pd->p[d];
        }
        rp.elems = pd->loaded.p;
        rp.n_loaded = pd->n_loaded;
        rp.slot0 = pd->slot0;
        rp.ng = pd->ng;
        rp.rho = pd->rho;
        gauss_legendre(pd->ng, rp.g.x, rp.g.w);
        hipLaunchKernelGGL(elem_load_grad_kernel, dim3(pd->n_loaded), dim3(64), 0, st, rp, lt, u, h->grad_buf.p);
        YETI_HIP(hipGetLastError());
    }
    int blocks = (h->nb_cp + 255) / 256;
    hipLaunchKernelGGL(rhs_gather_kernel, dim3(blocks), dim3(256), 0, st, h->nb_cp, (const double *)nullptr,
                       h->cp_ptr.p, h->cp_ent.p, (const double *)h->grad_buf.p, g);
    YETI_HIP(hipGetLastError());
    return 0;
}

// ---- gradLinElastWork_AN: internal and external work gradients for given SOL and ADJ --------
// Fields f of an (nf, 3, nb_cp) column-major array sit at f + nf (3 cp + d).

// a[j] = ADJ[k, j] and back: out[k, j] = c g[j]
__global__ void field_extract_kernel(const double *adj, int32_t nadj, int32_t k, int64_t n3, double *a) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < n3) a[j] = adj[k + (int64_t)nadj * j];
}
__global__ void field_insert_kernel(const double *g, double c, int32_t nadj, int32_t k, int64_t n3, double *out) {
    const int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j < n3) out[k + (int64_t)nadj * j] = c * g[j];
}

// gradWint[k] = -ADJ_k^T (dK/dX) SOL and gradWext[k] = ADJ_k^T (dF/dX) over the active solid
// elements (gradtotalwork_fullAN.f90:17-300): the pairs (SOL, ADJ_k), VIB_MAXF per launch (the
// geometry and the state are evaluated once for them).
static int run_grad_lin_elast_work(yeti_asm *h, const double *sol, const double *adj, int32_t nadj, bool wint,
                                   bool wext, double *gint, double *gext, hipStream_t st) {
    const int64_t n3 = 3 * (int64_t)h->nb_cp;
    const unsigned blk = (unsigned)((n3 * nadj + 255) / 256), blk1 = (unsigned)((n3 + 255) / 256);
    if (wint) {
        int rc = run_shape_grad(h, GRAD_PAIRS, sol, adj, nullptr, nadj, gint, -1.0, false, nullptr, st);
        if (rc) return rc;
    } else {
        hipLaunchKernelGGL(fill_zero_kernel, dim3(blk), dim3(256), 0, st, gint, (int32_t *)nullptr, (int32_t *)nullptr,
                           n3 * nadj);
        YETI_HIP(hipGetLastError());
    }
    if (wext) {
        if (!h->ref_infos_ok)
            return set_error(YETI_ERR_INVALID_ARGUMENT,
                             "load_additionalInfos holds fewer than 6 values per centrifugal load");
        wext = h->any_centrifugal;   // without one the term is zero
    }
    if (wext) {
        if (h->gw_vec.n < (size_t)n3) {
            YETI_HIP(h->gw_vec.alloc(n3));
            YETI_HIP(h->gw_vec2.alloc(n3));
        }
        for (int k = 0; k < nadj; ++k) {
            hipLaunchKernelGGL(field_extract_kernel, dim3(blk1), dim3(256), 0, st, adj, nadj, k, n3, h->gw_vec.p);
            YETI_HIP(hipGetLastError());
            int rc = run_load_grad(h, h->gw_vec.p, h->gw_vec2.p, st, true);
            if (rc) return rc;
            // run_load_grad gives 2 a^T dF/dX
            hipLaunchKernelGGL(field_insert_kernel, dim3(blk1), dim3(256), 0, st, (const double *)h->gw_vec2.p, 0.5, nadj,
                               k, n3, gext);
            YETI_HIP(hipGetLastError());
        }
    } else {
        hipLaunchKernelGGL(fill_zero_kernel, dim3(blk), dim3(256), 0, st, gext, (int32_t *)nullptr, (int32_t *)nullptr,
                           n3 * nadj);
        YETI_HIP(hipGetLastError());
    }
    return 0;
}

static int run_rhs(yeti_asm *h, double *F, hipStream_t st) {
    LoadTable lt;
    lt.jdltype = h->jdl.p;
    lt.adlmag = h->adlmag.p;
    lt.add_off = h->add_off.p;
    lt.add_infos = h->add_infos.p;
    lt.elem_loads = h->elem_loads.p;
    lt.elem_loads_ptr = h->elem_loads_ptr.p;
    lt.nodal_dist = h->nodal_dist.p;
    lt.nb_n_dist = h->nb_n_dist;
    for (auto *pd : h->patches) {
        if (pd->n_loaded == 0) continue;
        RhsPatch rp;
        rp.coords = h->coords.p;
        rp.ien = pd->ien.p;
        rp.weight = pd->weight.p;
        rp.nijk = pd->nijk.p;
        for (int d = 0; d < 3; ++d) {
            rp.U[d] = pd->U[d];
            rp.p[d] = pd->p[d];
        }
        rp.ng = pd->ng;
        rp.rho = pd->rho;
        gauss_legendre(pd->ng, rp.g.x, rp.g.w);
        // a grid holds fewer than 2^32 threads: 2^23 elements of 256 per launch
        constexpr int32_t MOST = 1 << 23;
        for (int32_t e0 = 0; e0 < pd->n_loaded; e0 += MOST) {
            rp.elems = pd->loaded.p + e0;
            rp.n_loaded = std::min(MOST, pd->n_loaded - e0);
            rp.slot0 = pd->slot0 + e0;
            hipLaunchKernelGGL(elem_rhs_kernel, dim3(rp.n_loaded), dim3(256), rhs_smem_bytes(rp), st, rp, lt, h->rhs_buf.p);
            YETI_HIP(hipGetLastError());
        }
    }
    int blocks = (h->nb_cp + 255) / 256;
    hipLaunchKernelGGL(rhs_gather_kernel, dim3(blocks), dim3(256), 0, st, h->nb_cp, h->F_conc.p,
                       h->cp_ptr.p, h->cp_ent.p, h->rhs_buf.p, F);
    YETI_HIP(hipGetLastError());
    return 0;
}

static int create(const yeti_system_inputs *in, int layout, yeti_asm **out) {
    *out = nullptr;
    if (!in) return set_error(YETI_ERR_INVALID_ARGUMENT, "null inputs");
    if (layout != YETI_LAYOUT_PACKED && layout != YETI_LAYOUT_SLOTTED)
        return set_error(YETI_ERR_INVALID_ARGUMENT, "unknown layout %d", layout);
    // every id the set-up and the kernels gather through is checked here, before any device call
    if (int rc0 = validate_system_inputs(in, false)) return rc0;
    if ((int64_t)in->nb_cp * 3 > INT32_MAX)
        return set_error(YETI_ERR_SIZE_OVERFLOW, "dof ids exceed int32");
    std::vector<std::string> types;
    int rc = parse_elt_types(in, types);
    if (rc) return rc;

    auto *h = new yeti_asm();
    h->layout = layout;
    h->nb_cp = in->nb_cp;
    h->nb_dof_tot = in->nb_dof_tot;
    h->nb_data_cap = in->nb_data;
    h->nb_n_dist = std::max(1, in->nb_n_dist);
    auto fail = [&](int code) {
        delete h;
        return code;
    };
    if (hipError_t e = h->coords.upload(in->COORDS3D, 3 * (size_t)in->nb_cp); e != hipSuccess)
        return fail(set_error(YETI_ERR_DEVICE, "upload coords: %s", hipGetErrorString(e)));

    // load bookkeeping: which loads act on which (global, 1-based) element
    std::vector<int64_t> load_off(in->nb_load + 1, 0);
    for (int il = 0; il < in->nb_load; ++il) load_off[il + 1] = load_off[il] + in->load_target_nbelem[il];
    std::vector<std::vector<int32_t>> loads_of_elem(in->nb_elem);
    for (int il = 0; il < in->nb_load; ++il) {
        int t = in->JDLType[il];
        bool elem_load = (t > 9 && t < 100) || t == 101 || t == 102;
        if (!elem_load) continue;
        for (int64_t k = load_off[il]; k < load_off[il + 1]; ++k) {
            int64_t el = in->indDLoad[k];
            if (el >= 1 && el <= in->nb_elem) {
                auto &v = loads_of_elem[el - 1];
                if (v.empty() || v.back() != il) v.push_back(il);
            }
        }
    }

    int64_t kv = 0, woff = 0, ieoff = 0, eloff = 0, count = 0;
    std::vector<int32_t> elem_loads, elem_loads_ptr(1, 0);
    std::vector<std::pair<int32_t, int64_t>> cp_contrib;   // (cp0, entry)
    int32_t slot = 0;
    for (int ip = 0; ip < in->nb_patch; ++ip) {
        auto *pd = new PatchDev();
        h->patches.push_back(pd);
        for (int d = 0; d < 3; ++d) pd->p[d] = in->Jpqr[3 * ip + d];
        int nkv[3] = {in->Nkv[3 * ip], in->Nkv[3 * ip + 1], in->Nkv[3 * ip + 2]};
        pd->nnode = in->NNODE[ip];
        pd->nelem = in->nb_elem_patch[ip];
        int nn_geo = (pd->p[0] + 1) * (pd->p[1] + 1) * (pd->p[2] + 1);
        const std::string &ty = types[ip];
        pd->u1 = ty == "U1";
        bool u0 = ty == "U0";
        pd->ng = gauss_per_dir(in->NBINT[ip]);
        double E = in->MATERIAL_PROPERTIES[(int64_t)in->n_mat_props_max * ip];
        double nu = in->MATERIAL_PROPERTIES[(int64_t)in->n_mat_props_max * ip + 1];
        pd->lam = E * nu / ((1.0 + nu) * (1.0 - 2.0 * nu));
        pd->mu = E / (2.0 * (1.0 + nu));
        pd->rho = in->RHO[ip];
        const int64_t nde = 9LL * pd->nnode * (pd->nnode - 1) / 2 + 6LL * pd->nnode;
        // active elements and their slots
        std::vector<int32_t> act;
        std::vector<int64_t> offs;
        int64_t c = count;
        for (int e = 0; e < pd->nelem; ++e) {
            bool a = in->activeElement[eloff + e] == 1;
            if (layout == YETI_LAYOUT_SLOTTED) {
                if (a) {
                    act.push_back(e);
                    offs.push_back(count + (int64_t)e * nde);
                } else {
                    h->zero_ranges.push_back({count + (int64_t)e * nde, nde});
                }
            } else if (a) {
                act.push_back(e);
                offs.push_back(c);
                c += nde;
            }
        }
        int64_t next = layout == YETI_LAYOUT_SLOTTED ? count + (int64_t)pd->nelem * nde : c;
        if (!act.empty() && !pd->u1 && !u0)
            return fail(set_error(YETI_ERR_UNSUPPORTED_ELEMENT, "patch %d: element type %s is not supported",
                                  ip + 1, ty.c_str()));
        if (!act.empty()) {
            if (pd->nnode != nn_geo)
                return fail(set_error(YETI_ERR_INVALID_ARGUMENT, "patch %d: NNODE=%d but degrees give %d",
                                      ip + 1, pd->nnode, nn_geo));
            if (!kernel_available(pd->p[0], pd->p[1], pd->p[2], pd->ng))
                return fail(set_error(YETI_ERR_UNSUPPORTED_DEGREE,
                                      "patch %d: degrees (%d,%d,%d) with %d Gauss points per direction",
                                      ip + 1, pd->p[0], pd->p[1], pd->p[2], pd->ng));
        }
        // void elements (U0) keep their slots with zero values and real dof ids, as the
        // reference emits its zero AMATRX (build_system_elemStorage.f90:185-188,260-293)
        if (u0) pd->lam = pd->mu = 0.0;
        pd->u1 = pd->u1 || u0;
        pd->n_active = (int32_t)act.size();
        hipError_t e1 = hipSuccess;
        pd->tab_n = act.empty() ? 0 : std::max(std::max(pd->p[0], pd->p[1]), pd->p[2]) + 1;
        {
            std::vector<double> k, tab;
            size_t at[6] = {0, 0, 0, 0, 0, 0};
            for (int d = 0; d < 3; ++d) {
                at[d] = k.size();
                k.insert(k.end(), in->Ukv + kv, in->Ukv + kv + nkv[d]);
                kv += nkv[d];
            }
            double gx[MAX_NG], gw[MAX_NG];
            if (pd->tab_n > 0) gauss_legendre(pd->ng, gx, gw);
            for (int d = 0; d < 3 && pd->tab_n > 0; ++d) {
                basis_table(pd->p[d], k.data() + at[d], nkv[d], pd->tab_n, pd->ng, gx, tab);
                at[3 + d] = k.size();
                k.insert(k.end(), tab.begin(), tab.end());
            }
            e1 = pd->knots.upload(k.data(), k.size());
            for (int d = 0; d < 3; ++d) {
                pd->U[d] = pd->knots.p + at[d];
                if (pd->tab_n > 0) pd->tab[d] = pd->knots.p + at[3 + d];
            }
        }
        if (e1 == hipSuccess) e1 = pd->ien.upload(in->IEN + ieoff, (size_t)pd->nnode * pd->nelem);
        if (e1 == hipSuccess) e1 = pd->weight.upload(in->weight + woff, (size_t)nn_geo * pd->nelem);
        if (e1 == hipSuccess) e1 = pd->nijk.upload(in->Nijk + 3 * eloff, 3 * (size_t)pd->nelem);
        if (e1 == hipSuccess) e1 = pd->elems.upload(act.data(), act.size());
        if (e1 == hipSuccess) e1 = pd->offs.upload(offs.data(), offs.size());
        // loaded elements of this patch
        std::vector<int32_t> loaded;
        pd->slot0 = slot;
        if (pd->u1 && !u0) {
            for (int e = 0; e < pd->nelem; ++e)
                if (in->activeElement[eloff + e] == 1 && !loads_of_elem[eloff + e].empty()) loaded.push_back(e);
            if ((slot + (int64_t)loaded.size()) * RHS_MAXN > INT32_MAX)   // cp_ent holds int32 entries
                return fail(set_error(YETI_ERR_SIZE_OVERFLOW, "%lld loaded elements", slot + (long long)loaded.size()));
            for (int32_t e : loaded) {
                for (int il : loads_of_elem[eloff + e]) elem_loads.push_back(il);
                elem_loads_ptr.push_back((int32_t)elem_loads.size());
                for (int a = 0; a < pd->nnode; ++a) {
                    int32_t cp = in->IEN[ieoff + (int64_t)pd->nnode * e + a] - 1;
                    cp_contrib.push_back({cp, (int64_t)slot * RHS_MAXN + a});
                }
                ++slot;
            }
        }
        pd->n_loaded = (int32_t)loaded.size();
        if (e1 == hipSuccess) e1 = pd->loaded.upload(loaded.data(), loaded.size());
        if (e1 != hipSuccess) return fail(set_error(YETI_ERR_DEVICE, "upload patch %d: %s", ip + 1, hipGetErrorString(e1)));
        if (pd->u1 && pd->nnode > PATCH_MAXN)
            return fail(set_error(YETI_ERR_UNSUPPORTED_DEGREE, "patch %d: too many nodes", ip + 1));
        woff += (int64_t)nn_geo * pd->nelem;
        ieoff += (int64_t)pd->nnode * pd->nelem;
        eloff += pd->nelem;
        count = next;
    }
    h->nb_data = count;
    h->n_loaded_total = slot;
    for (auto *pd : h->patches) {
        h->v_ien.push_back(pd->ien.p);
        h->v_elems.push_back(pd->elems.p);
        h->v_offs.push_back(pd->offs.p);
        h->v_nnode.push_back(pd->nnode);
        h->v_nactive.push_back(pd->u1 ? pd->n_active : 0);
    }
    // concentrated loads: assignment in load order (build_system_elemStorage.f90:137-152)
    std::vector<double> Fc((size_t)in->nb_dof_tot, 0.0);
    for (int il = 0; il < in->nb_load; ++il) {
        int t = in->JDLType[il];
        if (t / 10 < 1)
            for (int64_t k = load_off[il]; k < load_off[il + 1]; ++k) {
                int64_t dof = (int64_t)(in->indDLoad[k] - 1) * 3 + t - 1;
                if (dof < 0 || dof >= in->nb_dof_tot)
                    return fail(set_error(YETI_ERR_INVALID_ARGUMENT, "concentrated load %d targets dof %lld",
                                          il + 1, (long long)dof));
                Fc[dof] = in->ADLMAG[il];
            }
    }
    // CP -> RHS entries, element order kept by a stable sort on the CP id
    std::stable_sort(cp_contrib.begin(), cp_contrib.end(),
                     [](const std::pair<int32_t, int64_t> &a, const std::pair<int32_t, int64_t> &b) {
                         return a.first < b.first;
                     });
    std::vector<int32_t> cp_ptr(in->nb_cp + 1, 0), cp_ent(cp_contrib.size());
    for (size_t k = 0; k < cp_contrib.size(); ++k) {
        cp_ptr[cp_contrib[k].first + 1]++;
        cp_ent[k] = (int32_t)cp_contrib[k].second;
    }
    for (int i = 0; i < in->nb_cp; ++i) cp_ptr[i + 1] += cp_ptr[i];
    std::vector<int32_t> jdl(in->JDLType, in->JDLType + in->nb_load);
    std::vector<int32_t> add_off(in->nb_load + 1, 0);
    for (int il = 0; il < in->nb_load; ++il) add_off[il + 1] = add_off[il] + in->nb_load_additionalInfos[il];
    // gradLinElastWork_AN reads the k-th centrifugal load's axis points A, B at values 6k+1..6k+6
    // of load_additionalInfos, whatever the other loads hold (its loadcount advances for type 101
    // only, optim/gradUELMAT_solid.f90:378-398)
    std::vector<int32_t> add_off_ref(in->nb_load + 1, 0);
    int64_t n101 = 0;
    for (int il = 0; il < in->nb_load; ++il)
        if (in->JDLType[il] == 101) add_off_ref[il] = (int32_t)(6 * n101++);
    h->any_centrifugal = n101 > 0;
    h->ref_infos_ok = 6 * n101 <= std::max<int64_t>(0, in->len_load_additionalInfos);
    if (in->nb_load > 0 && add_off[in->nb_load] > std::max<int64_t>(0, in->len_load_additionalInfos))
        return fail(set_error(YETI_ERR_INVALID_ARGUMENT, "load_additionalInfos holds %lld values, the loads name %d",
                              (long long)in->len_load_additionalInfos, add_off[in->nb_load]));
    // a nodal-distribution load (type 4) reads row `field` of nodal_dist at every CP of its elements
    for (int il = 0; il < in->nb_load; ++il) {
        const int t = in->JDLType[il];
        if (t < 10 || t > 99 || t % 10 != 4) continue;
        const int field = in->nb_load_additionalInfos[il] > 0 ? (int)in->load_additionalInfos[add_off[il]] : 0;
        if (field < 1 || field > std::max(1, in->nb_n_dist) || in->nb_cp_n_dist < in->nb_cp)
            return fail(set_error(YETI_ERR_INVALID_ARGUMENT,
                                  "load %d: distribution %d not in nodal_dist (%d x %d, %d control points)", il + 1,
                                  field, in->nb_n_dist, in->nb_cp_n_dist, in->nb_cp));
    }
    hipError_t e2 = h->F_conc.upload(Fc.data(), Fc.size());
    if (e2 == hipSuccess) e2 = h->jdl.upload(jdl.data(), jdl.size());
    if (e2 == hipSuccess) e2 = h->adlmag.upload(in->ADLMAG, in->nb_load);
    if (e2 == hipSuccess) e2 = h->add_off.upload(add_off.data(), add_off.size());
    if (e2 == hipSuccess) e2 = h->add_off_ref.upload(add_off_ref.data(), add_off_ref.size());
    if (e2 == hipSuccess) e2 = h->add_infos.upload(in->load_additionalInfos, std::max<int64_t>(1, in->len_load_additionalInfos));
    if (e2 == hipSuccess) e2 = h->elem_loads.upload(elem_loads.data(), elem_loads.size());
    if (e2 == hipSuccess) e2 = h->elem_loads_ptr.upload(elem_loads_ptr.data(), elem_loads_ptr.size());
    if (e2 == hipSuccess) e2 = h->cp_ptr.upload(cp_ptr.data(), cp_ptr.size());
    if (e2 == hipSuccess) e2 = h->cp_ent.upload(cp_ent.data(), cp_ent.size());
    if (e2 == hipSuccess)
        e2 = h->nodal_dist.upload(in->nodal_dist, (size_t)std::max(1, in->nb_n_dist) * std::max(1, in->nb_cp_n_dist));
    if (e2 == hipSuccess && slot > 0) e2 = h->rhs_buf.alloc((size_t)slot * 3 * RHS_MAXN);
    if (e2 != hipSuccess) return fail(set_error(YETI_ERR_DEVICE, "upload loads: %s", hipGetErrorString(e2)));
    *out = h;
    return 0;
}

struct AsmView {
    int32_t nb_cp;
    int32_t npatch;
    const int32_t *const *ien;
    const int32_t *const *elems;
    const int64_t *const *offs;
    const int32_t *nnode;
    const int32_t *n_active;
};

int asm_view(const yeti_asm *h, AsmView *v) {
    if (!h) return set_error(YETI_ERR_INVALID_ARGUMENT, "null assembly handle");
    v->nb_cp = h->nb_cp;
    v->npatch = (int32_t)h->patches.size();
    v->ien = h->v_ien.data();
    v->elems = h->v_elems.data();
    v->offs = h->v_offs.data();
    v->nnode = h->v_nnode.data();
    v->n_active = h->v_nactive.data();
    return 0;
}

}  // namespace yeti

// ------------------------------------------------------------------------------------------
// C ABI
extern "C" {

const char *yeti_last_error(void) { return yeti::last_error().c_str(); }

int32_t yeti_version(void) { return 0x000100; }

int32_t yeti_device_count(void) {
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess) return 0;
    return n;
}

int32_t yeti_asm_create(const yeti_system_inputs *in, int32_t layout, yeti_asm **out) {
    if (!out) return yeti::set_error(YETI_ERR_INVALID_ARGUMENT, "null handle pointer");
    yeti::last_error().clear();
    return yeti::create(in, layout, out);
}

int32_t yeti_asm_create_in(const yeti_system_inputs *in, int32_t layout, void *arena, size_t arena_bytes,
                           void *stream, yeti_asm **out, size_t *used) {
    if (!out) return yeti::set_error(YETI_ERR_INVALID_ARGUMENT, "null handle pointer");
    *out = nullptr;
    yeti::last_error().clear();
    yeti::Arena a;
    a.base = (char *)arena;
    a.size = arena ? arena_bytes : 0;
    yeti::AllocScope scope(&a, (hipStream_t)stream);
    yeti_asm *h = nullptr;
    int rc = yeti::create(in, layout, &h);
    if (used) *used = a.used;
    if (rc) return rc;
    if (!arena) {
        delete h;   // counting only
        return 0;
    }
    *out = h;
    return 0;
}

int64_t yeti_asm_nb_data(const yeti_asm *h) { return h ? h->nb_data : -1; }

int32_t yeti_asm_run_coo(yeti_asm *h, double *Kd, int32_t *Kr, int32_t *Kc, double *F, void *stream) {
    if (!h || !Kd || !Kr || !Kc || !F) return yeti::set_error(YETI_ERR_INVALID_ARGUMENT, "null argument");
    hipStream_t st = (hipStream_t)stream;
    int rc = yeti::run_elements(h, Kd, Kr, Kc, st);
    if (rc) return rc;
    return yeti::run_rhs(h, F, st);
}

int32_t yeti_asm_run_coo_matrix(yeti_asm *h, double *Kd, int32_t *Kr, int32_t *Kc, void *stream) {
    if (!h || !Kd || !Kr || !Kc) return yeti::set_error(YETI_ERR_INVALID_ARGUMENT, "null argument");
    return yeti::run_elements(h, Kd, Kr, Kc, (hipStream_t)stream);
}

int32_t yeti_asm_run_coo_values(yeti_asm *h, double *Kd, void *stream) {
    if (!h || !Kd) return yeti::set_error(YETI_ERR_INVALID_ARGUMENT, "null argument");
    return yeti::run_elements(h, Kd, nullptr, nullptr, (hipStream_t)stream);
}

int32_t yeti_asm_run_mass_coo(yeti_asm *h, double *Md, int32_t *Mr, int32_t *Mc, void *stream) {
    if (!h || !Md || (!Mr) != (!Mc)) return yeti::set_error(YETI_ERR_INVALID_ARGUMENT, "null argument");
    return yeti::run_mass(h, Md, Mr, Mc, (hipStream_t)stream);
}

int32_t yeti_asm_run_vib_grad(yeti_asm *h, const double *vect, const double *vals, int32_t nb_frq, double *gradV,
                              void *stream) {
    if (!h || !vect || !vals || !gradV || nb_frq < 1)
        return yeti::set_error(YETI_ERR_INVALID_ARGUMENT, "null argument or nb_frq < 1");
    return yeti::run_shape_grad(h, yeti::GRAD_MODES, nullptr, vect, vals, nb_frq, gradV, 1.0, true, nullptr,
                                (hipStream_t)stream);
}

int32_t yeti_asm_strain_energy_grad(yeti_asm *h, const double *u, double *g, void *stream) {
    if (!h || !u || !g) return yeti::set_error(YETI_ERR_INVALID_ARGUMENT, "null argument");
    return yeti::run_strain_energy_grad(h, u, g, (hipStream_t)stream);
}

int32_t yeti_asm_volume_grad(yeti_asm *h, double *vol, double *g, void *stream) {
    if (!h || !vol || !g) return yeti::set_error(YETI_ERR_INVALID_ARGUMENT, "null argument");
    return yeti::run_shape_grad(h, yeti::GRAD_VOLUME, nullptr, nullptr, nullptr, 1, g, 1.0, false, vol,
                                (hipStream_t)stream);
}

int32_t yeti_grad_lin_elast_work(yeti_asm *h, const double *SOL, const double *ADJ, int32_t nadj, int32_t computeWint,
                                 int32_t computeWext, double *gradWint, double *gradWext, void *stream) {
    if (!h || !SOL || !ADJ || !gradWint || !gradWext || nadj < 1)
        return yeti::set_error(YETI_ERR_INVALID_ARGUMENT, "null argument or nadj < 1");
    return yeti::run_grad_lin_elast_work(h, SOL, ADJ, nadj, computeWint != 0, computeWext != 0, gradWint, gradWext,
                                         (hipStream_t)stream);
}

int32_t yeti_asm_run_rhs(yeti_asm *h, double *F, void *stream) {
    if (!h || !F) return yeti::set_error(YETI_ERR_INVALID_ARGUMENT, "null argument");
    return yeti::run_rhs(h, F, (hipStream_t)stream);
}

int32_t yeti_asm_load_shape_grad(yeti_asm *h, const double *u, double *g, void *stream) {
    if (!h || !u || !g) return yeti::set_error(YETI_ERR_INVALID_ARGUMENT, "null argument");
    return yeti::run_load_grad(h, u, g, (hipStream_t)stream);
}

int32_t yeti_asm_update_coords(yeti_asm *h, const double *coords, void *stream) {
    if (!h || !coords) return yeti::set_error(YETI_ERR_INVALID_ARGUMENT, "null argument");
    YETI_HIP(hipMemcpyAsync(h->coords.p, coords, 3 * sizeof(double) * (size_t)h->nb_cp, hipMemcpyDeviceToDevice,
                            (hipStream_t)stream));
    return 0;
}

int32_t yeti_asm_set_timing(yeti_asm *h, int32_t on) {
    if (!h) return yeti::set_error(YETI_ERR_INVALID_ARGUMENT, "null handle");
    h->timing = on != 0;
    return 0;
}

int32_t yeti_asm_kernel_times(yeti_asm *h, float *ms, int32_t cap, int32_t *n) {
    if (!h || !n) return yeti::set_error(YETI_ERR_INVALID_ARGUMENT, "null argument");
    *n = h->ev_used;
    for (int k = 0; k < h->ev_used && k < cap; ++k) {
        YETI_HIP(hipEventSynchronize(h->ev[2 * k + 1]));
        YETI_HIP(hipEventElapsedTime(&ms[k], h->ev[2 * k], h->ev[2 * k + 1]));
    }
    return 0;
}

void yeti_asm_destroy(yeti_asm *h) { delete h; }

int32_t yeti_sys_linmat_lindef_static(const yeti_system_inputs *in, int32_t layout, double *Kdata,
                                      int32_t *Krow, int32_t *Kcol, double *F) {
    if (!in || !Kdata || !Krow || !Kcol || !F) return yeti::set_error(YETI_ERR_INVALID_ARGUMENT, "null argument");
    yeti::last_error().clear();
    yeti_asm *h = nullptr;
    int rc = yeti::create(in, layout, &h);
    if (rc) return rc;
    int64_t nd = h->nb_data;
    if (nd > in->nb_data) {
        yeti_asm_destroy(h);
        return yeti::set_error(YETI_ERR_SIZE_OVERFLOW, "nb_data=%lld but the layout needs %lld",
                               (long long)in->nb_data, (long long)nd);
    }
    yeti::DevBuf<double> dK, dF;
    yeti::DevBuf<int32_t> dR, dC;
    hipError_t e = dK.alloc(std::max<int64_t>(nd, 1));
    if (e == hipSuccess) e = dR.alloc(std::max<int64_t>(nd, 1));
    if (e == hipSuccess) e = dC.alloc(std::max<int64_t>(nd, 1));
    if (e == hipSuccess) e = dF.alloc(std::max(in->nb_dof_tot, 1));
    if (e != hipSuccess) {
        yeti_asm_destroy(h);
        return yeti::set_error(YETI_ERR_DEVICE, "device allocation: %s", hipGetErrorString(e));
    }
    rc = yeti_asm_run_coo(h, dK.p, dR.p, dC.p, dF.p, nullptr);
    yeti_asm_destroy(h);
    if (rc) return rc;
    YETI_HIP(hipMemcpy(Kdata, dK.p, nd * sizeof(double), hipMemcpyDeviceToHost));
    YETI_HIP(hipMemcpy(Krow, dR.p, nd * sizeof(int32_t), hipMemcpyDeviceToHost));
    YETI_HIP(hipMemcpy(Kcol, dC.p, nd * sizeof(int32_t), hipMemcpyDeviceToHost));
    YETI_HIP(hipMemcpy(F, dF.p, in->nb_dof_tot * sizeof(double), hipMemcpyDeviceToHost));
    // entries beyond what the layout uses stay zero, as the reference's zero-initialised arrays
    if (in->nb_data > nd) {
        std::memset(Kdata + nd, 0, (in->nb_data - nd) * sizeof(double));
        std::memset(Krow + nd, 0, (in->nb_data - nd) * sizeof(int32_t));
        std::memset(Kcol + nd, 0, (in->nb_data - nd) * sizeof(int32_t));
    }
    return 0;
}

}  // extern "C"
