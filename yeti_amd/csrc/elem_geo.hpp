// elem_geo.hpp -- geometry pass of the element stiffness kernels of degrees 3 and 4 (included by
// assembly.hip, which defines GaussRule and bspline_ders before including it): the Jacobian of the
// NURBS map (shap.f90:94-178) reduced to 12 numbers per Gauss point, written to HBM for
// elem_p3_kernel and elem_general_kernel<8, 0>.
#pragma once

typedef double f64x2 __attribute__((ext_vector_type(2)));

constexpr int ELEM_NGEO = 12;   // per Gauss point: A[m][c] (9), dW/dxi_m / W (3)

template <int P, int NG>
struct ElemCfg {
    static constexpr int NP1 = P + 1;
    static constexpr int NN = NP1 * NP1 * NP1;          // nodes (CPs) per element
    static constexpr int NQ = NG * NG * NG;             // Gauss points per element
    // the record of an element: 12 geometry values per Gauss point ([v][q]); at p = 3 then the 1D basis
    // tables B, dB ([which][d][g][i]), the node weights and the nodes' dof bases 3 (IEN - 1) (int32,
    // from double offset DOFOFF), which elem_general_kernel fetches itself
    static constexpr bool NODES = P == 3;
    static constexpr int NTAB = 2 * 3 * NG * NP1;
    static constexpr int64_t DOFOFF = (int64_t)ELEM_NGEO * NQ + NTAB + NN;
    static constexpr int64_t REC = NODES ? DOFOFF + (NN + 1) / 2 : (int64_t)ELEM_NGEO * NQ;
};

struct PatchArgs {
    const double *coords;     // (3, nb_cp)
    const int32_t *ien;       // (nnode, nelem_patch), 1-based
    const double *weight;     // (nnode, nelem_patch)
    const int32_t *nijk;      // (3, nelem_patch), 1-based spans
    const double *U0, *U1, *U2;  // knot vectors
    const int32_t *elems;     // active elements of this launch (patch-local 0-based)
    const int64_t *offs;      // COO offset per active element
    int32_t n_active;
    double lam, mu;
    GaussRule g;
};

// ---------------------------------------------------------------------------------------
// Geometry pass: per active element gi a record of REC doubles at geo + gi REC: for Gauss point
// q, [v NQ + q] with v = 3 m + c: A[m][c] = sqrt(w |det J|) / W dxi_m/dx_c; v = 9 + m:
// dW/dxi_m / W; at p = 3 then the element's 1D basis tables (values and derivatives at the abscissae,
// reversed local index), its node weights and its nodes' dof bases. J is the derivative with respect
// to the knot parameters (shap.f90:133-153); w |det J| includes the parent-to-parameter factors
// (shap.f90:156-178) and the Gauss weights (UELMAT.f90:118-119).
// One wave per element, 4 per workgroup. The 16 sums a Gauss point needs (W, dW/dxi_m, and
// sum w x_c R and its xi derivatives, before the division by W) are tensor-product contractions
// of the four nodal quantities (w, w x, w y, w z), evaluated by sum factorisation through LDS:
// along xi_0 (values and derivatives at the NG abscissae), then xi_1, then xi_2, one lane per
// Gauss point in the last stage (NP1^3 NG + ... multiply-adds per quantity instead of NP1^3 NG^3).
template <int P, int NG>
__global__ void __launch_bounds__(256) elem_geo_kernel(PatchArgs pa, double *__restrict__ geo) {
    using C = ElemCfg<P, NG>;
    constexpr int NP1 = C::NP1, NN = C::NN, NQ = C::NQ;
    constexpr int EPB = 4;                              // elements per workgroup, one per wave
    constexpr int NT1 = 4 * 2 * NG * NP1 * NP1;         // stage 0: [quantity][B | dB][g0][k][j]
    constexpr int NT2 = 4 * 3 * NG * NG * NP1;          // stage 1: [quantity][v][g0][g1][k]
    __shared__ double cp[EPB][4][NN];                   // (w, w x, w y, w z) per node
    __shared__ double tab[EPB][3][2][NG][NP1];          // [d][B | dB][g][i], i <-> basis P - i
    __shared__ double hh[EPB][3];                       // half span per direction
    __shared__ double T1[EPB][NT1];
    __shared__ double T2[EPB][NT2];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t gi = (int64_t)blockIdx.x * EPB + wv;
    const bool act = gi < pa.n_active;   // wave-uniform; inactive waves still meet the barriers
    const int e = act ? pa.elems[gi] : 0;
    double *rec = geo + gi * C::REC;
    if (act) {
        for (int a = lane; a < NN; a += 64) {
            const int32_t cp1 = pa.ien[(int64_t)NN * e + a];
            const double *xp = pa.coords + 3 * (int64_t)(cp1 - 1);
            const double w = pa.weight[(int64_t)NN * e + a];
            if (C::NODES) {
                reinterpret_cast<int32_t *>(rec + C::DOFOFF)[a] = 3 * (cp1 - 1);
                rec[ELEM_NGEO * NQ + C::NTAB + a] = w;
            }
            cp[wv][0][a] = w;
            cp[wv][1][a] = w * xp[0];
            cp[wv][2][a] = w * xp[1];
            cp[wv][3][a] = w * xp[2];
        }
        if (lane < 3 * NG) {   // 1D bases of direction d at abscissa g
            const int d = lane / NG, g = lane - d * NG;
            const double *U = d == 0 ? pa.U0 : d == 1 ? pa.U1 : pa.U2;
            const int span1 = pa.nijk[3 * (int64_t)e + d];
            const double u0 = U[span1 - 1], u1 = U[span1];
            const double u = ((u1 - u0) * pa.g.x[g] + (u1 + u0)) * 0.5;
            double N[NP1], dN[NP1];
            bspline_ders<P>(span1 - 1, u, U, N, dN);
#pragma unroll
            for (int i = 0; i < NP1; ++i) {   // local index i <-> basis function P - i
                tab[wv][d][0][g][i] = N[P - i];
                tab[wv][d][1][g][i] = dN[P - i];
                if (C::NODES) {
                    double *tb = rec + ELEM_NGEO * NQ + (d * NG + g) * NP1;
                    tb[i] = N[P - i];
                    tb[3 * NG * NP1 + i] = dN[P - i];
                }
            }
            if (g == 0) hh[wv][d] = 0.5 * (u1 - u0);
        }
    }
    __syncthreads();
    if (act) {   // stage 0: contract i (xi_0)
        for (int o = lane; o < NT1; o += 64) {
            const int j = o % NP1, k = (o / NP1) % NP1, g0 = (o / (NP1 * NP1)) % NG, v = (o / (NP1 * NP1 * NG)) % 2,
                      qn = o / (NP1 * NP1 * NG * 2);
            double s = 0.0;
#pragma unroll
            for (int i = 0; i < NP1; ++i) s += tab[wv][0][v][g0][i] * cp[wv][qn][i + NP1 * (j + NP1 * k)];
            T1[wv][o] = s;
        }
    }
    __syncthreads();
    if (act) {   // stage 1: contract j (xi_1); v = 0: B0 B1, 1: dB0 B1, 2: B0 dB1
        for (int o = lane; o < NT2; o += 64) {
            const int k = o % NP1, g1 = (o / NP1) % NG, g0 = (o / (NP1 * NG)) % NG, v = (o / (NP1 * NG * NG)) % 3,
                      qn = o / (NP1 * NG * NG * 3);
            const double *t1 = &T1[wv][(((qn * 2 + (v == 1 ? 1 : 0)) * NG + g0) * NP1 + k) * NP1];
            double s = 0.0;
#pragma unroll
            for (int j = 0; j < NP1; ++j) s += t1[j] * tab[wv][1][v == 2 ? 1 : 0][g1][j];
            T2[wv][o] = s;
        }
    }
    __syncthreads();
    if (!act) return;
    // stage 2: contract k (xi_2), one lane per Gauss point, and the point's Jacobian work
    for (int q = lane; q < NQ; q += 64) {
        const int g0 = q % NG, g1 = (q / NG) % NG, g2 = q / (NG * NG);
        double s[16];   // 0: W, 1-3: dW/dxi_m, 4 + c: sum w x_c R, 7 + 3 c + m: its xi_m derivative
#pragma unroll
        for (int qn = 0; qn < 4; ++qn) {
            double val = 0.0, d0 = 0.0, d1 = 0.0, d2 = 0.0;
            const double *t2 = &T2[wv][((qn * 3) * NG * NG + g0 * NG + g1) * NP1];
#pragma unroll
            for (int k = 0; k < NP1; ++k) {
                const double bz = tab[wv][2][0][g2][k], dz = tab[wv][2][1][g2][k];
                const double t0 = t2[k];
                val += t0 * bz;
                d2 += t0 * dz;
                d0 += t2[NG * NG * NP1 + k] * bz;
                d1 += t2[2 * NG * NG * NP1 + k] * bz;
            }
            if (qn == 0) {
                s[0] = val;
                s[1] = d0;
                s[2] = d1;
                s[3] = d2;
            } else {
                s[3 + qn] = val;
                s[7 + 3 * (qn - 1) + 0] = d0;
                s[7 + 3 * (qn - 1) + 1] = d1;
                s[7 + 3 * (qn - 1) + 2] = d2;
            }
        }
        const double Wi = 1.0 / s[0];
        const double dw[3] = {s[1] * Wi, s[2] * Wi, s[3] * Wi};
        double J[3][3];
#pragma unroll
        for (int r2 = 0; r2 < 3; ++r2)
#pragma unroll
            for (int c = 0; c < 3; ++c) J[r2][c] = (s[7 + 3 * r2 + c] - s[4 + r2] * dw[c]) * Wi;
        const double m00 = J[1][1] * J[2][2] - J[1][2] * J[2][1];
        const double m01 = J[1][2] * J[2][0] - J[1][0] * J[2][2];
        const double m02 = J[1][0] * J[2][1] - J[1][1] * J[2][0];
        const double det = J[0][0] * m00 + J[0][1] * m01 + J[0][2] * m02;
        const double om = pa.g.w[g0] * pa.g.w[g1] * pa.g.w[g2] * fabs(det * hh[wv][0] * hh[wv][1] * hh[wv][2]);
        const double f = sqrt(om) * Wi / det;
        double A[9];   // A[3 m + c] = f * (adj J)[m][c]
        A[0] = m00 * f;
        A[1] = (J[0][2] * J[2][1] - J[0][1] * J[2][2]) * f;
        A[2] = (J[0][1] * J[1][2] - J[0][2] * J[1][1]) * f;
        A[3] = m01 * f;
        A[4] = (J[0][0] * J[2][2] - J[0][2] * J[2][0]) * f;
        A[5] = (J[0][2] * J[1][0] - J[0][0] * J[1][2]) * f;
        A[6] = m02 * f;
        A[7] = (J[0][1] * J[2][0] - J[0][0] * J[2][1]) * f;
        A[8] = (J[0][0] * J[1][1] - J[0][1] * J[1][0]) * f;
        double *out = rec + q;
#pragma unroll
        for (int v = 0; v < 9; ++v) out[v * NQ] = A[v];
#pragma unroll
        for (int m = 0; m < 3; ++m) out[(9 + m) * NQ] = dw[m];
    }
}
