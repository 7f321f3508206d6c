// shape_grad.hpp -- element kernels of the shape gradients (included by assembly.hip, which
// defines PatchArgs, GaussRule and f64x2).
//
// For a pair of displacement fields (u, v), an eigenvalue lam and the density rho, an element adds
// to its node a
//   g_a[m] = sum_q dv_q [ (sig_u : grad v - lam rho u.v) dR_a/dx_m
//                         - sum_ik (sig_u,ik dv_i/dx_m + sig_v,ik du_i/dx_m) dR_a/dx_k ],
// the derivative of int sig(u) : eps(v) - lam rho u.v with respect to control point a, and
// rho u.v dv to the pair's mass. The callers use it three ways (GradKind):
//   GRAD_MODES   v = u, one pair per field: the natural-frequency gradient
//                (gradvibration_fullAN.f:22-189 with gradUELMASSMAT1, gradUELMASSMAT_solid.f:22-332,
//                which write it in the covariant basis) and, with lam = 0, the strain energy's;
//   GRAD_PAIRS   u = field 0, v = fields 1, 2, ...: the internal work of a state and its adjoints
//                (gradUELMAT1adj, optim/gradUELMAT_solid.f90:18-479);
//   GRAD_VOLUME  no field, the tensor dv I and the mass dv: volume and its gradient
//                (optim/gradvolume.f90:16-355).
#pragma once

enum GradKind { GRAD_MODES = 0, GRAD_PAIRS = 1, GRAD_VOLUME = 2 };

constexpr int VIB_MAXF = 4;      // pairs per launch

struct GradFields {
    const double *f0, *fk;       // GRAD_PAIRS: field 0, and the others; GRAD_MODES: fk
    int32_t nk, k0, nf;          // fields k0 .. k0 + nf - 1 of the nk interleaved in fk
    double vals[VIB_MAXF];       // eigenvalues
    double rho;
};

// 1D basis tables of a patch per knot span: B and dB at the Gauss points in local node order
// ([B | dB][g][i], zero for i above the direction's degree) and half the span's length.
template <int N, int Q>
constexpr int grad_rec() { return (2 * Q * N + 2) / 2 * 2; }

// tables live in the constant address space: with a wave-uniform element they are scalar loads
typedef const __attribute__((address_space(4))) double *GradTab;

struct GradArgs {
    const double *coords;
    const int32_t *ien;
    const double *weight;
    const int32_t *nijk;
    const double *tab[3];
    const int32_t *elems;
    int32_t n_active;
    int32_t n[3];                // nodes per direction (at most N)
    double lam, mu;
    GaussRule g;
    GradFields f;
    double *eg;                  // [element-node entry][pair][3]
    int64_t ebase;
    double *em;                  // [workgroup][VIB_MAXF]
};

// Sum factorisation per element, N >= degrees + 1, Q Gauss points per direction. A wave carries
// EPW elements, LPE lanes each, and never meets a barrier: what its lanes exchange goes through its
// own LDS. A quantity (4 for the geometry: w, w x; 3 for a field: w u) is contracted along xi_0
// (one lane per node line), xi_1, and xi_2 (one lane per Gauss point, values and derivatives in
// registers); the point's tensor is then carried back the same way. Tables of a one-element wave
// are read with scalar loads. LDS strides are odd, so that lanes on neighbouring lines meet
// different banks. Bound by vector issue at 3 waves per SIMD (registers): about 1100 instructions
// per field and wave, 420 of them FP64. Against one workgroup per element that multiplied every
// node with every point in chunks of 16 points and 5 barriers each: 33x29x26 p=3 with 4 modes
// 4044 -> 257 us, 47x31x22 p=2 with a state and two adjoints 1078 -> 131 us, volume 1078 -> 48 us.
template <int N, int Q>
struct Grad {
    static constexpr int NNP = N * N * N, NQ = Q * Q * Q;
    static constexpr int EPW = N == 2 ? 8 : N == 3 ? 2 : 1;   // elements per wave
    static constexpr int LPE = 64 / EPW;                      // lanes per element
    static constexpr int PPL = (NQ + LPE - 1) / LPE;          // points per lane
    static constexpr int WPB = N == 5 ? 2 : 4;                // waves per workgroup (LDS: three workgroups per CU)
    static constexpr int S0 = (4 * N * N) | 1;                // nodes       [i][line, quantity]
    static constexpr int S1 = (4 * N * Q) | 1;                // after xi_0  [B | dB][j][..]
    static constexpr int S2 = (4 * Q * Q) | 1;                // after xi_1  [v, d0, d1][k][..]
    static constexpr int S3 = (3 * Q * Q) | 1;                // points      [g2][v, d0, d1, d2][..]
    static constexpr int S4 = (3 * Q * N) | 1;                // back xi_2   [g1][3][..]
    static constexpr int S5 = (3 * N * N) | 1;                // back xi_1   [g0][2][..]
    static constexpr int cmax(int a, int b) { return a > b ? a : b; }
    // the stages alternate between two buffers
    static constexpr int NA = cmax(cmax(N * S0, 3 * N * S2), cmax(3 * Q * S4, 3 * NNP));
    static constexpr int NB = cmax(cmax(2 * N * S1, 4 * Q * S3), 2 * Q * S5);
    static constexpr int NEL = NA + NB + NNP;                 // + the node weights
};

template <int N, int Q, int KIND>
__global__ void __launch_bounds__((64 * Grad<N, Q>::WPB)) __attribute__((amdgpu_waves_per_eu(N == 5 ? 1 : 3)))
shape_grad_kernel(GradArgs ga) {
    using C = Grad<N, Q>;
    constexpr int LPE = C::LPE, PPL = C::PPL, NQ = C::NQ, NNP = C::NNP, REC = grad_rec<N, Q>();
    __shared__ double sm[C::WPB * C::EPW][C::NEL];
    __shared__ double msum[C::WPB][VIB_MAXF];
    const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int sub = lane / LPE, ll = lane % LPE;
    double *bufA = sm[wv * C::EPW + sub], *bufB = bufA + C::NA, *sw = bufB + C::NB;
    const int n0 = ga.n[0], n1 = ga.n[1], n2 = ga.n[2], nn = n0 * n1 * n2;
    const int nout = KIND == GRAD_VOLUME ? 1 : ga.f.nf;
    double macc[VIB_MAXF] = {0.0, 0.0, 0.0, 0.0};
    const int64_t stride = (int64_t)gridDim.x * C::WPB * C::EPW;
    for (int64_t gw = ((int64_t)blockIdx.x * C::WPB + wv) * C::EPW; gw < ga.n_active; gw += stride) {
        // a wave's last elements may be past the end: they repeat the last one and store nothing
        const int64_t gi = gw + sub;
        const bool act = gi < ga.n_active;
        int e = ga.elems[act ? gi : (int64_t)ga.n_active - 1];
        if (C::EPW == 1) e = __builtin_amdgcn_readfirstlane(e);
        GradTab tb[3];
        double half = 1.0;
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            int s = ga.nijk[3 * (int64_t)e + d] - 1;
            if (C::EPW == 1) s = __builtin_amdgcn_readfirstlane(s);
            tb[d] = (GradTab)(ga.tab[d] + (int64_t)s * REC);
            half *= tb[d][2 * Q * N];
        }
        // the nodes: their ids stay in registers for the fields
        constexpr int NPL = (NNP + LPE - 1) / LPE;
        int64_t cp[NPL];
        // positions and fields are taken relative to the element's node 0 (held by its first lane):
        // derivatives do not see the difference, and no digits go into it
        auto origin = [&](double v) { return __shfl(v, lane - ll, 64); };
        double xo[3];
        wave_lds_sync();
#pragma unroll
        for (int r = 0; r < NPL; ++r) {
            const int pn = ll + LPE * r, i = pn % N, j = (pn / N) % N, k = pn / (N * N);
            const bool in = pn < NNP && i < n0 && j < n1 && k < n2;
            cp[r] = -1;
            double w = 0.0, x0 = 0.0, x1 = 0.0, x2 = 0.0;
            if (in) {
                const int a = i + n0 * (j + n1 * k);
                cp[r] = (int64_t)ga.ien[(int64_t)nn * e + a] - 1;
                w = ga.weight[(int64_t)nn * e + a];
                x0 = ga.coords[3 * cp[r]];
                x1 = ga.coords[3 * cp[r] + 1];
                x2 = ga.coords[3 * cp[r] + 2];
            }
            if (r == 0) {
                xo[0] = origin(x0);
                xo[1] = origin(x1);
                xo[2] = origin(x2);
            }
            x0 = w * (x0 - xo[0]);
            x1 = w * (x1 - xo[1]);
            x2 = w * (x2 - xo[2]);
            if (pn < NNP) {
                double *p = bufA + i * C::S0 + j + N * k;
                p[0] = w;
                p[N * N] = x0;
                p[2 * N * N] = x1;
                p[3 * N * N] = x2;
                sw[pn] = w;
            }
        }
        wave_lds_sync();
        // contractions of NQT quantities along xi_0 (bufA -> bufB) and xi_1 (bufB -> bufA)
        auto forward = [&](auto nqt) {
            constexpr int NQT = decltype(nqt)::value;
            for (int t = ll; t < NQT * N * N; t += LPE) {
                const int jk = t % (N * N), j = jk % N, k = jk / N, m = t / (N * N);
                double x[N];
#pragma unroll
                for (int i = 0; i < N; ++i) x[i] = bufA[i * C::S0 + t];
#pragma unroll
                for (int g = 0; g < Q; ++g) {
                    double v = 0.0, d = 0.0;
#pragma unroll
                    for (int i = 0; i < N; ++i) {
                        v += x[i] * tb[0][g * N + i];
                        d += x[i] * tb[0][Q * N + g * N + i];
                    }
                    bufB[j * C::S1 + g + Q * k + Q * N * m] = v;
                    bufB[(N + j) * C::S1 + g + Q * k + Q * N * m] = d;
                }
            }
            wave_lds_sync();
            for (int t = ll; t < NQT * Q * N; t += LPE) {
                const int g0 = t % Q, k = (t / Q) % N, m = t / (Q * N);
                double x[N], y[N];
#pragma unroll
                for (int j = 0; j < N; ++j) {
                    x[j] = bufB[j * C::S1 + t];
                    y[j] = bufB[(N + j) * C::S1 + t];
                }
#pragma unroll
                for (int g = 0; g < Q; ++g) {
                    double v = 0.0, d0 = 0.0, d1 = 0.0;
#pragma unroll
                    for (int j = 0; j < N; ++j) {
                        const double b = tb[1][g * N + j];
                        v += x[j] * b;
                        d0 += y[j] * b;
                        d1 += x[j] * tb[1][Q * N + g * N + j];
                    }
                    double *p = bufA + k * C::S2 + g0 + Q * g + Q * Q * m;
                    p[0] = v;
                    p[N * C::S2] = d0;
                    p[2 * N * C::S2] = d1;
                }
            }
            wave_lds_sync();
        };
        // the lane's points: tables along xi_2, and the value and derivatives of quantity m there
        double bz[PPL][N], dz[PPL][N];
#pragma unroll
        for (int r = 0; r < PPL; ++r) {
            const int q = min(ll + LPE * r, NQ - 1), g2 = q / (Q * Q);
#pragma unroll
            for (int k = 0; k < N; ++k) {
                bz[r][k] = tb[2][g2 * N + k];
                dz[r][k] = tb[2][Q * N + g2 * N + k];
            }
        }
        auto at_point = [&](int r, int m, double *o) {   // o: value, d/dxi_0, d/dxi_1, d/dxi_2
            const int q = min(ll + LPE * r, NQ - 1);
            const double *p = bufA + q % (Q * Q) + Q * Q * m;
            o[0] = o[1] = o[2] = o[3] = 0.0;
#pragma unroll
            for (int k = 0; k < N; ++k) {
                const double v = p[k * C::S2];
                o[0] += v * bz[r][k];
                o[3] += v * dz[r][k];
                o[1] += p[(N + k) * C::S2] * bz[r][k];
                o[2] += p[(2 * N + k) * C::S2] * bz[r][k];
            }
        };
        forward(std::integral_constant<int, 4>{});
        double A[PPL][9], Wi[PPL], dw[PPL][3], dv[PPL];   // A[3 m + c] = dxi_m / dx_c
#pragma unroll
        for (int r = 0; r < PPL; ++r) {
            const int q = min(ll + LPE * r, NQ - 1);
            double s[4], J[3][3];
            at_point(r, 0, s);
            Wi[r] = 1.0 / s[0];
#pragma unroll
            for (int m = 0; m < 3; ++m) dw[r][m] = s[1 + m] * Wi[r];
#pragma unroll
            for (int c = 0; c < 3; ++c) {
                at_point(r, 1 + c, s);
#pragma unroll
                for (int m = 0; m < 3; ++m) J[c][m] = (s[1 + m] - s[0] * dw[r][m]) * Wi[r];
            }
            A[r][0] = J[1][1] * J[2][2] - J[1][2] * J[2][1];
            A[r][1] = J[0][2] * J[2][1] - J[0][1] * J[2][2];
            A[r][2] = J[0][1] * J[1][2] - J[0][2] * J[1][1];
            A[r][3] = J[1][2] * J[2][0] - J[1][0] * J[2][2];
            A[r][4] = J[0][0] * J[2][2] - J[0][2] * J[2][0];
            A[r][5] = J[0][2] * J[1][0] - J[0][0] * J[1][2];
            A[r][6] = J[1][0] * J[2][1] - J[1][1] * J[2][0];
            A[r][7] = J[0][1] * J[2][0] - J[0][0] * J[2][1];
            A[r][8] = J[0][0] * J[1][1] - J[0][1] * J[1][0];
            const double det = J[0][0] * A[r][0] + J[0][1] * A[r][3] + J[0][2] * A[r][6];
            const double di = 1.0 / det;
#pragma unroll
            for (int c = 0; c < 9; ++c) A[r][c] *= di;
            // 0 at the lanes past the last point, which repeat it
            dv[r] = ll + LPE * r < NQ ? ga.g.w[q % Q] * ga.g.w[(q / Q) % Q] * ga.g.w[q / (Q * Q)] * (det * half) : 0.0;
        }
        // field at the points: u and D[i][k] = du_i / dx_k
        auto field = [&](const double *f, int fs, double (*u)[3], double (*D)[3][3]) {
            double uo[3];
            wave_lds_sync();
#pragma unroll
            for (int r = 0; r < NPL; ++r) {
                const int pn = ll + LPE * r, i = pn % N, jk = pn / N;
                double x[3];
#pragma unroll
                for (int c = 0; c < 3; ++c) {
                    x[c] = cp[r] >= 0 ? f[fs * (c + 3 * cp[r])] : 0.0;
                    if (r == 0) uo[c] = origin(x[c]);
                }
                if (pn < NNP) {
                    const double w = sw[pn];
                    double *p = bufA + i * C::S0 + jk;
#pragma unroll
                    for (int c = 0; c < 3; ++c) p[c * N * N] = w * (x[c] - uo[c]);
                }
            }
            wave_lds_sync();
            forward(std::integral_constant<int, 3>{});
#pragma unroll
            for (int r = 0; r < PPL; ++r)
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    double s[4], d[3];
                    at_point(r, i, s);
                    u[r][i] = uo[i] + s[0] * Wi[r];
#pragma unroll
                    for (int m = 0; m < 3; ++m) d[m] = (s[1 + m] - s[0] * dw[r][m]) * Wi[r];
#pragma unroll
                    for (int k = 0; k < 3; ++k)
                        D[r][i][k] = d[0] * A[r][k] + d[1] * A[r][3 + k] + d[2] * A[r][6 + k];
                }
        };
        auto stress = [&](const double D[3][3], double s[3][3]) {
            const double tr = ga.lam * (D[0][0] + D[1][1] + D[2][2]);
#pragma unroll
            for (int i = 0; i < 3; ++i)
#pragma unroll
                for (int k = 0; k < 3; ++k) s[i][k] = ga.mu * (D[i][k] + D[k][i]) + (i == k ? tr : 0.0);
        };
        // back: the tensors T[m][k] of the lane's points (g_a[m] = sum_q T[m][k] dR_a/dx_k) to the
        // element's nodes, stored as pair f
        auto backward = [&](const double (*T)[3][3], int f) {
            wave_lds_sync();
#pragma unroll
            for (int r = 0; r < PPL; ++r) {
                const int q = ll + LPE * r;
                if (q < NQ) {
                    double *p = bufB + (q / (Q * Q)) * 4 * C::S3 + q % (Q * Q);
#pragma unroll
                    for (int m = 0; m < 3; ++m) {
                        double t0 = 0.0;
#pragma unroll
                        for (int n = 0; n < 3; ++n) {
                            const double c = Wi[r] * (T[r][m][0] * A[r][3 * n] + T[r][m][1] * A[r][3 * n + 1] +
                                                      T[r][m][2] * A[r][3 * n + 2]);
                            p[(1 + n) * C::S3 + Q * Q * m] = c;
                            t0 -= c * dw[r][n];
                        }
                        p[Q * Q * m] = t0;
                    }
                }
            }
            wave_lds_sync();
            for (int t = ll; t < 3 * Q * Q; t += LPE) {   // xi_2: (g0, g1, m)
                const int g0 = t % Q, g1 = (t / Q) % Q, m = t / (Q * Q);
                double x[Q][4];
#pragma unroll
                for (int g = 0; g < Q; ++g)
#pragma unroll
                    for (int v = 0; v < 4; ++v) x[g][v] = bufB[(g * 4 + v) * C::S3 + t];
#pragma unroll
                for (int k = 0; k < N; ++k) {
                    double v = 0.0, d0 = 0.0, d1 = 0.0;
#pragma unroll
                    for (int g = 0; g < Q; ++g) {
                        const double b = tb[2][g * N + k];
                        v += x[g][0] * b + x[g][3] * tb[2][Q * N + g * N + k];
                        d0 += x[g][1] * b;
                        d1 += x[g][2] * b;
                    }
                    double *p = bufA + g1 * 3 * C::S4 + g0 + Q * k + Q * N * m;
                    p[0] = v;
                    p[C::S4] = d0;
                    p[2 * C::S4] = d1;
                }
            }
            wave_lds_sync();
            for (int t = ll; t < 3 * Q * N; t += LPE) {   // xi_1: (g0, k, m)
                const int g0 = t % Q, k = (t / Q) % N, m = t / (Q * N);
                double x[Q][3];
#pragma unroll
                for (int g = 0; g < Q; ++g)
#pragma unroll
                    for (int v = 0; v < 3; ++v) x[g][v] = bufA[(g * 3 + v) * C::S4 + t];
#pragma unroll
                for (int j = 0; j < N; ++j) {
                    double v = 0.0, d0 = 0.0;
#pragma unroll
                    for (int g = 0; g < Q; ++g) {
                        const double b = tb[1][g * N + j];
                        v += x[g][0] * b + x[g][2] * tb[1][Q * N + g * N + j];
                        d0 += x[g][1] * b;
                    }
                    double *p = bufB + g0 * 2 * C::S5 + j + N * k + N * N * m;
                    p[0] = v;
                    p[C::S5] = d0;
                }
            }
            wave_lds_sync();
            for (int t = ll; t < 3 * N * N; t += LPE) {   // xi_0: (j, k, m)
                const int j = t % N, k = (t / N) % N, m = t / (N * N);
                double x[Q][2];
#pragma unroll
                for (int g = 0; g < Q; ++g)
#pragma unroll
                    for (int v = 0; v < 2; ++v) x[g][v] = bufB[(g * 2 + v) * C::S5 + t];
#pragma unroll
                for (int i = 0; i < N; ++i) {
                    double v = 0.0;
#pragma unroll
                    for (int g = 0; g < Q; ++g)
                        v += x[g][0] * tb[0][g * N + i] + x[g][1] * tb[0][Q * N + g * N + i];
                    if (i < n0 && j < n1 && k < n2)
                        bufA[3 * (i + n0 * (j + n1 * k)) + m] = v * sw[i + N * (j + N * k)];
                }
            }
            wave_lds_sync();
            double *out = ga.eg + 3 * (nout * (ga.ebase + gi * nn) + f);
            if (act)
                for (int x = ll; x < 3 * nn; x += LPE) out[3 * (nout - 1) * (x / 3) + x] = bufA[x];
        };
        const double live = act ? 1.0 : 0.0;
        if constexpr (KIND == GRAD_VOLUME) {
            double T[PPL][3][3];
#pragma unroll
            for (int r = 0; r < PPL; ++r) {
#pragma unroll
                for (int m = 0; m < 3; ++m)
#pragma unroll
                    for (int k = 0; k < 3; ++k) T[r][m][k] = m == k ? dv[r] : 0.0;
                macc[0] += live * dv[r];
            }
            backward(T, 0);
        } else {
            double u[PPL][3], D[PPL][3][3], v[PPL][3], H[PPL][3][3];
            if constexpr (KIND == GRAD_PAIRS) field(ga.f.f0, 1, u, D);
#pragma unroll 1
            for (int f = 0; f < nout; ++f) {
                double ms = 0.0;
                field(ga.f.fk + ga.f.k0 + f, ga.f.nk, v, H);
                double T[PPL][3][3];
#pragma unroll
                for (int r = 0; r < PPL; ++r) {
                    double sv[3][3];
                    stress(H[r], sv);
                    double W = 0.0;
                    if constexpr (KIND == GRAD_PAIRS) {
                        double su[3][3];
                        stress(D[r], su);
#pragma unroll
                        for (int i = 0; i < 3; ++i)
#pragma unroll
                            for (int k = 0; k < 3; ++k) W += su[i][k] * H[r][i][k];
#pragma unroll
                        for (int m = 0; m < 3; ++m)
#pragma unroll
                            for (int k = 0; k < 3; ++k) {
                                double t = m == k ? W : 0.0;
#pragma unroll
                                for (int i = 0; i < 3; ++i) t -= H[r][i][m] * su[i][k] + D[r][i][m] * sv[i][k];
                                T[r][m][k] = dv[r] * t;
                            }
                    } else {
#pragma unroll
                        for (int i = 0; i < 3; ++i)
#pragma unroll
                            for (int k = 0; k < 3; ++k) W += sv[i][k] * H[r][i][k];
                        const double uu = ga.f.rho * (v[r][0] * v[r][0] + v[r][1] * v[r][1] + v[r][2] * v[r][2]);
                        W -= ga.f.vals[f] * uu;
                        ms += live * uu * dv[r];
#pragma unroll
                        for (int m = 0; m < 3; ++m)
#pragma unroll
                            for (int k = 0; k < 3; ++k)
                                T[r][m][k] = dv[r] * ((m == k ? W : 0.0) - 2.0 * (H[r][0][m] * sv[0][k] + H[r][1][m] * sv[1][k] +
                                                                                  H[r][2][m] * sv[2][k]));
                    }
                }
#pragma unroll
                for (int k = 0; k < VIB_MAXF; ++k) macc[k] += k == f ? ms : 0.0;
                backward(T, f);
            }
        }
    }
    // this workgroup's share of each pair's mass, in a fixed order
#pragma unroll
    for (int f = 0; f < VIB_MAXF; ++f) {
        double m = macc[f];
        for (int o = 32; o > 0; o >>= 1) m += __shfl_xor(m, o, 64);
        if (lane == 0) msum[wv][f] = m;
    }
    __syncthreads();
    if (threadIdx.x < VIB_MAXF) {
        double m = 0.0;
        for (int w = 0; w < C::WPB; ++w) m += msum[w][threadIdx.x];
        ga.em[(int64_t)blockIdx.x * VIB_MAXF + threadIdx.x] = m;
    }
}
