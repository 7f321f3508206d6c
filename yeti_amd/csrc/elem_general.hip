// elem_general.hip -- element stiffness and mass matrices for run-time degrees and Gauss orders,
// up to 64 nodes, and stiffness at p = 4, on the FP64 matrix cores.
//
// Stiffness: K_ab[k][l] = lam S^kl_ab + mu S^lk_ab + mu delta_kl tr S_ab with
// S^kl_ab = sum_q G_k[a][q] G_l[b][q], G_c[a][q] = sqrt(w_q |det J_q|) dR_a/dx_c (UELMAT.f90:22-225 with
// stiffmatrix_byCP, stiffmatrix.F90:130-225). Mass: M_ab[k][k] = rho sum_q w_q det J_q R_a R_b, det J
// signed, off-diagonal entries 0 (compute_CMASSMatrix.f:22-215, UMASSMAT.f:220-330). Both in the COO
// order of build_system_elemStorage.f90:260-293.
#include <algorithm>

#include "coo_entries.hpp"
#include "copy_out.hpp"
#include "elem_general.hpp"

namespace yeti {

typedef double f64x2 __attribute__((ext_vector_type(2)));

// One workgroup per element, NT = 16-node tiles, one wave per node-tile pair I <= J, so that a lane
// ends with all nine S^kl of its node pairs and needs no exchange to contract them. Gauss points in
// chunks of QC:
//   1. PARTS lanes per point split the nodes' sums (W, dW, x, dx/du) and add them by shuffles;
//   2. every thread owns a point and writes G (mass: R) for its share of the nodes to LDS;
//   3. each wave adds the chunk to its pair's tiles (v_mfma_f64_16x16x4f64, two K steps per LDS read).
// The entries are then laid out in LDS in COO order (up to NT = 2 the whole element, above one tile
// column J at a time) and copied by all threads front to back; their rows and columns come from
// entry_tab. The mass keeps only M_ab, a <= b, in LDS and expands it on the way out.
// Bound by FP64 issue (matrix and vector instructions do not overlap): 64^3 p = 2 takes 3.8 ms of its
// 5.07 ms without the stores, whose floor is 2.1 ms; the mass at 61x53x47 p = 2 takes 1.0 of 1.99 ms.
// Against vector sums of every node pair from LDS and block-wise stores: 45x14x11 degrees (2,3,1)
// 1018 -> 216 us; mass 61x53x47 p = 2 2.61 -> 1.99 ms, 64^3 p = 1 1.91 -> 0.69 ms.
// NT = 8 (125 nodes): 36 pairs of nine tiles are more accumulators than a CU has registers for, hence
// four workgroups per element. Each builds G again and no two fit a CU (stage of 120 KB); at 23x18x13
// the matrix instructions of the busiest SIMD take 1.6 of 3.76 ms (at 2.4 GHz). Against one persistent
// workgroup of 12 waves, 4 of them building G, with spilled accumulators: values 5.18 -> 3.76 ms, with
// indices 6.05 -> 4.27 ms, 4x4x4 296 -> 95 us. One half for G and two barriers per chunk: 3.90 ms.
template <int NT, int MODE>
struct Gen {
    static constexpr int NNP = 16 * NT;
    // a workgroup takes an element, or at NT = 8 (p = 4) a quarter of it: the tile columns 0-3, 4-5, 6
    // or 7 (10, 11, 7 and 8 pairs) on 11 waves, its geometry from the record of elem_geo_kernel
    static constexpr int PASSES = NT == 8 ? 4 : 1;
    static constexpr int WAVES = NT == 8 ? 11 : NT * (NT + 1) / 2;
    static constexpr int NTH = 64 * WAVES;
    static constexpr int QC = NT <= 2 ? 32 : 16;            // Gauss points per chunk
    __host__ __device__ static constexpr int column(int pass) {   // first tile column of a pass
        return NT != 8 ? (pass == 0 ? 0 : NT) : pass == 0 ? 0 : pass == 1 ? 4 : pass == 2 ? 6 : pass == 3 ? 7 : 8;
    }
    static constexpr int PARTS = NT == 1 ? 2 : NT == 2 ? 4 : 16;   // lanes per point, step 1
    static constexpr int RS = QC + 2;                       // G row (doubles): rows on different banks
    static constexpr int NG_ = MODE == 0 ? 3 : 1;           // arrays per node
    static constexpr int TILES = MODE == 0 ? 9 : 1;
    static constexpr int GDBL = NG_ * NNP * RS;
    // NT = 8: the chunks alternate between two halves, one barrier each; a half is written again once
    // every wave has met the barrier after its last read
    static constexpr int GBUF = NT == 8 ? 2 : 1;
    static constexpr int WPE = MODE == 1 ? 4 : 3;           // waves per SIMD
    static_assert(NT == 8 || PARTS * QC <= NTH, "one pass over the chunk's points");
};

constexpr int GEN_NGEO = 12;

// sum over PARTS adjacent lanes (a power of two up to 16), in every lane of the group
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v) { return v + __builtin_amdgcn_mov_dpp(v, CTRL, 0xF, 0xF, true); }
template <int PARTS>
__device__ __forceinline__ double parts_sum(double v) {
    v = dpp_add<0xB1>(v);                          // quad_perm [1, 0, 3, 2]
    if constexpr (PARTS >= 4) v = dpp_add<0x4E>(v);  // quad_perm [2, 3, 0, 1]
    if constexpr (PARTS >= 16) {
        v = dpp_add<0x124>(v);                     // row_ror 4, then 8
        v = dpp_add<0x128>(v);
    }
    return v;
}

// x / n for x < 1024, n <= 81 with m = ceil(65536 / n): x (m n - 65536) < 65536
__device__ __forceinline__ int div_by(int x, int m) { return (x * m) >> 16; }

static_assert(GEN_MAXN == ENTRY_NODES, "entry_tab holds every element");
static_assert(coo_start(16) % 8 == 0 && coo_start(32) % 8 == 0 && coo_start(48) % 8 == 0 &&
                  coo_start(GEN_MAXN) % 8 == 0,
              "the rounds' table rows are copied 16 bytes at a time");

// Largest number of entries of a round: the whole element up to NT = 2, else a tile column
template <int NT>
__host__ __device__ constexpr int gen_round_entries(int nn) {
    if (NT <= 2) return coo_start(nn);
    const int last = coo_start(nn) - coo_start(16 * (NT - 1));
    const int prev = coo_start(16 * (NT - 1)) - coo_start(16 * (NT - 2));
    return last > prev ? last : prev;
}

// dynamic LDS: G of a chunk or the values of a round (doubles); mass: then the round's table rows
template <int NT, int MODE>
__host__ __device__ constexpr int gen_values(int nn) {
    const int v = MODE == 1 ? 1 + nn * (nn + 1) / 2 : gen_round_entries<NT>(nn);
    constexpr int g = Gen<NT, MODE>::GBUF * Gen<NT, MODE>::GDBL;
    return v > g ? v : g;
}

template <int NT, int MODE, bool IDX>
__global__ void __launch_bounds__((Gen<NT, MODE>::NTH)) __attribute__((amdgpu_waves_per_eu(Gen<NT, MODE>::WPE)))
elem_general_kernel(GenArgs ga, double *__restrict__ Kd, int32_t *__restrict__ Kr, int32_t *__restrict__ Kc) {
    using C = Gen<NT, MODE>;
    constexpr int NNP = C::NNP, QC = C::QC, RS = C::RS, NTH = C::NTH, TILES = C::TILES;
    // G of a chunk; after the last one the values of a round; for the mass then the round's rows of
    // entry_tab (a load among the stores of the copy would wait for them: one counter covers both)
    extern __shared__ __attribute__((aligned(16))) double sm[];
    __shared__ __attribute__((aligned(16))) double gq[MODE == 0 ? GEN_NGEO : 2][NT == 8 ? 2 : QC];   // sqrt(dv) dxi_m/dx_c / W (9), dW/dxi_m / W (3); mass: 1/W, dv
    __shared__ double tb[3][2 * MAX_NG * (GEN_MAXP + 1) + 2];   // per direction: [B | dB][g][i], half span
    __shared__ __attribute__((aligned(16))) double xw[NNP][4];
    __shared__ int32_t dof[3 * NNP];
    const int t = threadIdx.x, lane = t & 63, wv = __builtin_amdgcn_readfirstlane(t >> 6);
    const int nl = lane & 15, kg = lane >> 4;
    const int n0 = ga.n[0], n1 = ga.n[1], NL = n1 * ga.n[2], NN = n0 * NL;
    const int ng = ga.ng, NQ = ng * ng * ng, TN = ga.tab_n, rec = 2 * ng * TN + 2;
    const int mg = (65535 + ng) / ng, mg2 = (65535 + ng * ng) / (ng * ng), mn1 = (65535 + n1) / n1;
    // one element per workgroup (a loop over elements would keep the entries' indices in registers
    // from one to the next)
    {
        const int64_t item = xcd_element(blockIdx.x, (int64_t)ga.n_active * C::PASSES);
        if (item >= (int64_t)ga.n_active * C::PASSES) return;
        const int64_t gi = item / C::PASSES;
        const int pass = (int)(item % C::PASSES), J0 = C::column(pass), J1 = C::column(pass + 1);
        const int e = ga.elems[gi];
        for (int a = t; a < NNP; a += NTH) {
            const bool in = a < NN;
            const int32_t cp = in ? ga.ien[(int64_t)NN * e + a] - 1 : 0;
            const int32_t c0 = ga.ien[(int64_t)NN * e] - 1;
            // positions relative to node 0: their derivatives do not see it
            for (int c = 0; c < 3; ++c) {
                xw[a][c] = in ? ga.coords[3 * (int64_t)cp + c] - ga.coords[3 * (int64_t)c0 + c] : 0.0;
                dof[3 * a + c] = 3 * cp + c;
            }
            xw[a][3] = in ? ga.weight[(int64_t)NN * e + a] : 0.0;
        }
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const double *src = ga.tab[d] + (int64_t)(ga.nijk[3 * (int64_t)e + d] - 1) * rec;
            for (int x = t; x < rec; x += NTH) tb[d][x] = src[x];
        }
        uint16_t *et = reinterpret_cast<uint16_t *>(sm + (gen_values<NT, MODE>(NN) + 1) / 2 * 2);
        auto load_tab = [&](int x0, int x1) {
            typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
            const u32x4 *src = reinterpret_cast<const u32x4 *>(entry_tab.v + x0);
            for (int x = t; x < (x1 - x0 + 7) / 8; x += NTH) reinterpret_cast<u32x4 *>(et)[x] = src[x];
        };
        constexpr int ROUNDS = NT <= 2 ? 1 : NT;
        if (ROUNDS == 1 && MODE == 1) load_tab(0, coo_start(NN));
        f64x4 acc[TILES];
#pragma unroll
        for (int s = 0; s < TILES; ++s) acc[s] = f64x4{0.0, 0.0, 0.0, 0.0};
        // pair of the wave, column by column: pr = J (J + 1) / 2 + I
        const int pr = J0 * (J0 + 1) / 2 + wv;
        const int J = pr < 1 ? 0 : pr < 3 ? 1 : pr < 6 ? 2 : pr < 10 ? 3 : pr < 15 ? 4 : pr < 21 ? 5 : pr < 28 ? 6 : 7;
        const int I = pr - J * (J + 1) / 2;
        const bool has = J < J1 && I <= J;   // not a wave beyond the pass's pairs
        // NT = 8: the thread's point of the next chunk, from the record ([12][points], xi_0 fastest)
        const double *geo = NT == 8 ? ga.geo + gi * ga.geo_rec : nullptr;
        double Ap[NT == 8 ? GEN_NGEO : 1];
        if constexpr (NT == 8) {
#pragma unroll
            for (int m = 0; m < GEN_NGEO; ++m) Ap[m] = geo[m * NQ + min(t % QC, NQ - 1)];
        }
        __syncthreads();
        for (int q0 = 0; q0 < NQ; q0 += QC) {
            const int nq = min(NQ - q0, QC);
            // 1. geometry of the chunk's points (3D rule: i slowest, k fastest, GaussLegendre.f90:175-186):
            // along a node line (j, k) first, then the line's sums with its xi_1, xi_2 functions
            if constexpr (NT != 8) {
                const int qq = t / C::PARTS, part = t % C::PARTS;
                double s[16];
#pragma unroll
                for (int m = 0; m < 16; ++m) s[m] = 0.0;
                const int q = q0 + qq, g0 = div_by(q, mg2), g1 = div_by(q - g0 * ng * ng, mg), g2 = q - ng * (ng * g0 + g1);
                if (qq < nq) {
                    const double *T0 = &tb[0][g0 * TN], *T1 = &tb[1][g1 * TN], *T2 = &tb[2][g2 * TN];
                    const int dB = ng * TN;
                    for (int l = part; l < NL; l += C::PARTS) {
                        const int k = div_by(l, mn1), j = l - n1 * k;
                        double v[4] = {0.0, 0.0, 0.0, 0.0}, d[4] = {0.0, 0.0, 0.0, 0.0};   // of w, w x_r
                        for (int i = 0; i < n0; ++i) {
                            const f64x2 p0 = *reinterpret_cast<const f64x2 *>(&xw[i + n0 * l][0]);
                            const f64x2 p1 = *reinterpret_cast<const f64x2 *>(&xw[i + n0 * l][2]);
                            const double b = T0[i] * p1.y, db = T0[dB + i] * p1.y;
                            v[0] += b;
                            v[1] += b * p0.x;
                            v[2] += b * p0.y;
                            v[3] += b * p1.x;
                            d[0] += db;
                            d[1] += db * p0.x;
                            d[2] += db * p0.y;
                            d[3] += db * p1.x;
                        }
                        const double b1 = T1[j], b2 = T2[k], b12 = b1 * b2, d1 = T1[dB + j] * b2, d2 = b1 * T2[dB + k];
                        s[0] += v[0] * b12;
                        s[1] += d[0] * b12;
                        s[2] += v[0] * d1;
                        s[3] += v[0] * d2;
#pragma unroll
                        for (int r = 0; r < 3; ++r) {
                            s[4 + r] += v[1 + r] * b12;
                            s[7 + 3 * r] += d[1 + r] * b12;
                            s[8 + 3 * r] += v[1 + r] * d1;
                            s[9 + 3 * r] += v[1 + r] * d2;
                        }
                    }
                }
#pragma unroll
                for (int m = 0; m < 16; ++m) s[m] = parts_sum<C::PARTS>(s[m]);
                if (part == 0 && qq < nq) {
                    const double Wi = 1.0 / s[0];
                    const double dw[3] = {s[1] * Wi, s[2] * Wi, s[3] * Wi};
                    double Jm[3][3];
#pragma unroll
                    for (int r = 0; r < 3; ++r)
#pragma unroll
                        for (int c = 0; c < 3; ++c) Jm[r][c] = (s[7 + 3 * r + c] - s[4 + r] * dw[c]) * Wi;
                    double A[9];   // adj J, [m][c]
                    A[0] = Jm[1][1] * Jm[2][2] - Jm[1][2] * Jm[2][1];
                    A[1] = Jm[0][2] * Jm[2][1] - Jm[0][1] * Jm[2][2];
                    A[2] = Jm[0][1] * Jm[1][2] - Jm[0][2] * Jm[1][1];
                    A[3] = Jm[1][2] * Jm[2][0] - Jm[1][0] * Jm[2][2];
                    A[4] = Jm[0][0] * Jm[2][2] - Jm[0][2] * Jm[2][0];
                    A[5] = Jm[0][2] * Jm[1][0] - Jm[0][0] * Jm[1][2];
                    A[6] = Jm[1][0] * Jm[2][1] - Jm[1][1] * Jm[2][0];
                    A[7] = Jm[0][1] * Jm[2][0] - Jm[0][0] * Jm[2][1];
                    A[8] = Jm[0][0] * Jm[1][1] - Jm[0][1] * Jm[1][0];
                    const double det = Jm[0][0] * A[0] + Jm[0][1] * A[3] + Jm[0][2] * A[6];
                    const double dv = ga.g.w[g0] * ga.g.w[g1] * ga.g.w[g2] * (det * (tb[0][2 * ng * TN] * tb[1][2 * ng * TN] * tb[2][2 * ng * TN]));
                    if (MODE == 0) {
                        const double f = sqrt(fabs(dv)) * Wi / det;
#pragma unroll
                        for (int m = 0; m < 9; ++m) gq[m][qq] = A[m] * f;
#pragma unroll
                        for (int m = 0; m < 3; ++m) gq[9 + m][qq] = dw[m];
                    } else {
                        gq[0][qq] = Wi;
                        gq[1][qq] = ga.rho * dv;
                    }
                } else if (MODE == 1 && part == 0 && qq < QC) {
                    gq[1][qq] = 0.0;
                }
            }
            if (NT != 8) __syncthreads();
            double *smg = C::GBUF == 2 ? sm + (q0 / QC % 2) * C::GDBL : sm;
            // 2. G of the chunk, zero past the nodes and past the points (up to a multiple of 8)
            {
                constexpr int PER = NTH / QC;      // threads per point
                const int qq = t % QC, part = t / QC, nq8 = (nq + 7) & ~7;
                if (part < PER && qq < nq8) {
                    const bool inq = qq < nq;
                    const int q = inq ? q0 + qq : q0, qs = div_by(q, mg2), g1 = div_by(q - qs * ng * ng, mg),
                              qf = q - ng * (ng * qs + g1);
                    const int g0 = NT == 8 ? qf : qs, g2 = NT == 8 ? qs : qf;
                    const double *T0 = &tb[0][g0 * TN], *T1 = &tb[1][g1 * TN], *T2 = &tb[2][g2 * TN];
                    const int dB = ng * TN;
                    double A[GEN_NGEO];
#pragma unroll
                    for (int m = 0; m < (MODE == 0 ? GEN_NGEO : 1); ++m) {
                        if constexpr (NT == 8) A[m] = inq ? Ap[m] : 0.0;
                        else A[m] = inq ? gq[m][qq] : 0.0;
                    }
                    for (int l = part; l < NL; l += PER) {
                        const int k = div_by(l, mn1), j = l - n1 * k;
                        const double b1 = T1[j], b2 = T2[k], b12 = b1 * b2, d1 = T1[dB + j] * b2, d2 = b1 * T2[dB + k];
                        for (int i = 0; i < n0; ++i) {
                            const int a = i + n0 * l;
                            const double w = xw[a][3], bw = T0[i] * w, N = bw * b12;
                            if (MODE == 0) {
                                const double t0 = T0[dB + i] * w * b12 - N * A[9];
                                const double t1 = bw * d1 - N * A[10];
                                const double t2 = bw * d2 - N * A[11];
#pragma unroll
                                for (int c = 0; c < 3; ++c)
                                    smg[(c * NNP + a) * RS + qq] = t0 * A[c] + t1 * A[3 + c] + t2 * A[6 + c];
                            } else {
                                smg[a * RS + qq] = N * A[0];
                            }
                        }
                    }
                    for (int a = NN + part; a < NNP; a += PER)
#pragma unroll
                        for (int c = 0; c < C::NG_; ++c) smg[(c * NNP + a) * RS + qq] = 0.0;
                }
            }
            if constexpr (NT == 8) {
                const int qn = min(q0 + QC + t % QC, NQ - 1);
#pragma unroll
                for (int m = 0; m < GEN_NGEO; ++m) Ap[m] = geo[m * NQ + qn];
            }
            __syncthreads();
            // 3. K step 2v uses point 8v + 2 kg, step 2v + 1 point 8v + 2 kg + 1, in A and B alike
            const int nv = has ? (nq + 7) / 8 : 0;
#pragma unroll 1
            for (int v = 0; v < nv; ++v) {
                const int qo = 8 * v + 2 * kg;
                if constexpr (MODE == 0) {
                    f64x2 a[3], b[3];
#pragma unroll
                    for (int c = 0; c < 3; ++c) {
                        a[c] = *reinterpret_cast<const f64x2 *>(&smg[(c * NNP + 16 * I + nl) * RS + qo]);
                        b[c] = *reinterpret_cast<const f64x2 *>(&smg[(c * NNP + 16 * J + nl) * RS + qo]);
                    }
#pragma unroll
                    for (int s = 0; s < 9; ++s)
                        acc[s] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s / 3].x, b[s % 3].x, acc[s], 0, 0, 0);
#pragma unroll
                    for (int s = 0; s < 9; ++s)
                        acc[s] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[s / 3].y, b[s % 3].y, acc[s], 0, 0, 0);
                } else {
                    const f64x2 dv = *reinterpret_cast<const f64x2 *>(&gq[1][qo]);
                    const f64x2 a = *reinterpret_cast<const f64x2 *>(&smg[(16 * I + nl) * RS + qo]) * dv;
                    const f64x2 b = *reinterpret_cast<const f64x2 *>(&smg[(16 * J + nl) * RS + qo]);
                    acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.x, acc[0], 0, 0, 0);
                    acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.y, acc[0], 0, 0, 0);
                }
            }
            if (C::GBUF == 1) __syncthreads();
        }
        if (C::GBUF == 2) __syncthreads();
        const int64_t base = ga.offs[gi];
        double *Ke = Kd + base;
        int32_t *Re = IDX ? Kr + base : nullptr, *Ce = IDX ? Kc + base : nullptr;
        const double lam = ga.lam, mu = ga.mu;
        if constexpr (MODE == 1) {
            // M_ab at 1 + b (b + 1) / 2 + a, the diagonal halved; entry 0 is the zero of k != l
            const int b = 16 * J + nl;
            if (t == 0) sm[0] = 0.0;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int a = 16 * I + 4 * r + kg;
                if (a <= b && b < NN) sm[1 + b * (b + 1) / 2 + a] = a < b ? acc[0][r] : 0.5 * acc[0][r];
            }
        }
#pragma unroll 1
        for (int rd = NT == 8 ? J0 : 0; rd < (NT == 8 ? J1 : ROUNDS); ++rd) {
            const int x0 = ROUNDS == 1 ? 0 : coo_start(16 * rd);
            const int x1 = ROUNDS == 1 ? coo_start(NN) : coo_start(min(16 * rd + 16, NN));
            if (ROUNDS > 1 && MODE == 1) load_tab(x0, x1);
            if (MODE == 0 && (ROUNDS == 1 || J == rd)) {
                // register r of lane l holds row (l >> 4) + 4 r and column l & 15 of a tile
                const int b = 16 * J + nl;
                double *col = sm + coo_start(b) - x0;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int a = 16 * I + 4 * r + kg;
                    double K[9];   // [k + 3 l]
                    const double tr = mu * (acc[0][r] + acc[4 % TILES][r] + acc[8 % TILES][r]);
#pragma unroll
                    for (int k = 0; k < 3; ++k)
#pragma unroll
                        for (int l = 0; l < 3; ++l)
                            K[k + 3 * l] = lam * acc[(3 * k + l) % TILES][r] + mu * acc[(3 * l + k) % TILES][r] +
                                           (k == l ? tr : 0.0);
                    if (b >= NN || a > b) continue;
                    double *s = col + 9 * a;
                    if (a < b) {
#pragma unroll
                        for (int x = 0; x < 9; ++x) s[x] = K[x];
                    } else {   // (0,0) (0,1) (1,1) (0,2) (1,2) (2,2), the diagonal halved
                        s[0] = 0.5 * K[0];
                        s[1] = K[3];
                        s[2] = 0.5 * K[4];
                        s[3] = K[6];
                        s[4] = K[7];
                        s[5] = 0.5 * K[8];
                    }
                }
            }
            if constexpr (MODE == 0) {
                // the stiffness has no LDS to spare for the table: its words for the thread's rows and
                // columns are loaded now, before the first store
                typedef uint16_t u16x4 __attribute__((ext_vector_type(4), aligned(2)));
                typedef int32_t i32x4 __attribute__((ext_vector_type(4), aligned(4)));
                constexpr bool TAB = IDX && NT != 8;
                constexpr int U = TAB ? (gen_round_entries<NT>(NNP) + 4 * NTH - 1) / (4 * NTH) : 1;
                const int n = x1 - x0;
                u16x4 rc[U];
                int head = 0, end = 0, xs = -1;   // xs: a single entry before or after the 16-byte ones
                unsigned rs = 0;
                if (TAB) {
                    head = min(n, (int)((0 - reinterpret_cast<uintptr_t>(Re + x0)) / 4 % 32));
                    end = head + (n - head) / 4 * 4;
                    xs = t < head ? t : t - head < n - end ? end + t - head : -1;
                    const uint16_t *tab = entry_tab.v + x0;
                    rs = tab[max(xs, 0)];
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int x = head + 4 * (t + NTH * u);
                        if (x < end) rc[u] = *reinterpret_cast<const u16x4 *>(tab + x);
                    }
                }
                __syncthreads();
                if (IDX && NT == 8) {
                    // 9-bit dofs, which entry_tab does not hold: row by row
                    for (int b = 16 * rd + wv; b < min(16 * rd + 16, NN); b += C::WAVES) {
                        int32_t *Rb = Re + coo_start(b), *Cb = Ce + coo_start(b);
                        for (int y = lane; y < 9 * b + 6; y += 64) {
                            const int a = y < 9 * b ? y / 9 : b, m = y - 9 * a;
                            const int kk = a < b ? m % 3 : (0x210100 >> (4 * m)) & 15;
                            const int ll = a < b ? m / 3 : (0x222110 >> (4 * m)) & 15;
                            Rb[y] = dof[3 * a + kk];
                            Cb[y] = dof[3 * b + ll];
                        }
                    }
                }
                if (TAB) {
                    if (xs >= 0) {
                        Re[x0 + xs] = dof[rs & 255];
                        Ce[x0 + xs] = dof[rs >> 8];
                    }
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int x = head + 4 * (t + NTH * u);
                        if (x < end) {
                            i32x4 r, c;
#pragma unroll
                            for (int y = 0; y < 4; ++y) {
                                r[y] = dof[rc[u][y] & 255];
                                c[y] = dof[rc[u][y] >> 8];
                            }
                            *reinterpret_cast<i32x4 *>(Re + x0 + x) = r;
                            *reinterpret_cast<i32x4 *>(Ce + x0 + x) = c;
                        }
                    }
                }
                store_run<NTH>(Ke + x0, n, t, [&](int x) { return sm[x]; });
            } else {
                __syncthreads();
                store_run<NTH>(Ke + x0, x1 - x0, t, [&](int x) {
                    const int r = et[x] & 255, c = et[x] >> 8, a = (r * 171) >> 9, b = (c * 171) >> 9;   // / 3
                    return sm[r - 3 * a == c - 3 * b ? 1 + b * (b + 1) / 2 + a : 0];
                });
                if (IDX) {
                    store_run<NTH>(Re + x0, x1 - x0, t, [&](int x) { return dof[et[x] & 255]; });
                    store_run<NTH>(Ce + x0, x1 - x0, t, [&](int x) { return dof[et[x] >> 8]; });
                }
            }
            if (rd + 1 < (NT == 8 ? J1 : ROUNDS)) __syncthreads();
        }
    }
}

template <int NT, int MODE>
static size_t gen_smem_bytes(int nn) {
    return sizeof(double) * (size_t)((gen_values<NT, MODE>(nn) + 1) / 2 * 2) +
           (MODE == 1 ? sizeof(uint16_t) * (size_t)((gen_round_entries<NT>(nn) + 7) / 8 * 8) : 0);
}

// A grid holds fewer than 2^32 threads; of a larger one only the remainder is launched, without an
// error. The elements go in runs below that (p = 1, 64 threads each: 67,108,856 elements, 161 GB of
// values).
template <int NT, int MODE>
static int launch_kind(GenArgs ga, double *Kd, int32_t *Kr, int32_t *Kc, hipStream_t st) {
    using C = Gen<NT, MODE>;
    constexpr int64_t MOST = (0xffffffffLL / C::NTH / XCDS * XCDS) / C::PASSES;
    const size_t lds = gen_smem_bytes<NT, MODE>(ga.n[0] * ga.n[1] * ga.n[2]);
    const int64_t n = ga.n_active;
    for (int64_t e0 = 0; e0 < n; e0 += MOST) {
        ga.n_active = (int32_t)std::min(MOST, n - e0);
        const dim3 grid(xcd_grid((int64_t)ga.n_active * C::PASSES)), block(C::NTH);
        if (Kr) hipLaunchKernelGGL((elem_general_kernel<NT, MODE, true>), grid, block, lds, st, ga, Kd, Kr, Kc);
        else hipLaunchKernelGGL((elem_general_kernel<NT, MODE, false>), grid, block, lds, st, ga, Kd, Kr, Kc);
        YETI_HIP(hipGetLastError());
        ga.elems += ga.n_active;
        ga.offs += ga.n_active;
        if (ga.geo) ga.geo += ga.n_active * ga.geo_rec;
    }
    return 0;
}

template <int NT>
static int launch_nt(const GenArgs &ga, bool mass, double *Kd, int32_t *Kr, int32_t *Kc, hipStream_t st) {
    return mass ? launch_kind<NT, 1>(ga, Kd, Kr, Kc, st) : launch_kind<NT, 0>(ga, Kd, Kr, Kc, st);
}

int launch_elem_general(const GenArgs &ga, bool mass, double *Kd, int32_t *Kr, int32_t *Kc, hipStream_t st) {
    const int nn = ga.n[0] * ga.n[1] * ga.n[2];
    if (ga.geo && nn == 125 && ga.tab_n == 5 && ga.ng == 5 && !mass) return launch_kind<8, 0>(ga, Kd, Kr, Kc, st);
    if (nn < 1 || nn > GEN_MAXN || ga.tab_n < 1 || ga.tab_n > GEN_MAXP + 1 || ga.ng < 1 || ga.ng > MAX_NG)
        return set_error(YETI_ERR_UNSUPPORTED_DEGREE, "general element kernel: %d nodes, %d points", nn, ga.ng);
    switch ((nn + 15) / 16) {
    case 1: return launch_nt<1>(ga, mass, Kd, Kr, Kc, st);
    case 2: return launch_nt<2>(ga, mass, Kd, Kr, Kc, st);
    case 3: return launch_nt<3>(ga, mass, Kd, Kr, Kc, st);
    default: return launch_nt<4>(ga, mass, Kd, Kr, Kc, st);
    }
}

}  // namespace yeti
