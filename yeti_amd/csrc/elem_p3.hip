// elem_p3.hip -- element stiffness for p = 3 with 4 Gauss points per direction, by sum factorisation
// on the FP64 matrix cores.
//
// Node pair (a, b), a = (i0, i1, i2), b = (j0, j1, j2), of an element:
//   K_ab[k][l] = w_a w_b sum_q sum_mn E_mn(q) D_m N_a(q) D_n N_b(q),
//   E_mn = lam c_mk c_nl + mu c_ml c_nk + mu d_kl sum_r c_mr c_nr,  m, n = 0..3,
// with D_0..D_2 the derivatives, D_3 the value, c_mk = A[m][k] of the geometry record and
// c_3k = -sum_m dw_m A[m][k] (the NURBS quotient rule). Every D_m N_a is a product of three 1D
// functions, so the sum over the 64 points is three contractions with the 4-point products of a
// direction's functions, over 16 pairs (i, j) each: xi_2, xi_0, xi_1. All of them are 16 x 16 x 4
// steps of v_mfma_f64_16x16x4f64, with no padding, and an accumulator tile is the next
// contraction's A operand as it stands:
//   1. A = E_mn, lane = g0 + 4 g1 + 16 g2, a Gauss point per lane; B = the xi_2 products, lane =
//      pair2 + 16 g2. D: lane = pair2 + 16 g0, register g1.
//   2. A = register g1 of it, B = the xi_0 products (lane = pair0 + 16 g0). D of g1: lane =
//      pair0 + 16 i2, register j2.
//   3. lane bits 4..5 (i2) and the tile index g1 change places (permlane swaps); A = (i2, j2): lane =
//      pair0 + 16 g1, B = the xi_1 products. D: lane = i1 + 4 j1 + 16 i0, register j0.
// One (k, l) takes 16 + 36 + 64 MFMAs (k < l, all node pairs; a > b gives the entry (l, k) of the
// transposed block) or 16 + 36 + 40 (k = l, i2 <= j2): 624 per element, where the products of all
// node pairs with all points take 1248 and the vector work of forming G.
//
// A persistent workgroup of 8 waves per CU: waves 0..5 compute one (k, l) each, waves 6 and 7 store.
// The element's entries lie in LDS in COO order in two regions, the tile rows max(i2, j2) < 3 and
// = 3. In step A of element e the compute waves fill the first region while the stores of the second
// one (element e - 1) run; in step B they fill the second one while the first one is stored. A store
// wave holds the dofs (entry_tab) of all its entries in registers and loads nothing between stores.
// 64^3 with indices 24.3 -> 15.1 ms per assembly, 40^3 values only 4.89 -> 3.20 ms, against
// warp-specialised products of all node pairs with all points (78 tiles of 16 K steps, chunks of G
// built beside them). With indices the stores (296 KB per element, 27k cycles at 6.7 TB/s) and the two
// compute waves of SIMDs 0 and 1 (13k cycles of MFMA) bound it, values only the compute waves.
#include <algorithm>
#include <type_traits>

#include "coo_entries.hpp"
#include "copy_out.hpp"
#include "elem_p3.hpp"

namespace yeti {

typedef double f64x2 __attribute__((ext_vector_type(2)));
typedef double f64x2u __attribute__((ext_vector_type(2), aligned(8)));
typedef int32_t i32x4u __attribute__((ext_vector_type(4), aligned(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

namespace p3 {
constexpr int NDE = 18528, SPLIT = 10440;              // entries, first entry of the rows of i2 or j2 = 3
constexpr int OTAB = 12 * 64, OW = OTAB + 96, ODOF = OW + 64, REC = ODOF + 32;   // geometry record (elem_geo_kernel)
constexpr int CWAVES = 6, SWAVES = 2, NTH = 64 * (CWAVES + SWAVES);
constexpr int SL = 64 * SWAVES;                        // store lanes
constexpr int WORDS = NDE / 4, WPL = (WORDS + SL - 1) / SL;   // four entries each; per lane

static_assert(coo_start(64) == NDE && coo_start(48) == SPLIT, "COO layout");

__device__ __forceinline__ f64x4 mm(double a, double b, f64x4 c) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0); }

// lane bit 5 (W = 32) or 4 (W = 16) changes places with "x or y"
template <int W>
__device__ __forceinline__ void swap_rows(double &x, double &y) {
    union U {
        double d;
        unsigned u[2];
    } a, b;
    a.d = x;
    b.d = y;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        if constexpr (W == 32) {
            const auto r = __builtin_amdgcn_permlane32_swap(a.u[h], b.u[h], false, false);
            a.u[h] = r[0];
            b.u[h] = r[1];
        } else {
            const auto r = __builtin_amdgcn_permlane16_swap(a.u[h], b.u[h], false, false);
            a.u[h] = r[0];
            b.u[h] = r[1];
        }
    }
    x = a.d;
    y = b.d;
}

// what a compute wave reads of an element: its Gauss point's geometry, the 1D functions i and j of
// its lane at point lane >> 4 of each direction, and the weight of node `lane`
struct Frag {
    double g[12], bi[3], bj[3], di[3], dj[3], w;
    __device__ __forceinline__ void load(const double *__restrict__ rec, int lane) {
        const int q = lane >> 4, i = lane & 3, j = (lane >> 2) & 3;
#pragma unroll
        for (int v = 0; v < 12; ++v) g[v] = rec[64 * v + lane];
#pragma unroll
        for (int d = 0; d < 3; ++d) {
            const double *t = rec + OTAB + (d * 4 + q) * 4;
            bi[d] = t[i];
            bj[d] = t[j];
            di[d] = t[48 + i];
            dj[d] = t[48 + j];
        }
        w = rec[OW + lane];
    }
};

// products of a direction's functions: (value | derivative of i) x (value | derivative of j)
struct Prod {
    double bb, bd, db, dd;
    __device__ __forceinline__ Prod(double bi, double bj, double di, double dj)
        : bb(bi * bj), bd(bi * dj), db(di * bj), dd(di * dj) {}
};
}  // namespace p3

template <bool IDX>
__global__ void __launch_bounds__(p3::NTH, 2)
elem_p3_kernel(const double *__restrict__ geo, const int64_t *__restrict__ offs, int32_t n, double lam, double mu,
               double *__restrict__ Kd, int32_t *__restrict__ Kr, int32_t *__restrict__ Kc) {
    using namespace p3;
    __shared__ __attribute__((aligned(16))) double st[NDE];
    __shared__ int32_t dofs[SWAVES][192];
    __shared__ __attribute__((aligned(16))) double wls[CWAVES][64];   // node weights, a copy per compute wave
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    __shared__ __attribute__((aligned(16))) int32_t start8[64];   // byte offset of a node's row of entries
    if (threadIdx.x < 64) start8[threadIdx.x] = 8 * coo_start(threadIdx.x);
    __syncthreads();
    const int64_t nidx = (int64_t)xcd_per(n) * XCDS;
    // element of step index s of this workgroup, -1 past the end of its XCD's run
    auto elem_at = [&](int64_t s) -> int64_t {
        const int64_t x = blockIdx.x + s * gridDim.x;
        if (x >= nidx) return -1;
        const int64_t gi = xcd_element(x, n);
        return gi < n ? gi : -1;
    };
    // the run's elements come first: the first -1 ends the workgroup's work
    if (elem_at(0) < 0) return;
    if (wv < CWAVES) {
        // SIMD w mod 4: waves 0, 4 and 1 carry the cheaper k = l
        const int k = wv == 0 ? 0 : wv == 4 ? 1 : wv == 1 ? 2 : wv == 2 ? 0 : wv == 3 ? 0 : 1;
        const int l = wv == 0 ? 0 : wv == 4 ? 1 : wv == 1 ? 2 : wv == 2 ? 1 : wv == 3 ? 2 : 2;
        const bool diag = k == l;
        const int i1 = lane & 3, j1 = (lane >> 2) & 3, i0 = lane >> 4;
        const int a0 = i0 + 4 * i1, b1 = 4 * j1;
        // byte offsets of the lane's entries in a row of b (a < b), of a (a > b) and of the diagonal block
        const int dpos = diag ? (k == 0 ? 0 : k == 1 ? 2 : 5) : k + l == 1 ? 1 : k + l == 2 ? 3 : 4;
        const int up = 72 * a0 + 8 * (k + 3 * l), low = 72 * b1 + 8 * (l + 3 * k), dg = 72 * b1 + 8 * dpos;
        double *wl = wls[wv];
        Frag f;
        f.load(geo + elem_at(0) * REC, lane);
        for (int64_t s = 0;; ++s) {
            // ---- step A ----
            wl[lane] = f.w;   // put reads other lanes' weights
            wave_lds_sync();
            f64x4 D[4][4];   // [combination][g1, then i2]
            double ck[4], cl[4], c[4][3];
#pragma unroll
            for (int r = 0; r < 3; ++r) {
#pragma unroll
                for (int m = 0; m < 3; ++m) c[m][r] = f.g[3 * m + r];
                c[3][r] = -(f.g[9] * c[0][r] + f.g[10] * c[1][r] + f.g[11] * c[2][r]);
            }
#pragma unroll
            for (int m = 0; m < 4; ++m) {
                ck[m] = k == 0 ? c[m][0] : k == 1 ? c[m][1] : c[m][2];
                cl[m] = l == 0 ? c[m][0] : l == 1 ? c[m][1] : c[m][2];
            }
            auto E = [&](int m, int q) {
                double e = lam * (ck[m] * cl[q]) + mu * (cl[m] * ck[q]);
                if (diag) e += mu * (c[m][0] * c[q][0] + c[m][1] * c[q][1] + c[m][2] * c[q][2]);
                return e;
            };
            const Prod P0(f.bi[0], f.bj[0], f.di[0], f.dj[0]), P1(f.bi[1], f.bj[1], f.di[1], f.dj[1]),
                P2(f.bi[2], f.bj[2], f.di[2], f.dj[2]);
            const f64x4 Z = {0.0, 0.0, 0.0, 0.0};
            {   // (d1, d1)
                const f64x4 t = mm(E(1, 1), P2.bb, Z);
#pragma unroll
                for (int g = 0; g < 4; ++g) D[0][g] = mm(t[g], P0.bb, Z);
            }
            {   // (d1, v)
                const f64x4 t0 = mm(E(1, 0), P2.bb, Z);
                const f64x4 tv = mm(E(1, 3), P2.bb, mm(E(1, 2), P2.bd, Z));
#pragma unroll
                for (int g = 0; g < 4; ++g) D[1][g] = mm(t0[g], P0.bd, Z);
#pragma unroll
                for (int g = 0; g < 4; ++g) D[1][g] = mm(tv[g], P0.bb, D[1][g]);
            }
            {   // (v, d1)
                const f64x4 t0 = mm(E(0, 1), P2.bb, Z);
                const f64x4 tv = mm(E(3, 1), P2.bb, mm(E(2, 1), P2.db, Z));
#pragma unroll
                for (int g = 0; g < 4; ++g) D[2][g] = mm(t0[g], P0.db, Z);
#pragma unroll
                for (int g = 0; g < 4; ++g) D[2][g] = mm(tv[g], P0.bb, D[2][g]);
            }
            {   // (v, v)
                const f64x4 t00 = mm(E(0, 0), P2.bb, Z);
                const f64x4 t0v = mm(E(0, 3), P2.bb, mm(E(0, 2), P2.bd, Z));
                const f64x4 tv0 = mm(E(3, 0), P2.bb, mm(E(2, 0), P2.db, Z));
                const f64x4 tvv = mm(E(3, 3), P2.bb, mm(E(3, 2), P2.bd, mm(E(2, 3), P2.db, mm(E(2, 2), P2.dd, Z))));
#pragma unroll
                for (int g = 0; g < 4; ++g) D[3][g] = mm(t00[g], P0.dd, Z);
#pragma unroll
                for (int g = 0; g < 4; ++g) D[3][g] = mm(t0v[g], P0.db, D[3][g]);
#pragma unroll
                for (int g = 0; g < 4; ++g) D[3][g] = mm(tv0[g], P0.bd, D[3][g]);
#pragma unroll
                for (int g = 0; g < 4; ++g) D[3][g] = mm(tvv[g], P0.bb, D[3][g]);
            }
            // g1 <-> i2
#pragma unroll
            for (int x = 0; x < 4; ++x)
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    double t[4] = {D[x][0][r], D[x][1][r], D[x][2][r], D[x][3][r]};
                    swap_rows<32>(t[0], t[2]);
                    swap_rows<32>(t[1], t[3]);
                    swap_rows<16>(t[0], t[1]);
                    swap_rows<16>(t[2], t[3]);
#pragma unroll
                    for (int g = 0; g < 4; ++g) D[x][g][r] = t[g];
                }
            // the node pairs of two (i2, j2) tiles: contraction along xi_1 (the two chains in turn, so
            // that neither waits for its own last step), weights, entries to LDS
            auto put = [&](auto ic, auto jc, const f64x4 &v) {
                constexpr int i2 = decltype(ic)::value, j2 = decltype(jc)::value;
                typedef int32_t i32x4 __attribute__((ext_vector_type(4)));
                const double wa = wl[a0 + 16 * i2];
                const f64x2 w01 = *reinterpret_cast<const f64x2 *>(&wl[b1 + 16 * j2]),
                            w23 = *reinterpret_cast<const f64x2 *>(&wl[b1 + 16 * j2 + 2]);
                const double wb[4] = {w01.x, w01.y, w23.x, w23.y};
                const i32x4 sb = *reinterpret_cast<const i32x4 *>(&start8[b1 + 16 * j2]);   // j0 = 0..3
                const int sa = start8[a0 + 16 * i2];
                char *base = reinterpret_cast<char *>(st);
#pragma unroll
                for (int j0 = 0; j0 < 4; ++j0) {
                    const double val = v[j0] * (wa * wb[j0]);
                    if constexpr (i2 < j2) {
                        *reinterpret_cast<double *>(base + (sb[j0] + up) + 1152 * i2) = val;
                    } else if constexpr (i2 > j2) {
                        *reinterpret_cast<double *>(base + (sa + low) + (72 * j0 + 1152 * j2)) = val;
                    } else {
                        const int b0 = j0 + b1;   // against a0: the same i2 and j2
                        const int pos = a0 < b0 ? sb[j0] + up + 1152 * i2
                                                : a0 > b0 ? sa + low + (72 * j0 + 1152 * j2) : sb[j0] + dg + (72 * j0 + 1152 * j2);
                        if (!(diag && a0 > b0))
                            *reinterpret_cast<double *>(base + pos) = diag && a0 == b0 ? 0.5 * val : val;
                    }
                }
            };
            auto tile2 = [&](auto ic, auto jc, auto ic2, auto jc2) {
                constexpr int i = decltype(ic)::value, j = decltype(jc)::value;
                constexpr int i_ = decltype(ic2)::value, j_ = decltype(jc2)::value;
                f64x4 v = mm(D[0][i][j], P1.dd, Z), u = mm(D[0][i_][j_], P1.dd, Z);
                v = mm(D[1][i][j], P1.db, v);
                u = mm(D[1][i_][j_], P1.db, u);
                v = mm(D[2][i][j], P1.bd, v);
                u = mm(D[2][i_][j_], P1.bd, u);
                v = mm(D[3][i][j], P1.bb, v);
                u = mm(D[3][i_][j_], P1.bb, u);
                put(ic, jc, v);
                put(ic2, jc2, u);
            };
            auto tile1 = [&](auto ic, auto jc) {
                constexpr int i = decltype(ic)::value, j = decltype(jc)::value;
                f64x4 v = mm(D[0][i][j], P1.dd, Z);
                v = mm(D[1][i][j], P1.db, v);
                v = mm(D[2][i][j], P1.bd, v);
                put(ic, jc, mm(D[3][i][j], P1.bb, v));
            };
            using I0 = std::integral_constant<int, 0>;
            using I1 = std::integral_constant<int, 1>;
            using I2 = std::integral_constant<int, 2>;
            using I3 = std::integral_constant<int, 3>;
            tile2(I0{}, I0{}, I0{}, I1{});
            tile2(I1{}, I1{}, I0{}, I2{});
            tile2(I1{}, I2{}, I2{}, I2{});
            if (!diag) {
                tile2(I1{}, I0{}, I2{}, I0{});
                tile1(I2{}, I1{});
            }
            __syncthreads();
            // ---- step B ----
            tile2(I0{}, I3{}, I1{}, I3{});
            tile2(I2{}, I3{}, I3{}, I3{});
            if (!diag) {
                tile2(I3{}, I0{}, I3{}, I1{});
                tile1(I3{}, I2{});
            }
            const int64_t next = elem_at(s + 1);
            if (next >= 0) f.load(geo + next * REC, lane);
            __syncthreads();
            if (next < 0) break;
        }
        // the last second region leaves in a last step A
        __syncthreads();
    } else {
        const int sw = wv - CWAVES, cl = lane + 64 * sw;
        u32x2 rc[IDX ? WPL : 1];   // the dofs of four entries
        if (IDX) {
#pragma unroll
            for (int i = 0; i < WPL; ++i) rc[i] = *reinterpret_cast<const u32x2 *>(entry_tab.v + 4 * min(cl + SL * i, WORDS - 1));
        }
        int32_t *dof = dofs[sw];
        // entries [x0, x1) of the element at base
        auto store = [&](auto x0c, auto x1c, int64_t base) {
            constexpr int X0 = decltype(x0c)::value, X1 = decltype(x1c)::value;
            // uniform pointers and one lane offset: no address register per iteration
            const unsigned l2 = 2 * cl, l4 = 4 * cl;
            const double *src = st + X0;
            double *Ke = Kd + base + X0;
            constexpr int FULL = (X1 - X0) / (2 * SL), REST = (X1 - X0) % (2 * SL);
#pragma unroll 4
            for (int i = 0; i < FULL; ++i) {
                *reinterpret_cast<f64x2u *>(Ke + l2) = *reinterpret_cast<const f64x2 *>(src + l2);
                Ke += 2 * SL;
                src += 2 * SL;
            }
            if ((int)l2 < REST) *reinterpret_cast<f64x2u *>(Ke + l2) = *reinterpret_cast<const f64x2 *>(src + l2);
            if (IDX) {
                constexpr int I0 = X0 / 4 / SL, I1 = (X1 / 4 + SL - 1) / SL;
                int32_t *Re = Kr + base + 4 * SL * I0, *Ce = Kc + base + 4 * SL * I0;
#pragma unroll
                for (int i = I0; i < I1; ++i) {
                    // every lane's word lies in the region, but for the first and last iteration
                    const bool in = (SL * i >= X0 / 4 || cl + SL * i >= X0 / 4) &&
                                    (SL * (i + 1) <= X1 / 4 || cl + SL * i < X1 / 4);
                    // opaque: the words stay packed in their registers instead of being taken apart once
                    // for all elements and spilled (a reload would wait for the stores before it)
                    uint32_t e2[2] = {rc[i][0], rc[i][1]};
                    asm volatile("" : "+v"(e2[0]), "+v"(e2[1]));
                    if (in) {
                        i32x4u r, c;
#pragma unroll
                        for (int u = 0; u < 4; ++u) {
                            const uint32_t e = e2[u / 2] >> (16 * (u % 2));
                            r[u] = dof[e & 255];
                            c[u] = dof[(e >> 8) & 255];
                        }
                        *reinterpret_cast<i32x4u *>(Re + l4) = r;
                        *reinterpret_cast<i32x4u *>(Ce + l4) = c;
                    }
                    Re += 4 * SL;
                    Ce += 4 * SL;
                    __builtin_amdgcn_sched_barrier(0);   // keeps the iterations' registers apart
                }
            }
        };
        using C0 = std::integral_constant<int, 0>;
        using CS = std::integral_constant<int, SPLIT>;
        using CN = std::integral_constant<int, NDE>;
        int64_t prev = -1;   // COO offset of element e - 1
        int64_t gi = elem_at(0);
        for (int64_t s = 0; gi >= 0; ++s) {
            // loads of this element before the stores of step A, used after them
            const int32_t d = reinterpret_cast<const int32_t *>(geo + gi * REC + ODOF)[lane];
            const int64_t base = offs[gi];
            if (prev >= 0) store(CS{}, CN{}, prev);
#pragma unroll
            for (int c = 0; c < 3; ++c) dof[3 * lane + c] = d + c;
            wave_lds_sync();
            __syncthreads();
            store(C0{}, CS{}, base);
            prev = base;
            gi = elem_at(s + 1);
            __syncthreads();
        }
        store(CS{}, CN{}, prev);
        __syncthreads();
    }
}

int launch_elem_p3(const double *geo, const int64_t *offs, int32_t n, double lam, double mu, int cus, double *Kd,
                   int32_t *Kr, int32_t *Kc, hipStream_t st) {
    if (n <= 0) return 0;
    const unsigned grid = (unsigned)std::min<int64_t>(xcd_grid(n), (int64_t)std::max(cus / XCDS, 1) * XCDS);
    if (Kr)
        hipLaunchKernelGGL((elem_p3_kernel<true>), dim3(grid), dim3(p3::NTH), 0, st, geo, offs, n, lam, mu, Kd, Kr, Kc);
    else
        hipLaunchKernelGGL((elem_p3_kernel<false>), dim3(grid), dim3(p3::NTH), 0, st, geo, offs, n, lam, mu, Kd, Kr, Kc);
    YETI_HIP(hipGetLastError());
    return 0;
}

}  // namespace yeti
