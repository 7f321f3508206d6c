// csr.hip -- the CSR form of K_side + K_side^T built on the device, and its FP64 SpMV.
//
// Reference behaviour replaced: the callers of sys_linmat_lindef_static turn its COO output into
// scipy's canonical CSC/CSR and add the transpose, `(K_side + K_side^T)`
// (overlay/iga_model.py:391-395; benchs/volume_force/test_volume_force_3d.py:69-79).
//
// Pattern (once, from the resident connectivity): CP -> (element, local node) incidence,
// sorted by element; per CP row the sorted set of CPs sharing an element (3x3 block pattern).
// Values (every assembly): a block's contributions are read from the COO values and summed in
// ascending element order -- deterministic, no floating-point atomics. Two ways, chosen at creation
// (CsrValues): the element rows of a CP streamed whole (row_values_kernel), or block by block from a list
// of each block's contributions (csr_values_kernel). Blocks J >= I are summed and written twice, as (I, J)
// and, transposed, as (J, I); short rows of a model numbered at random sum every block. Scalar CSR: dof
// row 3 I + k holds, for each block column J of CP row I (ascending), the columns 3 J, 3 J + 1, 3 J + 2:
// scipy's canonical layout of the structural pattern.
#include <algorithm>
#include <vector>

#include "common.hpp"
#include "copy_out.hpp"

namespace yeti {
// declared in assembly.hip
struct AsmView {
    int32_t nb_cp;
    int32_t npatch;
    const int32_t *const *ien;      // per patch, device
    const int32_t *const *elems;    // per patch active elements (patch-local), device
    const int64_t *const *offs;     // per patch COO offsets, device
    const int32_t *nnode;           // per patch, host
    const int32_t *n_active;        // per patch, host
};
int asm_view(const yeti_asm *h, AsmView *v);
}  // namespace yeti

// how the values are gathered
enum CsrValues {
    CSR_ROWS,    // element rows
    CSR_SHORT,   // blocks J >= I, 16 lanes per CP row
    CSR_LIST,    // blocks J >= I, one thread each
    CSR_EVERY,   // every block, one thread each
};

struct yeti_csr {
    int32_t nb_cp = 0;
    int64_t nblocks = 0;                 // 3x3 blocks
    yeti::DevBuf<int64_t> bptr;          // [nb_cp + 1]
    yeti::DevBuf<int32_t> bcol;          // [nblocks]
    yeti::DevBuf<int32_t> bdiag;         // [nb_cp] place of the diagonal block in its row (the row's length: none)
    yeti::DevBuf<uint16_t> mirror;       // [nblocks] block (I, J), J > I: place of block (J, I) in row J
    CsrValues kind = CSR_LIST;
    // CSR_ROWS:
    int32_t upper = 0;                   // most blocks J >= I of a row
    int32_t sstride = 0;                 // slots per incidence
    yeti::DevBuf<int64_t> iptr;          // [nb_cp + 1] incidences of each CP
    yeti::DevBuf<int64_t> irow;          // (COO position of the element's row of a << 10) | a
    yeti::DevBuf<uint16_t> slots;        // [incidence][b]: place of block (I, J_b) after the diagonal, b <= a
    // otherwise:
    int64_t nlist = 0;                   // listed blocks, row by row (CSR_LIST: J >= I; else all)
    yeti::DevBuf<int64_t> uptr;          // [nb_cp + 1] CSR_LIST: first listed block of each row (else bptr)
    yeti::DevBuf<int32_t> urow;          // [nlist] CP row of each (CSR_SHORT: none)
    yeti::DevBuf<int64_t> cptr;          // [nlist + 1] contribution offsets
    yeti::DevBuf<int64_t> contrib;       // (COO position << 2) | kind
    yeti::DevBuf<int64_t> rowptr;        // scalar CSR [3 nb_cp + 1]
    yeti::DevBuf<int32_t> colind;        // scalar CSR [9 nblocks]
};

namespace yeti {

// ---- incidence --------------------------------------------------------------------------
__global__ void inc_count_kernel(const int32_t *ien, const int32_t *elems, int n_active, int nn,
                                 int32_t *count) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)n_active * nn) return;
    int ea = (int)(t / nn), a = (int)(t % nn);
    int e = elems[ea];
    atomicAdd(&count[ien[(int64_t)nn * e + a] - 1], 1);
}

// entry = (patch << 58) | (active index << 10) | local node ; sorted per CP afterwards
__global__ void inc_fill_kernel(const int32_t *ien, const int32_t *elems, int n_active, int nn, int patch,
                                const int64_t *ptr, int32_t *cursor, int64_t *ent) {
    int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)n_active * nn) return;
    int ea = (int)(t / nn), a = (int)(t % nn);
    int e = elems[ea];
    int cp = ien[(int64_t)nn * e + a] - 1;
    int slot = atomicAdd(&cursor[cp], 1);
    ent[ptr[cp] + slot] = ((int64_t)patch << 58) | ((int64_t)ea << 10) | a;
}

__global__ void inc_sort_kernel(int32_t nb_cp, const int64_t *ptr, int64_t *ent) {
    int cp = blockIdx.x * blockDim.x + threadIdx.x;
    if (cp >= nb_cp) return;
    int64_t b = ptr[cp], n = ptr[cp + 1] - b;
    for (int64_t i = 1; i < n; ++i) {          // insertion sort: lists are short (<= 729)
        int64_t v = ent[b + i];
        int64_t j = i - 1;
        while (j >= 0 && ent[b + j] > v) {
            ent[b + j + 1] = ent[b + j];
            --j;
        }
        ent[b + j + 1] = v;
    }
}

// exclusive scan of int32/int64 counts into int64 offsets (single-pass over blocks of 1024,
// then block sums, then add): three small kernels.
template <typename T>
__global__ void scan_block_kernel(const T *in, int64_t n, int64_t *out, int64_t *bsum) {
    __shared__ int64_t s[1024];
    int64_t i = (int64_t)blockIdx.x * 1024 + threadIdx.x;
    int64_t v = i < n ? (int64_t)in[i] : 0;
    s[threadIdx.x] = v;
    __syncthreads();
    for (int o = 1; o < 1024; o <<= 1) {
        int64_t add = threadIdx.x >= (unsigned)o ? s[threadIdx.x - o] : 0;
        __syncthreads();
        s[threadIdx.x] += add;
        __syncthreads();
    }
    if (i < n) out[i] = s[threadIdx.x] - v;
    if (i == n - 1) out[n] = s[threadIdx.x];
    if (threadIdx.x == 1023) bsum[blockIdx.x] = s[1023];
}

__global__ void scan_add_kernel(int64_t *out, int64_t n, const int64_t *boff) {
    int64_t i = (int64_t)blockIdx.x * 1024 + threadIdx.x;
    if (i < n) out[i] += boff[blockIdx.x];
    if (i == n - 1) out[n] += boff[blockIdx.x];
}

// exclusive scan of n values into out[0..n], out[n] = total. Host-driven recursion.
template <typename T>
static int exclusive_scan(const T *in, int64_t n, int64_t *out, hipStream_t st) {
    if (n == 0) {
        YETI_HIP(hipMemsetAsync(out, 0, sizeof(int64_t), st));
        return 0;
    }
    int64_t nb = (n + 1023) / 1024;
    DevBuf<int64_t> bsum, boff;
    YETI_HIP(bsum.alloc(nb));
    YETI_HIP(boff.alloc(nb + 1));
    hipLaunchKernelGGL(scan_block_kernel<T>, dim3((unsigned)nb), dim3(1024), 0, st, in, n, out, bsum.p);
    YETI_HIP(hipGetLastError());
    if (nb > 1) {   // one block needs no carry; recursing on it would never end
        int rc = exclusive_scan<int64_t>(bsum.p, nb, boff.p, st);
        if (rc) return rc;
        hipLaunchKernelGGL(scan_add_kernel, dim3((unsigned)nb), dim3(1024), 0, st, out, n, boff.p);
        YETI_HIP(hipGetLastError());
    }
    return 0;
}

static int read_back(void *host, const void *dev, size_t bytes, hipStream_t st) {
    YETI_HIP(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, st));
    YETI_HIP(hipStreamSynchronize(st));
    return 0;
}

// ---- block pattern ----------------------------------------------------------------------
struct PatchIen {
    const int32_t *ien[8];
    const int32_t *elems[8];
    const int64_t *offs[8];
    int32_t nn[8];
};

constexpr int HASH = 4096;     // per-wave open-addressing set (>= 2 x 729 unique neighbours)

// One wave per CP row: collect the CPs of every element touching the row into an LDS hash set,
// then (pass 2) sort them into the row's block columns.
template <bool FILL>
__global__ void __launch_bounds__(256) row_pattern_kernel(int32_t nb_cp, const int64_t *inc_ptr,
                                                          const int64_t *inc, PatchIen pi,
                                                          int32_t *row_len, const int64_t *bptr,
                                                          int32_t *bcol, int32_t *overflow) {
    __shared__ int32_t table[4][HASH];
    __shared__ int32_t cnt[4];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int row = blockIdx.x * 4 + w;
    int32_t *T = table[w];
    for (int i = lane; i < HASH; i += 64) T[i] = -1;
    if (lane == 0) cnt[w] = 0;
    __syncthreads();
    if (row < nb_cp) {
        for (int64_t k = inc_ptr[row]; k < inc_ptr[row + 1]; ++k) {
            int64_t en = inc[k];
            int patch = (int)(en >> 58), ea = (int)((en >> 10) & ((1LL << 48) - 1));
            int nn = pi.nn[patch];
            int e = pi.elems[patch][ea];
            const int32_t *ie = pi.ien[patch] + (int64_t)nn * e;
            for (int b = lane; b < nn; b += 64) {
                int32_t J = ie[b] - 1;
                uint32_t h = ((uint32_t)J * 2654435761u) & (HASH - 1);
                int probe = 0;
                for (; probe < HASH; ++probe) {        // bounded: the table holds HASH keys
                    int32_t old = atomicCAS(&T[h], -1, J);
                    if (old == -1) {
                        atomicAdd(&cnt[w], 1);
                        break;
                    }
                    if (old == J) break;
                    h = (h + 1) & (HASH - 1);
                }
                if (probe == HASH) atomicOr(overflow, 1);
            }
        }
    }
    __syncthreads();
    const bool live = row < nb_cp;
    const int n = cnt[w];
    if (!FILL) {
        if (live && lane == 0) {
            row_len[row] = n;
            if (n > 1024) atomicOr(overflow, 1);   // more neighbours than the sort buffer holds
        }
        return;
    }
    // compact then rank-sort (n <= 729): each lane ranks its entries against all others.
    // Every wave reaches every barrier (rows past the end only skip the writes).
    __shared__ int32_t comp[4][1024];
    __shared__ int32_t pos[4];
    if (lane == 0) pos[w] = 0;
    __syncthreads();
    for (int i = lane; i < HASH; i += 64) {
        int32_t v = T[i];
        if (v >= 0) {
            int slot = atomicAdd(&pos[w], 1);
            if (slot < 1024) comp[w][slot] = v;
        }
    }
    __syncthreads();
    if (!live || n > 1024) return;
    const int64_t out = bptr[row];
    for (int i = lane; i < n; i += 64) {
        int32_t v = comp[w][i];
        int r = 0;
        for (int j = 0; j < n; ++j) r += comp[w][j] < v;
        bcol[out + r] = v;
    }
}

// Per row: count (pass 1) or write (pass 2) the contributions of its blocks from place `first` on (bdiag, or
// 0 when null), in element order; block i of the row is number lptr[row] + i of the list, or
// lptr[row] + i - first when `dense`.
// kind 0: block (a, b) stored as is (a < b); 1: stored as (b, a) (a > b, transpose);
// 2: diagonal block (a == b), stored as its 6 upper entries with the diagonal halved.
template <bool FILL>
__global__ void __launch_bounds__(64) contrib_kernel(int32_t nb_cp, const int64_t *inc_ptr, const int64_t *inc,
                                                     PatchIen pi, const int64_t *bptr, const int32_t *bcol,
                                                     const int32_t *bdiag, const int64_t *lptr, bool dense,
                                                     int32_t *bcount, const int64_t *cptr, int64_t *contrib) {
    __shared__ int32_t cur[1024];
    const int row = blockIdx.x, lane = threadIdx.x;
    if (row >= nb_cp) return;
    const int64_t b0 = bptr[row];
    const int first = bdiag ? bdiag[row] : 0;
    const int64_t u0 = lptr[row] - (dense ? first : 0);
    const int nb = (int)(bptr[row + 1] - b0);
    if (nb > 1024) return;      // rejected by the pattern pass (overflow flag)
    for (int i = lane; i < nb; i += 64) cur[i] = 0;
    __syncthreads();
    for (int64_t k = inc_ptr[row]; k < inc_ptr[row + 1]; ++k) {
        int64_t en = inc[k];
        int patch = (int)(en >> 58), ea = (int)((en >> 10) & ((1LL << 48) - 1)), a = (int)(en & 1023);
        int nn = pi.nn[patch];
        int e = pi.elems[patch][ea];
        int64_t base = pi.offs[patch][ea];
        const int32_t *ie = pi.ien[patch] + (int64_t)nn * e;
        for (int b = lane; b < nn; b += 64) {
            int32_t J = ie[b] - 1;
            int lo = 0, hi = nb - 1;       // binary search of J among the row's sorted columns
            while (lo < hi) {
                int mid = (lo + hi) >> 1;
                if (bcol[b0 + mid] < J) lo = mid + 1; else hi = mid;
            }
            if (lo < first) continue;
            // one contribution per (element, block): no two lanes hit the same block here
            int slot = cur[lo]++;
            if (FILL) {
                int64_t code;
                if (a < b) code = ((base + 9LL * b * (b - 1) / 2 + 6LL * b + 9LL * a) << 2) | 0;
                else if (a > b) code = ((base + 9LL * a * (a - 1) / 2 + 6LL * a + 9LL * b) << 2) | 1;
                else code = ((base + 9LL * a * (a - 1) / 2 + 6LL * a + 9LL * a) << 2) | 2;
                contrib[cptr[u0 + lo] + slot] = code;
            }
        }
        __syncthreads();
    }
    if (!FILL)
        for (int i = (dense ? first : 0) + lane; i < nb; i += 64) bcount[u0 + i] = cur[i];
}

// Number of blocks J >= I per row; flags[0]: the most of a row.
__global__ void __launch_bounds__(256) upper_count_kernel(int32_t nb_cp, const int64_t *bptr, const int32_t *bdiag,
                                                          int32_t *count, int32_t *flags) {
    const int64_t I = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int n = 0;
    if (I < nb_cp) count[I] = n = (int32_t)(bptr[I + 1] - bptr[I]) - bdiag[I];
    for (int o = 32; o > 0; o >>= 1) n = max(n, __shfl_xor(n, o, 64));
    if ((threadIdx.x & 63) == 0) atomicMax(&flags[0], n);
}

// flags[1]: set when local nodes of an active element are not numbered strictly against their CPs
__global__ void __launch_bounds__(256) order_kernel(const int32_t *ien, const int32_t *elems, int n_active, int nn,
                                                    int32_t *flags) {
    const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= (int64_t)n_active * nn || t % nn == 0) return;
    const int32_t *ie = ien + (int64_t)nn * elems[t / nn] + t % nn;
    if (ie[-1] <= ie[0]) flags[1] = 1;   // every writer writes the same
}

// CP row of each listed block
__global__ void __launch_bounds__(256) list_rows_kernel(int32_t nb_cp, const int64_t *lptr, int32_t *urow) {
    const int64_t I = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (I >= nb_cp) return;
    for (int64_t x = lptr[I] + (threadIdx.x & 63); x < lptr[I + 1]; x += 64) urow[x] = (int32_t)I;
}

// The diagonal block's place in each row, and for every block above it the place of its transpose.
__global__ void __launch_bounds__(256) mirror_kernel(int32_t nb_cp, const int64_t *__restrict__ bptr,
                                                     const int32_t *__restrict__ bcol, int32_t *__restrict__ bdiag,
                                                     uint16_t *__restrict__ mirror) {
    const int64_t I = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (I >= nb_cp) return;
    const int lane = threadIdx.x & 63;
    auto place = [&](int64_t row, int32_t col) {   // first column >= col
        int lo = 0, hi = (int)(bptr[row + 1] - bptr[row]);
        const int32_t *c = bcol + bptr[row];
        while (lo < hi) {
            const int mid = (lo + hi) >> 1;
            if (c[mid] < col) lo = mid + 1; else hi = mid;
        }
        return lo;
    };
    const int jd = place(I, (int32_t)I), nb = (int)(bptr[I + 1] - bptr[I]);
    if (lane == 0) bdiag[I] = jd;
    for (int j = jd + lane; j < nb; j += 64) mirror[bptr[I] + j] = (uint16_t)place(bcol[bptr[I] + j], (int32_t)I);
}

// Of the blocks above the diagonal of some rows (one per workgroup, spread over the model): flags[2] their
// number, flags[3] how many have their transpose right after that of the block in the row before.
__global__ void __launch_bounds__(64) adjacent_kernel(int32_t nb_cp, const int64_t *bptr, const int32_t *bcol,
                                                      const int32_t *bdiag, const uint16_t *mirror, int32_t *flags) {
    const int64_t I = (int64_t)blockIdx.x * nb_cp / gridDim.x, b0 = bptr[I];
    const int nb = (int)(bptr[I + 1] - b0);
    int n = 0, adj = 0;
    for (int j = bdiag[I] + 1 + threadIdx.x; j < nb; j += 64) {
        const int jm = mirror[b0 + j];
        ++n;
        if (jm > 0 && bcol[bptr[bcol[b0 + j]] + jm - 1] == I - 1) ++adj;
    }
    for (int o = 32; o > 0; o >>= 1) {
        n += __shfl_xor(n, o, 64);
        adj += __shfl_xor(adj, o, 64);
    }
    if (threadIdx.x == 0) {
        atomicAdd(&flags[2], n);
        atomicAdd(&flags[3], adj);
    }
}

__global__ void scalar_pattern_kernel(int32_t nb_cp, const int64_t *bptr, const int32_t *bcol,
                                      int64_t *rowptr, int32_t *colind) {
    int I = blockIdx.x * blockDim.x + threadIdx.x;
    if (I > nb_cp) return;
    if (I == nb_cp) {
        rowptr[3 * (int64_t)nb_cp] = 9 * bptr[nb_cp];
        return;
    }
    int64_t b0 = bptr[I];
    int nb = (int)(bptr[I + 1] - b0);
    for (int k = 0; k < 3; ++k) {
        int64_t r0 = 9 * b0 + 3LL * k * nb;
        rowptr[3 * (int64_t)I + k] = r0;
        for (int j = 0; j < nb; ++j) {
            int32_t J = bcol[b0 + j];
            colind[r0 + 3 * j + 0] = 3 * J;
            colind[r0 + 3 * j + 1] = 3 * J + 1;
            colind[r0 + 3 * j + 2] = 3 * J + 2;
        }
    }
}

// ---- values ------------------------------------------------------------------------------
// CSR_SHORT: SHORT_ROW lanes per CP row, one on each of its blocks J >= I (at most SHORT_ROW, p = 1: 14);
// else one thread per listed block (I, J). A block's contributions are summed in element order, UC of
// them in flight. Blocks J >= I are written also, transposed, as (J, I), so that each COO value is read
// once; each XCD takes one run of the list, so that the transposed blocks of neighbouring rows meet in
// its L2. CSR_EVERY lists every block: with control points numbered at random the transposes
// are 24-byte pieces of separate lines, which costs more than reading a short row's two or three
// contributions twice (random numbering, 72^3 p = 1: 1626 us mirrored, 892 us by itself; p = 2 at 34^3
// 882 us mirrored, 1115 us by itself). Blocks are dealt one by one, not row by row: rows differ in their
// blocks J >= I (random numbering: from none to all), and a small model has more blocks than lanes
// (against 64 lanes per row: 4^3 p = 4 111 -> 38 us, 8^3 p = 4 numbered at random 851 -> 222 us).
constexpr int SHORT_ROW = 16;

typedef double f64x2u __attribute__((ext_vector_type(2), aligned(8)));

template <int VT, int KIND>
__global__ void __launch_bounds__(VT) csr_values_kernel(int64_t nitem, const int64_t *__restrict__ lptr,
                                                        const int32_t *__restrict__ urow,
                                                        const int64_t *__restrict__ bptr,
                                                        const int32_t *__restrict__ bcol,
                                                        const int32_t *__restrict__ bdiag,
                                                        const uint16_t *__restrict__ mirror,
                                                        const int64_t *__restrict__ cptr,
                                                        const int64_t *__restrict__ contrib,
                                                        const double *__restrict__ Kdata,
                                                        double *__restrict__ vals) {
    constexpr int UC = 2;
    constexpr bool MIRROR = KIND != CSR_EVERY;
    int64_t x = xcd_element(blockIdx.x, (nitem + VT - 1) / VT) * VT + threadIdx.x;
    if (x >= nitem) return;
    const int32_t I = KIND == CSR_SHORT ? (int32_t)(x / SHORT_ROW) : urow[x];
    const int64_t b0 = bptr[I];
    const int nb = (int)(bptr[I + 1] - b0);
    int j;
    if (KIND == CSR_SHORT) {
        j = bdiag[I] + (int)(x % SHORT_ROW);
        if (j >= nb) return;
        x = b0 + j;
    } else {
        j = (int)(x - lptr[I]) + (KIND == CSR_LIST ? bdiag[I] : 0);
    }
    double v[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};   // v[k][l] = v[3k + l]
    const int32_t J = MIRROR ? bcol[b0 + j] : 0;
    const int jm = MIRROR ? mirror[b0 + j] : 0;
    const int64_t c1 = cptr[x + 1];
    for (int64_t c = cptr[x]; c < c1; c += UC) {
        double s[UC][9];
        int kind[UC];
#pragma unroll
        for (int u = 0; u < UC; ++u) {
            const int64_t code = contrib[min(c + u, c1 - 1)];
            kind[u] = c + u < c1 ? (int)(code & 3) : 3;
            const double *p = Kdata + (code >> 2);
            f64x2u t[4] = {};
            t[0] = *reinterpret_cast<const f64x2u *>(p);
            t[1] = *reinterpret_cast<const f64x2u *>(p + 2);
            t[2] = *reinterpret_cast<const f64x2u *>(p + 4);
            s[u][8] = 0.0;
            if ((code & 3) != 2) {   // a diagonal block has six entries
                t[3] = *reinterpret_cast<const f64x2u *>(p + 6);
                s[u][8] = p[8];
            }
#pragma unroll
            for (int y = 0; y < 8; ++y) s[u][y] = t[y / 2][y % 2];
        }
#pragma unroll
        for (int u = 0; u < UC; ++u) {
            const double *q = s[u];
            if (kind[u] < 2) {   // stored (k, l) at q[k + 3 l]; kind 1: the transpose of the stored block
                const bool tr = kind[u] == 1;
#pragma unroll
                for (int k = 0; k < 3; ++k)
#pragma unroll
                    for (int l = 0; l < 3; ++l) v[3 * k + l] += tr ? q[l + 3 * k] : q[k + 3 * l];
            } else if (kind[u] == 2) {   // diagonal block: side + side^T, (0,0) (0,1) (1,1) (0,2) (1,2) (2,2)
                v[0] += 2.0 * q[0]; v[4] += 2.0 * q[2]; v[8] += 2.0 * q[5];
                v[1] += q[1]; v[3] += q[1];
                v[2] += q[3]; v[6] += q[3];
                v[5] += q[4]; v[7] += q[4];
            }
        }
    }
    double *o = vals + 9 * b0 + 3 * j;
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int l = 0; l < 3; ++l) o[3LL * k * nb + l] = v[3 * k + l];
    if (MIRROR && J != I) {
        const int64_t m0 = bptr[J];
        const int mb = (int)(bptr[J + 1] - m0);
        o = vals + 9 * m0 + 3 * jm;
#pragma unroll
        for (int k = 0; k < 3; ++k)
#pragma unroll
            for (int l = 0; l < 3; ++l) o[3LL * k * mb + l] = v[3 * l + k];
    }
}

// Values by element rows. Local nodes are numbered against the CPs (b < a holds CPs J_b > I_a), so the
// 9 a + 6 COO entries of an element's row a are exactly its contributions to the blocks J >= I of the
// CP I of a: one wave per CP row streams those runs whole, element after element, into the row's
// blocks in LDS (entry x of a run goes to entry x mod 9 of block x / 9, through the incidence's slots).
// Every address is added to by one wave in a fixed order. Then the row is written with consecutive
// lanes on consecutive values, and its transposes. Loads run one group of RG ahead.
constexpr int ROW_WAVES = 2;   // rows per workgroup (LDS: 12 waves per CU at p = 3)

template <int NSL>   // slots per lane: 1 up to 64 nodes per element, 2 up to 128
__global__ void __launch_bounds__(64 * ROW_WAVES)
row_values_kernel(int32_t nb_cp, int32_t upper, int32_t sstride, const int64_t *__restrict__ bptr,
                  const int32_t *__restrict__ bcol, const int32_t *__restrict__ bdiag,
                  const uint16_t *__restrict__ mirror, const int64_t *__restrict__ iptr,
                  const int64_t *__restrict__ irow, const uint16_t *__restrict__ slots,
                  const double *__restrict__ Kdata, double *__restrict__ vals) {
    constexpr int RG = 5;
    extern __shared__ double racc[];
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    double *acc = racc + wv * 9 * upper;
    const int64_t I = xcd_element(blockIdx.x, ((int64_t)nb_cp + ROW_WAVES - 1) / ROW_WAVES) * ROW_WAVES + wv;
    if (I >= nb_cp) return;   // waves of a workgroup share nothing
    const int64_t b0 = bptr[I];
    const int nb = (int)(bptr[I + 1] - b0), jd = bdiag[I], nu = nb - jd;
    for (int x = lane; x < 9 * nu; x += 64) acc[x] = 0.0;
    wave_lds_sync();
    const int64_t k1 = iptr[I + 1];
    int64_t k = iptr[I], code = k < k1 ? irow[k] : 0, next = k + 1 < k1 ? irow[k + 1] : 0;
    int x0 = 0;
    double v[RG];
    uint16_t sl[NSL] = {};   // slots of b = lane, lane + 64
    auto fetch = [&](int64_t kk, int64_t cd, int xx, double (&o)[RG], uint16_t (&so)[NSL]) {
        const int a = (int)(cd & 1023), len = 9 * a + 6;
        const double *run = Kdata + (cd >> 10);
#pragma unroll
        for (int u = 0; u < RG; ++u) {
            const int x = xx + lane + 64 * u;
            o[u] = x < len ? run[x] : 0.0;
        }
        if (xx == 0) {
            const uint16_t *sp = slots + kk * sstride;
#pragma unroll
            for (int h = 0; h < NSL; ++h) so[h] = lane + 64 * h <= a ? sp[lane + 64 * h] : 0;
        }
    };
    if (k < k1) fetch(k, code, 0, v, sl);
    while (k < k1) {
        const int a = (int)(code & 1023), len = 9 * a + 6;
        // the group after this one
        int64_t kn = k, cn = code;
        int xn = x0 + 64 * RG;
        if (xn >= len) {
            ++kn;
            xn = 0;
            cn = next;   // loaded an incidence ahead of its run
            next = kn + 1 < k1 ? irow[kn + 1] : 0;
        }
        double w[RG];
        uint16_t sn[NSL];
#pragma unroll
        for (int h = 0; h < NSL; ++h) sn[h] = sl[h];
        if (kn < k1) fetch(kn, cn, xn, w, sn);
#pragma unroll
        for (int u = 0; u < RG; ++u) {
            // uniform: the run's last group may be short (at p = 4 the branches cost more than they save)
            if (NSL == 1 && x0 + 64 * u >= len) break;
            const int x = x0 + lane + 64 * u;
            const int b = (x * 7282) >> 16;   // x / 9 for x < 7282
            int slot = __shfl((int)sl[0], b & 63, 64);
            if (NSL > 1) {
                const int s1 = __shfl((int)sl[NSL - 1], b & 63, 64);
                slot = b < 64 ? slot : s1;
            }
            double *p = acc + 9 * slot;
            const int m = x - 9 * b;
            if (b < a) {
                p[m] += v[u];
            } else if (x < len) {   // diagonal block: (0,0) (0,1) (1,1) (0,2) (1,2) (2,2), side + side^T
                const int kk = (0x210100 >> (4 * m)) & 15, ll = (0x222110 >> (4 * m)) & 15;
                p[3 * kk + ll] += kk == ll ? 2.0 * v[u] : v[u];
                if (kk != ll) p[3 * ll + kk] += v[u];
            }
        }
        wave_lds_sync();   // other lanes may add the next run's entries to these addresses (a run's are distinct)
#pragma unroll
        for (int u = 0; u < RG; ++u) v[u] = w[u];
#pragma unroll
        for (int h = 0; h < NSL; ++h) sl[h] = sn[h];
        k = kn;
        code = cn;
        x0 = xn;
    }
    wave_lds_sync();
    // row I: 3 nu consecutive values for each dof
    for (int kk = 0; kk < 3; ++kk) {
        double *o = vals + 9 * b0 + 3LL * kk * nb + 3 * jd;
        for (int y = lane; y < 3 * nu; y += 64) {
            const int j = y / 3;
            o[y] = acc[9 * j + 3 * kk + (y - 3 * j)];
        }
    }
    // the transposes, in the rows of the blocks' columns
    for (int j = 1 + lane; j < nu; j += 64) {
        const int32_t J = bcol[b0 + jd + j];
        const int64_t m0 = bptr[J];
        const int mb = (int)(bptr[J + 1] - m0);
        double *o = vals + 9 * m0 + 3 * (int)mirror[b0 + jd + j];
#pragma unroll
        for (int kk = 0; kk < 3; ++kk)
#pragma unroll
            for (int l = 0; l < 3; ++l) o[3LL * kk * mb + l] = acc[9 * j + 3 * l + kk];
    }
}

// Per CP row: the element rows and slots of its incidences.
__global__ void __launch_bounds__(64) slot_kernel(int32_t nb_cp, const int64_t *inc_ptr, const int64_t *inc, PatchIen pi,
                                                  const int64_t *bptr, const int32_t *bcol, const int32_t *bdiag,
                                                  int32_t sstride, int64_t *irow, uint16_t *slots) {
    const int row = blockIdx.x, lane = threadIdx.x;
    if (row >= nb_cp) return;
    const int64_t b0 = bptr[row];
    const int nb = (int)(bptr[row + 1] - b0), jd = bdiag[row];
    for (int64_t k = inc_ptr[row]; k < inc_ptr[row + 1]; ++k) {
        const int64_t en = inc[k];
        const int patch = (int)(en >> 58), ea = (int)((en >> 10) & ((1LL << 48) - 1)), a = (int)(en & 1023);
        const int nn = pi.nn[patch];
        const int32_t *ie = pi.ien[patch] + (int64_t)nn * pi.elems[patch][ea];
        if (lane == 0) irow[k] = ((pi.offs[patch][ea] + (9LL * a * a + 3LL * a) / 2) << 10) | a;
        for (int b = lane; b <= a; b += 64) {
            const int32_t J = ie[b] - 1;
            int lo = jd, hi = nb - 1;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (bcol[b0 + mid] < J) lo = mid + 1; else hi = mid;
            }
            slots[k * sstride + b] = (uint16_t)(lo - jd);
        }
    }
}

// ---- SpMV by nodal 3x3 blocks: one wave per CP row ---------------------------------------
// The three dof rows 3I, 3I+1, 3I+2 of a CP share their block columns; row 3I+k of block j is
// vals[9 b0 + 3 k nb + 3 j + l], l = 0..2 (b0 = bptr[I], nb blocks in the row). A lane takes
// blocks j = lane, lane + 64, ...: it reads the block column once (4 bytes per 9 entries instead
// of 4 per entry), x at 3J..3J+2, and 3 x 3 consecutive values, consecutive lanes on consecutive
// 24-byte runs. Rows of a masked-out dof give 0. MODE bits: 1 = |vals| |x| (the FP64 rounding
// bound of a product), 2 = block partials of x . y for the PCG.
template <int MODE>
__global__ void __launch_bounds__(256) block_spmv_kernel(int32_t nb_cp, const int64_t *__restrict__ bptr,
                                                         const int32_t *__restrict__ bcol,
                                                         const double *__restrict__ vals,
                                                         const double *__restrict__ x,
                                                         const uint8_t *__restrict__ mask,
                                                         double *__restrict__ y, double *__restrict__ partial,
                                                         const int32_t *__restrict__ pred) {
    if (pred && *pred == 0) return;   // predicated launch (device-side solver control)
    constexpr bool ABS = (MODE & 1) != 0, DOT = (MODE & 2) != 0;
    __shared__ double sh[4];
    const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
    double acc = 0.0;
    for (int64_t I = (int64_t)blockIdx.x * 4 + w; I < nb_cp; I += (int64_t)gridDim.x * 4) {
        const int64_t b0 = bptr[I];
        const int nb = (int)(bptr[I + 1] - b0);
        const double *v0 = vals + 9 * b0;
        double s0 = 0.0, s1 = 0.0, s2 = 0.0;
        for (int j = lane; j < nb; j += 64) {
            const int64_t J = bcol[b0 + j];
            double x0 = x[3 * J], x1 = x[3 * J + 1], x2 = x[3 * J + 2];
            const double *a0 = v0 + 3 * j, *a1 = a0 + 3 * (int64_t)nb, *a2 = a1 + 3 * (int64_t)nb;
            double c[9] = {a0[0], a0[1], a0[2], a1[0], a1[1], a1[2], a2[0], a2[1], a2[2]};
            if (ABS) {
                x0 = fabs(x0); x1 = fabs(x1); x2 = fabs(x2);
#pragma unroll
                for (int t = 0; t < 9; ++t) c[t] = fabs(c[t]);
            }
            s0 += c[0] * x0 + c[1] * x1 + c[2] * x2;
            s1 += c[3] * x0 + c[4] * x1 + c[5] * x2;
            s2 += c[6] * x0 + c[7] * x1 + c[8] * x2;
        }
        for (int o = 32; o > 0; o >>= 1) {
            s0 += __shfl_xor(s0, o, 64);
            s1 += __shfl_xor(s1, o, 64);
            s2 += __shfl_xor(s2, o, 64);
        }
        if (lane == 0) {
            double r[3] = {s0, s1, s2};
#pragma unroll
            for (int k = 0; k < 3; ++k) {
                if (mask && !mask[3 * I + k]) r[k] = 0.0;
                y[3 * I + k] = r[k];
                if (DOT) acc += r[k] * x[3 * I + k];
            }
        }
    }
    if (DOT) {
        double v = lane == 0 ? acc : 0.0;
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
        if (lane == 0) sh[w] = v;
        __syncthreads();
        if (threadIdx.x == 0) partial[blockIdx.x] = sh[0] + sh[1] + sh[2] + sh[3];
    }
}

constexpr int SPMV_MAX_BLOCKS = 4096;

// y = mask .* (A x) (mode 0), the same with |A| |x| (mode 1), or mode 2: y = mask .* (A x) and
// partial[b] = the grid block's share of x . y (grid of *nparts blocks, at most
// SPMV_MAX_BLOCKS). mask may be null.
int csr_block_spmv(const yeti_csr *c, const double *vals, const double *x, const uint8_t *mask, double *y,
                   double *partial, int mode, int *nparts, hipStream_t st, const int32_t *pred) {
    if (c->nb_cp <= 0) return 0;
    const unsigned g = (unsigned)std::min<int64_t>(SPMV_MAX_BLOCKS, ((int64_t)c->nb_cp + 3) / 4);
    if (nparts) *nparts = (int)g;
    switch (mode) {
    case 0: hipLaunchKernelGGL(block_spmv_kernel<0>, dim3(g), dim3(256), 0, st, c->nb_cp, c->bptr.p, c->bcol.p, vals, x,
                               mask, y, partial, pred); break;
    case 1: hipLaunchKernelGGL(block_spmv_kernel<1>, dim3(g), dim3(256), 0, st, c->nb_cp, c->bptr.p, c->bcol.p, vals, x,
                               mask, y, partial, pred); break;
    default: hipLaunchKernelGGL(block_spmv_kernel<2>, dim3(g), dim3(256), 0, st, c->nb_cp, c->bptr.p, c->bcol.p, vals,
                                x, mask, y, partial, pred); break;
    }
    YETI_HIP(hipGetLastError());
    return 0;
}

int64_t csr_nrows(const yeti_csr *c) { return 3 * (int64_t)c->nb_cp; }
const int64_t *csr_rowptr_dev(const yeti_csr *c) { return c->rowptr.p; }
const int32_t *csr_colind_dev(const yeti_csr *c) { return c->colind.p; }

}  // namespace yeti

using namespace yeti;

namespace yeti {
// ---- canonical form: scipy's K_side + K_side^T drops the entries that sum to exactly 0 ----
__global__ void __launch_bounds__(256) nz_count_kernel(int64_t nrows, const int64_t *rowptr, const double *vals,
                                                       int32_t *cnt) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nrows) return;
    int32_t n = 0;
    for (int64_t k = rowptr[r]; k < rowptr[r + 1]; ++k) n += vals[k] != 0.0;
    cnt[r] = n;
}

__global__ void __launch_bounds__(256) nz_compact_kernel(int64_t nrows, const int64_t *rowptr, const int32_t *colind,
                                                         const double *vals, const int64_t *newptr,
                                                         int32_t *colind_out, double *vals_out) {
    const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (r >= nrows) return;
    int64_t o = newptr[r];
    for (int64_t k = rowptr[r]; k < rowptr[r + 1]; ++k) {
        const double v = vals[k];
        if (v != 0.0) {
            colind_out[o] = colind[k];
            vals_out[o] = v;
            ++o;
        }
    }
}

}  // namespace yeti

extern "C" {

int32_t yeti_csr_drop_zeros(const yeti_csr *c, const double *vals_dev, int64_t *rowptr_out, int32_t *colind_out,
                            double *vals_out, int64_t *nnz_out, void *stream) {
    if (!c || !vals_dev || !rowptr_out || !colind_out || !vals_out || !nnz_out)
        return set_error(YETI_ERR_INVALID_ARGUMENT, "null argument");
    hipStream_t st = (hipStream_t)stream;
    const int64_t nrows = 3 * (int64_t)c->nb_cp;
    DevBuf<int32_t> cnt;
    YETI_HIP(cnt.alloc(std::max<int64_t>(nrows, 1)));
    const unsigned g = (unsigned)((nrows + 255) / 256);
    if (nrows > 0) {
        hipLaunchKernelGGL(nz_count_kernel, dim3(g), dim3(256), 0, st, nrows, c->rowptr.p, vals_dev, cnt.p);
        YETI_HIP(hipGetLastError());
    }
    int rc = exclusive_scan<int32_t>(cnt.p, nrows, rowptr_out, st);
    if (rc) return rc;
    if (nrows > 0) {
        hipLaunchKernelGGL(nz_compact_kernel, dim3(g), dim3(256), 0, st, nrows, c->rowptr.p, c->colind.p, vals_dev,
                           (const int64_t *)rowptr_out, colind_out, vals_out);
        YETI_HIP(hipGetLastError());
    }
    YETI_HIP(hipMemcpyAsync(nnz_out, rowptr_out + nrows, sizeof(int64_t), hipMemcpyDeviceToHost, st));
    YETI_HIP(hipStreamSynchronize(st));
    return 0;
}

int32_t yeti_csr_create_as(const yeti_asm *h, int32_t kind, void *stream, yeti_csr **out) {
    if (!h || !out) return set_error(YETI_ERR_INVALID_ARGUMENT, "null argument");
    *out = nullptr;
    if (kind < -1 || kind > CSR_EVERY) return set_error(YETI_ERR_INVALID_ARGUMENT, "CSR: no way %d to gather the values", kind);
    hipStream_t st = (hipStream_t)stream;
    AsmView v;
    int rc = asm_view(h, &v);
    if (rc) return rc;
    if (v.npatch > 8) return set_error(YETI_ERR_INVALID_ARGUMENT, "CSR build supports up to 8 patches");
    auto *c = new yeti_csr();
    auto fail = [&](int code) {
        delete c;
        return code;
    };
    c->nb_cp = v.nb_cp;
    PatchIen pi{};
    for (int p = 0; p < v.npatch; ++p) {
        pi.ien[p] = v.ien[p];
        pi.elems[p] = v.elems[p];
        pi.offs[p] = v.offs[p];
        pi.nn[p] = v.nnode[p];
        if (v.nnode[p] > 729) return fail(set_error(YETI_ERR_UNSUPPORTED_DEGREE, "CSR: too many nodes per element"));
    }
    DevBuf<int32_t> cnt, cursor, rowlen, bcount, oflow, flags;
    DevBuf<int64_t> inc_ptr, inc;
    if (cnt.alloc(v.nb_cp) != hipSuccess || cursor.alloc(v.nb_cp) != hipSuccess ||
        inc_ptr.alloc(v.nb_cp + 1) != hipSuccess)
        return fail(set_error(YETI_ERR_DEVICE, "CSR: allocation failed"));
    if (hipMemsetAsync(cnt.p, 0, 4 * (size_t)v.nb_cp, st) != hipSuccess ||
        hipMemsetAsync(cursor.p, 0, 4 * (size_t)v.nb_cp, st) != hipSuccess)
        return fail(set_error(YETI_ERR_DEVICE, "CSR: memset failed"));
    for (int p = 0; p < v.npatch; ++p) {
        int64_t n = (int64_t)v.n_active[p] * v.nnode[p];
        if (n == 0) continue;
        hipLaunchKernelGGL(inc_count_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, v.ien[p],
                           v.elems[p], v.n_active[p], v.nnode[p], cnt.p);
    }
    if ((rc = exclusive_scan<int32_t>(cnt.p, v.nb_cp, inc_ptr.p, st))) return fail(rc);
    int64_t ninc = 0;
    if ((rc = read_back(&ninc, inc_ptr.p + v.nb_cp, 8, st))) return fail(rc);
    if (inc.alloc(std::max<int64_t>(ninc, 1)) != hipSuccess) return fail(set_error(YETI_ERR_DEVICE, "CSR: alloc inc"));
    for (int p = 0; p < v.npatch; ++p) {
        int64_t n = (int64_t)v.n_active[p] * v.nnode[p];
        if (n == 0) continue;
        hipLaunchKernelGGL(inc_fill_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, v.ien[p],
                           v.elems[p], v.n_active[p], v.nnode[p], p, inc_ptr.p, cursor.p, inc.p);
    }
    hipLaunchKernelGGL(inc_sort_kernel, dim3((v.nb_cp + 255) / 256), dim3(256), 0, st, v.nb_cp, inc_ptr.p, inc.p);
    // block pattern
    if (rowlen.alloc(v.nb_cp) != hipSuccess || c->bptr.alloc(v.nb_cp + 1) != hipSuccess ||
        oflow.alloc(1) != hipSuccess || hipMemsetAsync(oflow.p, 0, 4, st) != hipSuccess ||
        flags.alloc(4) != hipSuccess || hipMemsetAsync(flags.p, 0, 16, st) != hipSuccess)
        return fail(set_error(YETI_ERR_DEVICE, "CSR: alloc rows"));
    hipLaunchKernelGGL(row_pattern_kernel<false>, dim3((v.nb_cp + 3) / 4), dim3(256), 0, st, v.nb_cp, inc_ptr.p,
                       inc.p, pi, rowlen.p, nullptr, nullptr, oflow.p);
    int32_t of = 0;
    if ((rc = read_back(&of, oflow.p, 4, st))) return fail(rc);
    if (of) return fail(set_error(YETI_ERR_SIZE_OVERFLOW, "CSR: a control point has more than 1024 neighbours"));
    if ((rc = exclusive_scan<int32_t>(rowlen.p, v.nb_cp, c->bptr.p, st))) return fail(rc);
    if ((rc = read_back(&c->nblocks, c->bptr.p + v.nb_cp, 8, st))) return fail(rc);
    if (c->bcol.alloc(std::max<int64_t>(c->nblocks, 1)) != hipSuccess)
        return fail(set_error(YETI_ERR_DEVICE, "CSR: alloc bcol"));
    hipLaunchKernelGGL(row_pattern_kernel<true>, dim3((v.nb_cp + 3) / 4), dim3(256), 0, st, v.nb_cp, inc_ptr.p,
                       inc.p, pi, nullptr, c->bptr.p, c->bcol.p, oflow.p);
    if (c->bdiag.alloc(std::max<int64_t>(v.nb_cp, 1)) != hipSuccess ||
        c->mirror.alloc(std::max<int64_t>(c->nblocks, 1)) != hipSuccess)
        return fail(set_error(YETI_ERR_DEVICE, "CSR: alloc mirror"));
    hipLaunchKernelGGL(mirror_kernel, dim3((v.nb_cp + 3) / 4), dim3(256), 0, st, v.nb_cp, c->bptr.p, c->bcol.p, c->bdiag.p,
                       c->mirror.p);
    // CSR_ROWS: every element is numbered against its CPs, rows are long enough (at p = 1 a run is 36
    // entries on average) and there are enough of them to hide that a row is one wave's chain: by rows and
    // by blocks p = 2 14^3 43.6 and 42.6 us, 15^3 49.2 and 51.7; p = 3 10^3 112 and 96, 11^3 116 and 140;
    // p = 4 (half the waves per CU) 14^3 1.10 and 0.94 ms, 18^3 1.98 and 1.89, 24^3 4.08 and 4.36.
    // CSR_EVERY: short rows of which less than a quarter of the transposes follow that of the row before.
    int32_t nn_max = 1;
    for (int p = 0; p < v.npatch; ++p)
        if (v.n_active[p] > 0) nn_max = std::max(nn_max, v.nnode[p]);
    const int64_t mean = (c->nblocks / std::max(v.nb_cp, 1) + 1) / 2;
    const bool long_rows = mean > 32 && c->nblocks / 2 >= (nn_max <= 64 ? 1 << 18 : 1 << 21);
    int32_t fl[4] = {0, 0, 0, 0};
    hipLaunchKernelGGL(upper_count_kernel, dim3((v.nb_cp + 255) / 256), dim3(256), 0, st, v.nb_cp, c->bptr.p, c->bdiag.p,
                       rowlen.p, flags.p);
    for (int p = 0; p < v.npatch && (long_rows || kind == CSR_ROWS); ++p) {
        const int64_t n = (int64_t)v.n_active[p] * v.nnode[p];
        if (n == 0) continue;
        hipLaunchKernelGGL(order_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, v.ien[p], v.elems[p],
                           v.n_active[p], v.nnode[p], flags.p);
    }
    if (mean <= SHORT_ROW)
        hipLaunchKernelGGL(adjacent_kernel, dim3(std::min(v.nb_cp, 4096)), dim3(64), 0, st, v.nb_cp, c->bptr.p, c->bcol.p,
                           c->bdiag.p, c->mirror.p, flags.p);
    if ((rc = read_back(fl, flags.p, sizeof fl, st))) return fail(rc);
    const bool rows_fit = fl[1] == 0 && fl[0] > 0 && nn_max <= 128 && (size_t)fl[0] * 72 * ROW_WAVES <= 64 * 1024;
    if (kind >= 0) {
        if ((kind == CSR_ROWS && !rows_fit) || (kind == CSR_SHORT && fl[0] > SHORT_ROW))
            return fail(set_error(YETI_ERR_INVALID_ARGUMENT, "CSR: the values of this model cannot be gathered in way %d", kind));
        c->kind = (CsrValues)kind;
    } else if (long_rows && rows_fit) {
        c->kind = CSR_ROWS;
    } else if (mean <= SHORT_ROW && 4 * fl[3] < fl[2]) {
        c->kind = CSR_EVERY;
    } else if (mean <= SHORT_ROW && fl[0] <= SHORT_ROW) {
        c->kind = CSR_SHORT;
    }
    if (c->kind == CSR_ROWS) {
        c->upper = fl[0];
        c->sstride = nn_max;
        if (c->irow.alloc(std::max<int64_t>(ninc, 1)) != hipSuccess ||
            c->slots.alloc((size_t)std::max<int64_t>(ninc, 1) * nn_max) != hipSuccess ||
            c->iptr.alloc(v.nb_cp + 1) != hipSuccess ||
            hipMemcpyAsync(c->iptr.p, inc_ptr.p, 8 * (size_t)(v.nb_cp + 1), hipMemcpyDeviceToDevice, st) != hipSuccess)
            return fail(set_error(YETI_ERR_DEVICE, "CSR: alloc element rows"));
        hipLaunchKernelGGL(slot_kernel, dim3(v.nb_cp), dim3(64), 0, st, v.nb_cp, inc_ptr.p, inc.p, pi, c->bptr.p, c->bcol.p,
                           c->bdiag.p, c->sstride, c->irow.p, c->slots.p);
    } else {   // contributions per listed block
        const bool dense = c->kind == CSR_LIST;
        const int64_t *lptr = c->bptr.p;
        c->nlist = c->nblocks;
        if (dense) {
            if (c->uptr.alloc(v.nb_cp + 1) != hipSuccess) return fail(set_error(YETI_ERR_DEVICE, "CSR: alloc block list"));
            if ((rc = exclusive_scan<int32_t>(rowlen.p, v.nb_cp, c->uptr.p, st))) return fail(rc);
            if ((rc = read_back(&c->nlist, c->uptr.p + v.nb_cp, 8, st))) return fail(rc);
            lptr = c->uptr.p;
        }
        const int64_t nl = std::max<int64_t>(c->nlist, 1);
        if (bcount.alloc(nl) != hipSuccess || c->cptr.alloc(c->nlist + 1) != hipSuccess ||
            (c->kind != CSR_SHORT && c->urow.alloc(nl) != hipSuccess))
            return fail(set_error(YETI_ERR_DEVICE, "CSR: alloc contributions"));
        if (c->kind != CSR_SHORT)
            hipLaunchKernelGGL(list_rows_kernel, dim3((v.nb_cp + 3) / 4), dim3(256), 0, st, v.nb_cp, lptr, c->urow.p);
        const int32_t *first = c->kind == CSR_EVERY ? nullptr : c->bdiag.p;
        hipLaunchKernelGGL(contrib_kernel<false>, dim3(v.nb_cp), dim3(64), 0, st, v.nb_cp, inc_ptr.p, inc.p, pi, c->bptr.p,
                           c->bcol.p, first, lptr, dense, bcount.p, nullptr, nullptr);
        if ((rc = exclusive_scan<int32_t>(bcount.p, c->nlist, c->cptr.p, st))) return fail(rc);
        int64_t ncontrib = 0;
        if ((rc = read_back(&ncontrib, c->cptr.p + c->nlist, 8, st))) return fail(rc);
        if (c->contrib.alloc(std::max<int64_t>(ncontrib, 1)) != hipSuccess)
            return fail(set_error(YETI_ERR_DEVICE, "CSR: alloc contrib list (%lld entries)", (long long)ncontrib));
        hipLaunchKernelGGL(contrib_kernel<true>, dim3(v.nb_cp), dim3(64), 0, st, v.nb_cp, inc_ptr.p, inc.p, pi, c->bptr.p,
                           c->bcol.p, first, lptr, dense, nullptr, c->cptr.p, c->contrib.p);
    }
    // scalar pattern
    if (c->rowptr.alloc(3 * (int64_t)v.nb_cp + 1) != hipSuccess ||
        c->colind.alloc(std::max<int64_t>(9 * c->nblocks, 1)) != hipSuccess)
        return fail(set_error(YETI_ERR_DEVICE, "CSR: alloc scalar pattern"));
    hipLaunchKernelGGL(scalar_pattern_kernel, dim3((v.nb_cp + 256) / 256), dim3(256), 0, st, v.nb_cp, c->bptr.p,
                       c->bcol.p, c->rowptr.p, c->colind.p);
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(st) != hipSuccess)
        return fail(set_error(YETI_ERR_DEVICE, "CSR: pattern kernels failed"));
    *out = c;
    return 0;
}

int32_t yeti_csr_create(const yeti_asm *h, void *stream, yeti_csr **out) { return yeti_csr_create_as(h, -1, stream, out); }

int32_t yeti_csr_values_kind(const yeti_csr *c) { return c ? (int32_t)c->kind : -1; }

int64_t yeti_csr_nnz(const yeti_csr *c) { return c ? 9 * c->nblocks : -1; }
int32_t yeti_csr_nrows(const yeti_csr *c) { return c ? 3 * c->nb_cp : -1; }
const int64_t *yeti_csr_rowptr(const yeti_csr *c) { return c ? c->rowptr.p : nullptr; }
const int32_t *yeti_csr_colind(const yeti_csr *c) { return c ? c->colind.p : nullptr; }

int32_t yeti_csr_values(const yeti_csr *c, const double *Kdata_dev, double *vals_dev, void *stream) {
    if (!c || !Kdata_dev || !vals_dev) return set_error(YETI_ERR_INVALID_ARGUMENT, "null argument");
    if (c->nblocks == 0) return 0;
    if (c->kind == CSR_ROWS) {
        auto rows = [&](auto kern) {
            hipLaunchKernelGGL(kern, dim3(xcd_grid(((int64_t)c->nb_cp + ROW_WAVES - 1) / ROW_WAVES)), dim3(64 * ROW_WAVES),
                               (size_t)c->upper * 72 * ROW_WAVES, (hipStream_t)stream, c->nb_cp, c->upper, c->sstride,
                               c->bptr.p, c->bcol.p, c->bdiag.p, c->mirror.p, c->iptr.p, c->irow.p, c->slots.p, Kdata_dev,
                               vals_dev);
        };
        if (c->sstride <= 64) rows(row_values_kernel<1>);
        else rows(row_values_kernel<2>);
        YETI_HIP(hipGetLastError());
        return 0;
    }
    const int64_t nitem = c->kind == CSR_SHORT ? (int64_t)SHORT_ROW * c->nb_cp : c->nlist;
    auto go = [&](auto kern, int vt) {
        hipLaunchKernelGGL(kern, dim3(xcd_grid((nitem + vt - 1) / vt)), dim3(vt), 160 * vt, (hipStream_t)stream, nitem,
                           c->kind == CSR_LIST ? c->uptr.p : c->bptr.p, c->urow.p, c->bptr.p, c->bcol.p, c->bdiag.p,
                           c->mirror.p, c->cptr.p, c->contrib.p, Kdata_dev, vals_dev);
    };
    // Small workgroups spread short lists over the CUs (4^3 p = 3: 24.7 -> 20.1 us); long ones are 1 %
    // faster in larger ones. The LDS is not used: 160 bytes per thread let 4 waves onto a SIMD, where 6
    // evict more of what their neighbours read from L2 (90^3 p = 1 1343 -> 1261 us, 16^3 p = 4 1374 -> 1290).
    const bool small = nitem <= 1 << 21;
    switch (c->kind) {
    case CSR_SHORT: small ? go(csr_values_kernel<64, CSR_SHORT>, 64) : go(csr_values_kernel<256, CSR_SHORT>, 256); break;
    case CSR_EVERY: small ? go(csr_values_kernel<64, CSR_EVERY>, 64) : go(csr_values_kernel<256, CSR_EVERY>, 256); break;
    default: small ? go(csr_values_kernel<64, CSR_LIST>, 64) : go(csr_values_kernel<256, CSR_LIST>, 256); break;
    }
    YETI_HIP(hipGetLastError());
    return 0;
}

int32_t yeti_csr_spmv(const yeti_csr *c, const double *vals_dev, const double *x_dev, double *y_dev, void *stream) {
    if (!c || !vals_dev || !x_dev || !y_dev) return set_error(YETI_ERR_INVALID_ARGUMENT, "null argument");
    return csr_block_spmv(c, vals_dev, x_dev, nullptr, y_dev, nullptr, 0, nullptr, (hipStream_t)stream);
}

int32_t yeti_csr_spmv_abs(const yeti_csr *c, const double *vals_dev, const double *x_dev, double *y_dev, void *stream) {
    if (!c || !vals_dev || !x_dev || !y_dev) return set_error(YETI_ERR_INVALID_ARGUMENT, "null argument");
    return csr_block_spmv(c, vals_dev, x_dev, nullptr, y_dev, nullptr, 1, nullptr, (hipStream_t)stream);
}

int32_t yeti_csr_pattern_to_host(const yeti_csr *c, int64_t *rowptr_host, int32_t *colind_host) {
    if (!c || !rowptr_host || !colind_host) return set_error(YETI_ERR_INVALID_ARGUMENT, "null argument");
    YETI_HIP(hipDeviceSynchronize());
    YETI_HIP(hipMemcpy(rowptr_host, c->rowptr.p, (3 * (size_t)c->nb_cp + 1) * sizeof(int64_t), hipMemcpyDeviceToHost));
    if (c->nblocks > 0)
        YETI_HIP(hipMemcpy(colind_host, c->colind.p, 9 * (size_t)c->nblocks * sizeof(int32_t), hipMemcpyDeviceToHost));
    return 0;
}

void yeti_csr_destroy(yeti_csr *c) { delete c; }

}  // extern "C"
