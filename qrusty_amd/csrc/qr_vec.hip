// qr_vec.hip -- the eigensolver-step operations around the matvec, on the
// device: the CSR diagonal, a x + b y and the diagonal preconditioner.
//
// They replace pyqrusty's SpMat.diagonal (pyqrusty/src/lib.rs:118-125, sprs
// CsMat::diag().to_dense()), qrusty::accel::axpby / axpy / ax
// (qrusty/src/accel.rs:374-393) and precond / precond2 / reg
// (pyqrusty/src/lib.rs:436-468).  Complex arithmetic is num-complex's:
// products (a.re x.re - a.im x.im, a.re x.im + a.im x.re) and sums with no
// fused multiply-add (the library is built with -ffp-contract=off), division
// ((a c + b d) / (c c + d d), (b c - a d) / (c c + d d)), norm = hypot.
// Every kernel but k_diag_scan is a grid-stride loop over its elements.
#include "qr_internal.h"

namespace qr {

__device__ __forceinline__ double2 cmul(double2 a, double2 x) {
    return make_double2(a.x * x.x - a.y * x.y, a.x * x.y + a.y * x.x);
}

__device__ __forceinline__ double2 cdiv(double2 p, double2 q) {
    const double n = q.x * q.x + q.y * q.y;
    const double re = p.x * q.x + p.y * q.y;
    const double im = p.y * q.x - p.x * q.y;
    return make_double2(re / n, im / n);
}

// Diagonal entry of row r: the entry with column r, found by binary search in
// the row's ascending columns (as sprs CsVecView::get); 0 when absent.
__device__ __forceinline__ double2 diag_entry(uint64_t r, uint64_t nnz,
                                              const uint64_t *__restrict__ indptr,
                                              const uint64_t *__restrict__ indices,
                                              const double2 *__restrict__ data) {
    uint64_t lo = indptr[r], hi = indptr[r + 1];
    if (hi > nnz) hi = nnz;
    if (lo > hi) lo = hi;
    while (lo < hi) {  // first position with column >= r
        const uint64_t mid = lo + (hi - lo) / 2;
        if (indices[mid] < r) lo = mid + 1;
        else hi = mid;
    }
    if (lo < (indptr[r + 1] < nnz ? indptr[r + 1] : nnz) && indices[lo] == r) return data[lo];
    return make_double2(0.0, 0.0);
}

__global__ __launch_bounds__(256) void k_csr_diagonal(uint64_t n, uint64_t nnz,
                                                      const uint64_t *__restrict__ indptr,
                                                      const uint64_t *__restrict__ indices,
                                                      const double2 *__restrict__ data,
                                                      double2 *__restrict__ out) {
    for (uint64_t r = uint64_t(blockIdx.x) * 256 + threadIdx.x; r < n;
         r += uint64_t(gridDim.x) * 256)
        out[r] = diag_entry(r, nnz, indptr, indices, data);
}

// out = dx / reg(d - e, tol), reg(v) = tol + 0i when |v| < tol, else v
__device__ __forceinline__ double2 precond_entry(double2 d, double2 dx, double2 e, double tol) {
    double2 v = make_double2(d.x - e.x, d.y - e.y);
    if (hypot(v.x, v.y) < tol) v = make_double2(tol, 0.0);
    return cdiv(dx, v);
}

// Rows of 8 to kDiagScan entries in the mean: a wave takes 64 rows, one per lane
// for their bounds, their diagonal's value and the result, and 2^lpr_log2 lanes
// read a row's columns, four each, kDiagDepth rows in flight per lane group; the
// first entry of the row that has the diagonal column is its own.  Rows longer
// than their lanes' four entries are searched, each by its lane.
// What bounds it: memory.  A binary search per row, the other way, leaves its
// lines in the caches between dependent probes, where they thrash, but reads
// few lines of a long row.  Measured (precond, us, search / this): rings of 20,
// 23, 24 qubits (21 to 25 entries) 107 / 60, 794 / 562, 1651 / 1120; Poisson
// lengths of 9, 22, 35, 20 qubits 31 / 20, 85 / 35, 98 / 65; geometric ones of 30
// 75 / 55; one row of 2^19 entries, the others 12 in the mean 52 / 23; but 15 rows
// of 16 of one entry, the others 625, 20 / 44.  (A lane group for every row, whatever
// its length: rings 68, 569, 1186; the row of 2^19 entries 12400.)
constexpr double kDiagScan = 48.0;
constexpr int kDiagDepth = 4;
template <bool kPrecond>
__global__ __launch_bounds__(256) void k_diag_scan(uint64_t n, uint32_t lpr_log2, uint64_t nnz,
                                                   const uint64_t *__restrict__ indptr,
                                                   const uint64_t *__restrict__ indices,
                                                   const double2 *__restrict__ data,
                                                   const double2 *__restrict__ dx, double2 e, double tol,
                                                   double2 *__restrict__ out) {
    const uint32_t wl = threadIdx.x & 63u, lpr = 1u << lpr_log2, lane = wl & (lpr - 1u), group = wl >> lpr_log2;
    const uint32_t gw = 64u >> lpr_log2, shift = wl & ~(lpr - 1u);
    const uint64_t r0 = (uint64_t(blockIdx.x) * 4 + threadIdx.x / 64u) * 64;
    if (r0 >= n) return;
    const uint64_t r = r0 + wl, rr = r < n ? r : n - 1;
    const uint64_t lo = indptr[rr], hi = indptr[rr + 1] < nnz ? indptr[rr + 1] : nnz;
    // the wave's entries from `base` on, counted in 32 bits
    const uint64_t first = uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(lo >> 32)))) << 32 |
                           uint32_t(__builtin_amdgcn_readfirstlane(int(lo)));
    const uint64_t base = first < nnz ? first : nnz - 1;
    const uint32_t most = nnz - 1 - base < (1u << 30) ? uint32_t(nnz - 1 - base) : 1u << 30;
    const bool some = lo < hi, fits = !some || (hi - lo <= 4 * lpr && lo - base < (1u << 29));
    const uint32_t rel = some && fits ? uint32_t(lo - base) : 0u, len = some && fits ? uint32_t(hi - lo) : 0u;
    uint32_t at = ~0u;
    for (uint32_t s = 0; s < lpr; s += kDiagDepth) {
        uint64_t c[kDiagDepth][4];
        uint32_t l[kDiagDepth];
#pragma unroll
        for (int d = 0; d < kDiagDepth; ++d) {
            const int row = int((s + uint32_t(d)) * gw + group);
            const uint32_t o = uint32_t(__shfl(int(rel), row)) + lane;
            l[d] = uint32_t(__shfl(int(len), row));
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) {
                const uint32_t i = o + u * lpr;
                c[d][u] = indices[base + (i < most ? i : most)];
            }
        }
#pragma unroll
        for (int d = 0; d < kDiagDepth; ++d) {
            const uint64_t row = r0 + (s + uint32_t(d)) * gw + group;
            uint32_t pos = ~0u;
#pragma unroll
            for (int u = 3; u >= 0; --u) {
                const uint32_t i = lane + uint32_t(u) * lpr;
                const uint64_t met = __ballot(i < l[d] && c[d][u] == row) >> shift;
                const uint32_t mine = uint32_t(met) & (lpr == 32 ? ~0u : (1u << lpr) - 1u);
                if (mine) pos = uint32_t(u) * lpr + uint32_t(__builtin_ctz(mine));
            }
            // to the lane of the row
            const uint32_t got = uint32_t(__shfl(int(pos), int((wl & (gw - 1u)) << lpr_log2)));
            if (wl >> (6u - lpr_log2) == s + uint32_t(d)) at = got;
        }
    }
    if (r >= n) return;
    double2 d = make_double2(0.0, 0.0);
    if (!fits) d = diag_entry(r, nnz, indptr, indices, data);
    else if (at != ~0u) d = data[base + rel + at];
    out[r] = kPrecond ? precond_entry(d, dx[r], e, tol) : d;
}

// Lanes per row of k_diag_scan (0: not by it), 4 to 32: a quarter of the mean
// length, or, where the rows cannot be equal, of what most of them have
static uint32_t diag_lanes_log2(uint64_t nrows, uint64_t nnz) {
    const double mean = double(nnz) / double(nrows);
    if (mean < 8.0 || mean > kDiagScan) return 0;
    const double need = nnz % nrows ? mean + 2.0 * sqrt(mean) : mean;
    uint32_t l = 2;
    while (l < 5 && double(4u << l) < need) ++l;
    return l;
}

// z = a x + b y  (mode 0), a x + y (mode 1), a x (mode 2)
__global__ __launch_bounds__(256) void k_axpby(uint64_t n, int mode, double2 a,
                                               const double2 *__restrict__ x, double2 b,
                                               const double2 *__restrict__ y,
                                               double2 *__restrict__ z) {
    for (uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x; i < n;
         i += uint64_t(gridDim.x) * 256) {
        const double2 ax = cmul(a, x[i]);
        if (mode == 2) {
            z[i] = ax;
        } else {
            const double2 by = mode == 0 ? cmul(b, y[i]) : y[i];
            z[i] = make_double2(ax.x + by.x, ax.y + by.y);
        }
    }
}

// precond_entry of every row, the diagonal d either given (precond2) or
// searched in the CSR (precond)
__global__ __launch_bounds__(256) void k_precond(uint64_t n, const double2 *__restrict__ diag,
                                                 uint64_t nnz, const uint64_t *__restrict__ indptr,
                                                 const uint64_t *__restrict__ indices,
                                                 const double2 *__restrict__ data,
                                                 const double2 *__restrict__ dx, double2 e,
                                                 double tol, double2 *__restrict__ out) {
    for (uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x; i < n;
         i += uint64_t(gridDim.x) * 256) {
        const double2 d = diag ? diag[i] : diag_entry(i, nnz, indptr, indices, data);
        out[i] = precond_entry(d, dx[i], e, tol);
    }
}

static unsigned grid_for(uint64_t n) {
    const uint64_t b = (n + 255) / 256;
    return unsigned(b < 65536 ? (b ? b : 1) : 65536);
}

int launch_csr_diagonal(uint64_t nrows, uint64_t ncols, uint64_t nnz, const uint64_t *indptr,
                        const uint64_t *indices, const double *data, double *out, hipStream_t s) {
    const uint64_t n = nrows < ncols ? nrows : ncols;
    if (n == 0) return QR_OK;
    if (const uint32_t l = diag_lanes_log2(nrows, nnz)) {
        const uint64_t blocks = (n + 255) / 256;
        if (blocks <= 0x7FFFFFFFull) {
            hipLaunchKernelGGL(k_diag_scan<false>, dim3(unsigned(blocks)), dim3(256), 0, s, n, l, nnz, indptr,
                               indices, reinterpret_cast<const double2 *>(data), nullptr, double2{}, 0.0,
                               reinterpret_cast<double2 *>(out));
            QR_HIP_CHECK(hipGetLastError());
            return QR_OK;
        }
    }
    hipLaunchKernelGGL(k_csr_diagonal, dim3(grid_for(n)), dim3(256), 0, s, n, nnz, indptr,
                       indices, reinterpret_cast<const double2 *>(data),
                       reinterpret_cast<double2 *>(out));
    QR_HIP_CHECK(hipGetLastError());
    return QR_OK;
}

int launch_axpby(uint64_t n, int mode, const double *a, const double *x, const double *b,
                 const double *y, double *z, hipStream_t s) {
    if (n == 0) return QR_OK;
    const double2 a2 = make_double2(a[0], a[1]);
    const double2 b2 = b ? make_double2(b[0], b[1]) : make_double2(0.0, 0.0);
    hipLaunchKernelGGL(k_axpby, dim3(grid_for(n)), dim3(256), 0, s, n, mode, a2,
                       reinterpret_cast<const double2 *>(x), b2,
                       reinterpret_cast<const double2 *>(y), reinterpret_cast<double2 *>(z));
    QR_HIP_CHECK(hipGetLastError());
    return QR_OK;
}

int launch_precond(uint64_t n, const double *diag, uint64_t nnz, const uint64_t *indptr,
                   const uint64_t *indices, const double *data, const double *dx, const double *e,
                   double tol, double *out, hipStream_t s) {
    if (n == 0) return QR_OK;
    const uint32_t l = diag ? 0 : diag_lanes_log2(n, nnz);
    const uint64_t blocks = (n + 255) / 256;
    if (l && blocks <= 0x7FFFFFFFull) {
        hipLaunchKernelGGL(k_diag_scan<true>, dim3(unsigned(blocks)), dim3(256), 0, s, n, l, nnz, indptr, indices,
                           reinterpret_cast<const double2 *>(data), reinterpret_cast<const double2 *>(dx),
                           make_double2(e[0], e[1]), tol, reinterpret_cast<double2 *>(out));
        QR_HIP_CHECK(hipGetLastError());
        return QR_OK;
    }
    hipLaunchKernelGGL(k_precond, dim3(grid_for(n)), dim3(256), 0, s, n,
                       reinterpret_cast<const double2 *>(diag), nnz, indptr, indices,
                       reinterpret_cast<const double2 *>(data),
                       reinterpret_cast<const double2 *>(dx), make_double2(e[0], e[1]), tol,
                       reinterpret_cast<double2 *>(out));
    QR_HIP_CHECK(hipGetLastError());
    return QR_OK;
}

}  // namespace qr
