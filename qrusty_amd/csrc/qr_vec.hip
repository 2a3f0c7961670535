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

// Rows of 8 to kDiagScan entries in the mean: 2^lpr_log2 lanes read a row's
// columns, four each at a time, and the lane that meets the diagonal writes
// the row's result (the first lane, if none does).
// What bounds it: memory.  A binary search per row, the other way, leaves its
// lines in the caches between dependent probes, where they thrash, but reads
// few lines of a long row.  Measured (precond, us, search / scan): rings of 20,
// 23, 24 qubits (21 to 25 entries) 109 / 66, 815 / 582, 1671 / 1190; random
// operators of 4 entries, 24 qubits 214 / 400, 60, 22 qubits 442 / 474, 120, 21
// qubits 269 / 470.
constexpr double kDiagScan = 48.0;
template <bool kPrecond>
__global__ __launch_bounds__(256) void k_diag_scan(uint64_t n, uint32_t lpr_log2, uint64_t nnz,
                                                   const uint64_t *__restrict__ indptr,
                                                   const uint64_t *__restrict__ indices,
                                                   const double2 *__restrict__ data,
                                                   const double2 *__restrict__ dx, double2 e, double tol,
                                                   double2 *__restrict__ out) {
    const uint32_t lpr = 1u << lpr_log2, lane = threadIdx.x & (lpr - 1u);
    const uint64_t r = uint64_t(blockIdx.x) * (256u >> lpr_log2) + (threadIdx.x >> lpr_log2);
    if (r >= n) return;
    const uint64_t hi = indptr[r + 1] < nnz ? indptr[r + 1] : nnz;
    uint64_t at = ~uint64_t(0);
    for (uint64_t k = indptr[r] + lane; k < hi; k += 4 * lpr) {
        uint64_t c[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const uint64_t i = k + uint32_t(u) * lpr;
            c[u] = indices[i < nnz ? i : nnz - 1];
        }
#pragma unroll
        for (int u = 3; u >= 0; --u) {
            const uint64_t i = k + uint32_t(u) * lpr;
            if (c[u] == r && i < hi && i < at) at = i;
        }
    }
    const uint64_t met = __ballot(at != ~uint64_t(0)) >> ((threadIdx.x & 63u) & ~(lpr - 1u));
    const uint64_t mine = met & (lpr == 64 ? ~uint64_t(0) : (uint64_t(1) << lpr) - 1);
    // (a column that comes more than once in the row: its first entry)
    uint64_t first = at;
    if (mine & (mine - 1))
        for (uint32_t o = 1; o < lpr; o <<= 1) {
            const uint64_t other = __shfl_xor(first, int(o));
            first = other < first ? other : first;
        }
    if (mine ? at == ~uint64_t(0) || at != first : lane != 0) return;
    const double2 d = mine ? data[at] : make_double2(0.0, 0.0);
    out[r] = kPrecond ? precond_entry(d, dx[r], e, tol) : d;
}

// Lanes per row of k_diag_scan (0: not by it): a quarter of the mean length
static uint32_t diag_lanes_log2(uint64_t nrows, uint64_t nnz) {
    if (double(nnz) < 8.0 * double(nrows) || double(nnz) > kDiagScan * double(nrows)) return 0;
    uint32_t l = 2;
    while (l < 6 && (nrows << (l + 2)) < nnz) ++l;
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
        const uint64_t blocks = (n + (256u >> l) - 1) / (256u >> l);
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
    const uint64_t blocks = l ? (n + (256u >> l) - 1) / (256u >> l) : 0;
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
