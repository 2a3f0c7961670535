// qr_spadd.hip -- a*A + b*B of two CSR matrices of the same shape on the
// device: pyqrusty's a_spmat_p_b_spmat (pyqrusty/src/lib.rs:499-517), i.e.
// sprs CsMat::scale on clones and `&am1 + &am2` (sprs csmat_binop).
//
// Each row is the merge of the two rows' ascending columns: an entry in both
// gets a*v1 + b*v2, one in A only a*v1 + 0, one in B only 0 + b*v2 (complex
// products as num-complex, no fused multiply-add), and results equal to zero
// are dropped.  Two passes over the rows -- count, then (after a scan of the
// counts into indptr) fill.
//
// Two kernels.  k_spadd_few, where one matrix has one or two entries per row in
// the mean (spadd_few).  Otherwise k_spadd_tile: a block takes a tile of
// consecutive rows.  Their entries are contiguous in both inputs, so the block
// loads them coalesced into LDS (column and the already scaled value a*v1 or b*v2), a
// group of lanes per row merges in LDS (each lane from its own merge-path split
// of the row), and the fill pass writes the tile's merged entries to LDS and
// from there coalesced to the output, whose tile range is contiguous too.  A
// tile whose entries exceed the LDS capacity (long or uneven rows) is merged
// from global memory, one thread per row.
#include "qr_internal.h"
#include "qr_mv.h"

#include <hipcub/device/device_scan.hpp>

#include <cmath>

namespace qr {

__device__ __forceinline__ double2 cmul2(double2 a, double2 v) {
    return make_double2(a.x * v.x - a.y * v.y, a.x * v.y + a.y * v.x);
}

// Walks the merge of row r; for every kept entry calls emit(column, value).
// Row bounds are clamped to each matrix's nnz, so a malformed CSR cannot make
// the merge read out of bounds.
struct SpAddIn {
    double2 a, b;
    uint64_t nnz1, nnz2;
    const uint64_t *ip1, *ix1, *ip2, *ix2;
    const double2 *d1, *d2;
};

template <typename Emit>
__device__ __forceinline__ void merge_row(uint64_t r, const SpAddIn &in, Emit emit) {
    const double2 a = in.a, b = in.b;
    const uint64_t *__restrict__ ix1 = in.ix1;
    const uint64_t *__restrict__ ix2 = in.ix2;
    const double2 *__restrict__ d1 = in.d1;
    const double2 *__restrict__ d2 = in.d2;
    const uint64_t i1 = in.ip1[r + 1] < in.nnz1 ? in.ip1[r + 1] : in.nnz1;
    const uint64_t j1 = in.ip2[r + 1] < in.nnz2 ? in.ip2[r + 1] : in.nnz2;
    uint64_t i = in.ip1[r] < i1 ? in.ip1[r] : i1, j = in.ip2[r] < j1 ? in.ip2[r] : j1;
    const double2 zero = make_double2(0.0, 0.0);
    while (i < i1 || j < j1) {
        uint64_t col;
        double2 v;
        if (j >= j1 || (i < i1 && ix1[i] < ix2[j])) {
            col = ix1[i];
            const double2 p = cmul2(a, d1[i]);
            v = make_double2(p.x + zero.x, p.y + zero.y);
            ++i;
        } else if (i >= i1 || ix2[j] < ix1[i]) {
            col = ix2[j];
            const double2 q = cmul2(b, d2[j]);
            v = make_double2(zero.x + q.x, zero.y + q.y);
            ++j;
        } else {
            col = ix1[i];
            const double2 p = cmul2(a, d1[i]), q = cmul2(b, d2[j]);
            v = make_double2(p.x + q.x, p.y + q.y);
            ++i;
            ++j;
        }
        if (v.x != 0.0 || v.y != 0.0) emit(col, v);
    }
}

#ifndef QR_SPADD_CAP
#define QR_SPADD_CAP 512
#endif
// Threads per block: measured on the 24-qubit H - e*I (count + fill, ms) with
// 512-entry tiles, 256 threads 3.2 + 5.4, 128 threads 2.7 + 6.3.  The two
// passes need not share a tiling (for a CSR whose indptr ascends within nnz,
// each route of the merge gives a row the same entries), so each takes its
// faster one.  Count pass, threads / tile entries: 128 / 512 2.52-2.64 ms,
// 64 / 256 2.60, 64 / 512 2.85, 256 / 1024 2.98, 128 / 256 3.10,
// 128 / 1024 3.45.
#ifndef QR_SPADD_COUNT_THREADS
#define QR_SPADD_COUNT_THREADS 128
#endif
#ifndef QR_SPADD_COUNT_CAP
#define QR_SPADD_COUNT_CAP 512
#endif
constexpr int kSpCountThreads = QR_SPADD_COUNT_THREADS, kSpFillThreads = 256;
constexpr int kSpCountCap = QR_SPADD_COUNT_CAP;
constexpr int kSpCap = QR_SPADD_CAP;  // staged input entries (A + B) per tile
static_assert(kSpCap % kSpFillThreads == 0 && kSpCountCap % kSpCountThreads == 0,
              "whole staging rounds per thread");

__device__ __forceinline__ uint64_t clampu(uint64_t v, uint64_t lo, uint64_t hi) {
    return v < lo ? lo : (v > hi ? hi : v);
}

// Tile of rows [r0, r0 + rows_per_tile).  kFill = false writes counts[r];
// kFill = true writes the merged rows at ipo[r].
template <bool kFill, int kT, int kCap>
__global__ __launch_bounds__(kT) void k_spadd_tile(uint64_t nrows, uint32_t rows_per_tile,
                                                           uint32_t lpr,
                                                           SpAddIn in, uint64_t *__restrict__ counts,
                                                           const uint64_t *__restrict__ ipo,
                                                           uint64_t *__restrict__ ixo,
                                                           double2 *__restrict__ dout) {
    __shared__ uint64_t sc[kCap];
    __shared__ double2 sv[kCap];
    __shared__ uint64_t oc[kFill ? kCap : 1];
    __shared__ double2 ov[kFill ? kCap : 1];
    const uint32_t tid = threadIdx.x;
    const uint64_t r0 = uint64_t(blockIdx.x) * rows_per_tile;
    if (r0 >= nrows) return;
    const uint64_t r1 = r0 + rows_per_tile < nrows ? r0 + rows_per_tile : nrows;
    const uint64_t a0 = clampu(in.ip1[r0], 0, in.nnz1), a1 = clampu(in.ip1[r1], a0, in.nnz1);
    const uint64_t b0 = clampu(in.ip2[r0], 0, in.nnz2), b1 = clampu(in.ip2[r1], b0, in.nnz2);
    const uint64_t ea = a1 - a0, eb = b1 - b0;
    if (ea + eb > uint64_t(kCap)) {
        // global-memory merge, one thread per row.  For a CSR whose indptr
        // ascends within nnz it gives each row what the LDS merge gives; the
        // two passes tile the rows differently, so for a malformed one a row's
        // count may come from the other route, and the fill stops at the
        // row's end either way.
        for (uint64_t r = r0 + tid; r < r1; r += kT) {
            if (kFill) {
                uint64_t k = ipo[r];
                const uint64_t kend = ipo[r + 1];
                merge_row(r, in, [&](uint64_t c, double2 v) {
                    if (k < kend) {
                        ixo[k] = c;
                        dout[k] = v;
                    }
                    ++k;
                });
            } else {
                uint64_t n = 0;
                merge_row(r, in, [&](uint64_t, double2) { ++n; });
                counts[r] = n;
            }
        }
        return;
    }
    {
        // every load of this thread in flight at once: slot k < ea is A's
        // entry a0 + k, slot ea <= k < ea + eb B's entry b0 + k - ea
        constexpr int kPer = kCap / kT;
        uint64_t c[kPer];
        double2 v[kPer];
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const uint32_t k = tid + u * kT;
            if (k < ea) {
                c[u] = __builtin_nontemporal_load(in.ix1 + a0 + k);
                v[u].x = __builtin_nontemporal_load(&in.d1[a0 + k].x);
                v[u].y = __builtin_nontemporal_load(&in.d1[a0 + k].y);
            } else if (k < ea + eb) {
                c[u] = __builtin_nontemporal_load(in.ix2 + b0 + (k - ea));
                v[u].x = __builtin_nontemporal_load(&in.d2[b0 + (k - ea)].x);
                v[u].y = __builtin_nontemporal_load(&in.d2[b0 + (k - ea)].y);
            }
        }
#pragma unroll
        for (int u = 0; u < kPer; ++u) {
            const uint32_t k = tid + u * kT;
            if (k < ea + eb) {
                sc[k] = c[u];
                sv[k] = cmul2(k < ea ? in.a : in.b, v[u]);
            }
        }
    }
    __syncthreads();
    const uint64_t o0 = kFill ? ipo[r0] : 0;
    // lpr lanes per row (a power of two <= 64, so a row's lanes share a wave)
    const uint32_t lane = tid & (lpr - 1);
    for (uint64_t r = r0 + tid / lpr; r < r1; r += kT / lpr) {
        // row bounds inside the staged ranges: B's entries sit after A's
        const uint32_t ia = uint32_t(clampu(in.ip1[r], a0, a1) - a0);
        const uint32_t ia1 = uint32_t(clampu(in.ip1[r + 1], a0 + ia, a1) - a0);
        const uint32_t jb = uint32_t(ea + clampu(in.ip2[r], b0, b1) - b0);
        const uint32_t jb1 = uint32_t(ea + clampu(in.ip2[r + 1], b0 + (jb - ea), b1) - b0);
        const uint32_t na = ia1 - ia, nb = jb1 - jb, m = na + nb;
        const uint32_t seg = (m + lpr - 1) / lpr;
        // merge-path split (A first on equal columns) at the diagonals of this
        // lane and of the next
        auto split = [&](uint32_t d) {
            uint32_t lo = d > nb ? d - nb : 0, hi = d < na ? d : na;
            while (lo < hi) {
                const uint32_t mid = (lo + hi) >> 1;
                if (sc[ia + mid] <= sc[jb + d - 1 - mid]) lo = mid + 1;
                else hi = mid;
            }
            return lo;
        };
        const uint32_t d0 = lane * seg < m ? lane * seg : m;
        const uint32_t dE = d0 + seg < m ? d0 + seg : m;
        const uint32_t s0 = split(d0), sE = split(dE);
        uint32_t i = ia + s0, j = jb + (d0 - s0);
        const uint32_t iE = ia + sE, jE = jb + (dE - sE);
        // a B entry paired with the last A entry before this lane's start was
        // taken by the lane that holds that A entry
        if (i > ia && j < jb1 && sc[i - 1] == sc[j]) ++j;
        auto walk = [&](auto emit) {
            uint32_t wi = i, wj = j;
            while (wi < iE || wj < jE) {
                bool take_a, take_b;
                uint64_t col;
                if (wi >= iE) {
                    take_a = false;
                    take_b = true;
                    col = sc[wj];
                } else {
                    const uint64_t ca = sc[wi];
                    // the B entry at this lane's end may pair with its last A entry
                    const bool b_ok = wj < jE || (wj < jb1 && wi + 1 == iE);
                    const uint64_t cb = b_ok ? sc[wj] : ca;
                    take_a = !b_ok || ca <= cb;
                    take_b = b_ok && cb <= ca;
                    col = take_a ? ca : cb;
                }
                double2 v;
                // one side only: + 0 as the reference's binop does (a -0.0
                // component becomes +0.0)
                if (take_a && take_b) {
                    const double2 p = sv[wi++], q = sv[wj++];
                    v = make_double2(p.x + q.x, p.y + q.y);
                } else if (take_a) {
                    const double2 p = sv[wi++];
                    v = make_double2(p.x + 0.0, p.y + 0.0);
                } else {
                    const double2 q = sv[wj++];
                    v = make_double2(0.0 + q.x, 0.0 + q.y);
                }
                if (v.x != 0.0 || v.y != 0.0) emit(col, v);
            }
        };
        // kept entries of this lane; the fill pass walks again to emit them
        // from the slot after the lanes before it
        uint32_t n = 0;
        walk([&](uint64_t, double2) { ++n; });
        // inclusive sum of n over the row's lanes
        uint32_t incl = n;
        for (uint32_t o = 1; o < lpr; o <<= 1) {
            const uint32_t t = __shfl_up(incl, o, lpr);
            if (lane >= o) incl += t;
        }
        if (!kFill) {
            if (lane == lpr - 1) counts[r] = incl;
        } else {
            uint64_t k = ipo[r] - o0 + (incl - n);
            walk([&](uint64_t col, double2 v) {
                if (k < uint64_t(kCap)) {
                    oc[k] = col;
                    ov[k] = v;
                }
                ++k;
            });
        }
    }
    if (kFill) {
        __syncthreads();
        uint64_t total = ipo[r1] - o0;
        total = total < uint64_t(kCap) ? total : uint64_t(kCap);
        for (uint32_t k = tid; k < total; k += kT) {
            __builtin_nontemporal_store(oc[k], ixo + o0 + k);
            __builtin_nontemporal_store(ov[k].x, &dout[o0 + k].x);
            __builtin_nontemporal_store(ov[k].y, &dout[o0 + k].y);
        }
    }
}

// One matrix with few entries per row (H - e*I): 2^lpr_log2 lanes hold a row's
// entries of the longer matrix (in), that many at a time, and pass over the
// shorter one's; ballots give every entry its place among the kept ones.
// Nothing is staged: inputs are read and outputs written by consecutive lanes.
// Results as merge_row's, whichever matrix is the longer (the sums commute), and
// for rows in any order: a short entry meets the first of the long ones left
// whose column is not below its own, and joins it or comes before it.
// A wave takes 2^rpw_log2 consecutive rows, one per lane for their bounds and
// their entry of the shorter matrix, which the lanes of a row then fetch by
// shuffles.  Rows that have one such entry at most and fit their lanes run
// kSpDepth at a time per lane group and take few vector instructions; the others
// follow, one at a time, in pieces (kPieces: all do).
// What bounds it: the fill pass memory (10 GB at 5.3 TB/s for the 23-qubit
// ring), the count pass (5.2 GB at 5) that and its instructions.  Measured
// (H - e*I, count + fill us, staged tiles / this): 23-qubit ring 1540 + 3040 /
// 1130 + 1895; 16-qubit molecule (981 entries per row, which overflow the
// staged tile) 12350 + 21090 / 330 + 500; 992 random terms, 16 qubits 12430 +
// 22960 / 320 + 720.  Without the shared loads of the bounds (one row of two
// per lane group at a time) the ring took 1640 + 2065; 4 rows in flight 1190 +
// 1970.
constexpr int kSpDepth = 8;

__device__ __forceinline__ double2 nt_value(const double2 *p) {
    const dvec2 v = __builtin_nontemporal_load(reinterpret_cast<const dvec2 *>(p));
    return make_double2(v.x, v.y);
}
__device__ __forceinline__ void nt_store(uint64_t c, double2 v, uint64_t *ix, double2 *d) {
    __builtin_nontemporal_store(c, ix);
    __builtin_nontemporal_store(dvec2{v.x, v.y}, reinterpret_cast<dvec2 *>(d));
}
__device__ __forceinline__ uint64_t first_lane(uint64_t v) {
    return uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(int(v >> 32)))) << 32 |
           uint32_t(__builtin_amdgcn_readfirstlane(int(v)));
}

template <bool kFill, bool kPieces>
__global__ __launch_bounds__(256) void k_spadd_few(uint64_t nrows, uint32_t lpr_log2, uint32_t rpw_log2, SpAddIn in,
                                                   uint64_t *__restrict__ counts,
                                                   const uint64_t *__restrict__ ipo,
                                                   uint64_t *__restrict__ ixo, double2 *__restrict__ dout) {
    const uint32_t wl = threadIdx.x & 63u, lpr = 1u << lpr_log2, lane = wl & (lpr - 1u), group = wl >> lpr_log2;
    const uint32_t gw = 64u >> lpr_log2, shift = wl & ~(lpr - 1u);
    const uint64_t gmask = lpr == 64 ? ~uint64_t(0) : ((uint64_t(1) << lpr) - 1);
    const uint32_t mine0 = uint32_t(gmask << shift), mine1 = uint32_t((gmask << shift) >> 32);
    const uint64_t rw = (uint64_t(blockIdx.x) * 4 + threadIdx.x / 64u) << rpw_log2;  // the wave's first row
    if (rw >= nrows) return;
    const uint32_t rows = uint32_t(nrows - rw < (uint64_t(1) << rpw_log2) ? nrows - rw : uint64_t(1) << rpw_log2);
    // row rw + wl of each lane (of the last lanes: the last row)
    uint64_t i0, i1, j0, j1, po = 0, pe = 0;
    {
        const uint64_t r = rw + (wl < rows ? wl : rows - 1);
        i0 = in.ip1[r];
        i1 = in.ip1[r + 1];
        j0 = in.ip2[r];
        j1 = in.ip2[r + 1];
        if (kFill) {
            po = ipo[r];
            pe = ipo[r + 1];
        }
        i1 = i1 < in.nnz1 ? i1 : in.nnz1;
        i0 = i0 < i1 ? i0 : i1;
        j1 = j1 < in.nnz2 ? j1 : in.nnz2;
        j0 = j0 < j1 ? j0 : j1;
    }
    const uint64_t iw = first_lane(i0), pw = first_lane(po);
    const bool fits = !kPieces && i1 - i0 <= lpr && j1 - j0 <= 1 && i0 - iw < (1u << 27) &&
                      (!kFill || (po - pw < (1u << 27) && pe - po < (1u << 27)));
    if (!kPieces && __any(fits)) {
        // (iw < nnz1 unless the wave's rows are empty or the last)
        const uint64_t ia = iw < in.nnz1 ? iw : in.nnz1 - 1, left = in.nnz1 - 1 - ia;
        const uint32_t most = left < (1u << 28) ? uint32_t(left) : 1u << 28;
        const uint64_t jc = j0 < in.nnz2 ? j0 : in.nnz2 - 1;
        const uint64_t cb = in.ix2[jc];
        const double2 q = cmul2(in.b, in.d2[jc]);
        const bool hb = fits && j1 > j0;
        // (of a row that does not fit: none) the row's entries, whether it has one of the shorter matrix and
        // whether that alone is kept, and the room in the output
        const uint32_t meta = (fits ? uint32_t(i1 - i0) : 0u) | (hb ? 0x100u : 0u) |
                              (hb && (0.0 + q.x != 0.0 || 0.0 + q.y != 0.0) ? 0x200u : 0u) |
                              (kFill ? uint32_t(pe - po < 0xffff ? pe - po : 0xffff) << 16 : 0u);
        const uint32_t rel = fits ? uint32_t(i0 - iw) : 0u, orel = fits ? uint32_t(po - pw) : 0u;
        const uint64_t *ix1 = in.ix1 + ia;
        const double2 *d1 = in.d1 + ia;
        uint32_t count = 0;
        // the lowest and the highest lane of every row
        uint64_t lows = 1;
        for (uint32_t k = lpr; k < 64; k <<= 1) lows |= lows << k;
        const uint64_t highs = lows << (lpr - 1u);
        for (uint32_t s = 0; s * gw < rows; s += kSpDepth) {
            uint64_t c[kSpDepth];
            double2 v[kSpDepth];
            uint32_t mt[kSpDepth];
#pragma unroll
            for (int u = 0; u < kSpDepth; ++u) {
                const uint32_t row = (s + uint32_t(u)) * gw + group;
                mt[u] = uint32_t(__shfl(int(meta), int(row & 63u)));
                uint32_t at = uint32_t(__shfl(int(rel), int(row & 63u))) + lane;
                at = at < most ? at : most;
                c[u] = __builtin_nontemporal_load(ix1 + at);
                v[u] = nt_value(d1 + at);
            }
            // (all their loads before the first is used)
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < kSpDepth; ++u) {
                const uint32_t row = (s + uint32_t(u)) * gw + group;
                const bool have = row < rows && lane < (mt[u] & 0xffu);
                const uint64_t cr = __shfl(cb, int(row & 63u));
                const double qx = __shfl(q.x, int(row & 63u)), qy = __shfl(q.y, int(row & 63u));
                // of each row, the first entry whose column is not below the
                // short one's (no borrow leaves a row: its highest bit is set)
                const uint64_t from = __ballot(have && (mt[u] & 0x100u) && c[u] >= cr), any = from | highs;
                const uint64_t met = from & any & ~(any - lows) & __ballot(c[u] == cr);
                const bool both = __builtin_amdgcn_inverse_ballot_w64(met);
                const double2 p = cmul2(in.a, v[u]);
                // one side only: + 0 as the reference's binop does
                const double2 x = make_double2(p.x + (both ? qx : 0.0), p.y + (both ? qy : 0.0));
                const bool keep = have && (x.x != 0.0 || x.y != 0.0);
                const uint64_t kept = __ballot(keep);
                const uint32_t k0 = uint32_t(kept) & mine0, k1 = uint32_t(kept >> 32) & mine1;
                uint32_t n = __popc(k0) + __popc(k1);
                uint32_t before = kFill ? __builtin_amdgcn_mbcnt_hi(k1, __builtin_amdgcn_mbcnt_lo(k0, 0)) : 0;
                const bool alone = row < rows && (mt[u] & 0x200u) &&
                                   ((uint32_t(met) & mine0) | (uint32_t(met >> 32) & mine1)) == 0;
                const uint32_t to = kFill ? uint32_t(__shfl(int(orel), int(row & 63u))) : 0;
                if (__any(alone)) {
                    const uint64_t mine = uint64_t(mine1) << 32 | mine0, above = from & mine;
                    const uint64_t below = (above & (0 - above)) - 1;  // the lanes before it, or all
                    const uint32_t at = uint32_t(__popcll(kept & mine & below));
                    if (kFill && alone && lane == 0 && at < mt[u] >> 16)
                        nt_store(cr, make_double2(0.0 + qx, 0.0 + qy), ixo + pw + to + at, dout + pw + to + at);
                    before += alone && !((below >> wl) & 1u) ? 1u : 0u;
                    n += alone ? 1u : 0u;
                }
                if (kFill) {
                    if (keep && before < mt[u] >> 16) nt_store(c[u], x, ixo + pw + to + before, dout + pw + to + before);
                } else {
                    // to the lane of the row
                    const uint32_t mine = uint32_t(__shfl(int(n), int((wl & (gw - 1u)) << lpr_log2)));
                    if (wl >> (6u - lpr_log2) == s + uint32_t(u)) count = mine;
                }
            }
        }
        if (!kFill && wl < rows && fits) counts[rw + wl] = count;
    }
    auto vote = [&](bool p) { return (__ballot(p) >> shift) & gmask; };
    // the rows left, the lowest gw of them at a time
    for (uint64_t rest = __ballot(wl < rows && !fits); rest;) {
        uint32_t row = 64;
        for (uint32_t g = 0; g < gw && rest; ++g, rest &= rest - 1)
            if (group == g) row = uint32_t(__builtin_ctzll(rest));
        const int src = int(row & 63u);
        uint64_t i = __shfl(i0, src), j = __shfl(j0, src), pos = __shfl(po, src);
        const uint64_t iend = __shfl(i1, src), jend = __shfl(j1, src), kend = __shfl(pe, src);
        if (row == 64) continue;
        uint64_t next = 0;
        double2 vnext = make_double2(0.0, 0.0);
        auto load = [&](uint64_t at) {
            if (at + lane < iend) {
                next = __builtin_nontemporal_load(in.ix1 + at + lane);
                vnext = nt_value(in.d1 + at + lane);
            }
        };
        load(i);
        for (;;) {
            const bool have = i + lane < iend, last = i + lpr >= iend;
            const uint64_t col = next;
            const double2 va = vnext;
            load(i + lpr);  // the piece after this one
            const double2 p = cmul2(in.a, va);
            double2 q = make_double2(0.0, 0.0);
            // the lane that a short entry of column cc meets, of those from
            // `left` on (lpr: none, it comes after them); whether it joins it
            uint32_t left = 0;
            auto meet = [&](uint64_t cc, uint32_t &f) {
                const uint64_t ge = vote(have && lane >= left && col >= cc);
                f = ge ? uint32_t(__builtin_ctzll(ge)) : lpr;
                const bool joins = ge && __shfl(col, int(f & (lpr - 1u)), int(lpr)) == cc;
                left = f + (joins ? 1u : 0u);
                return joins;
            };
            uint64_t je = j;
            for (; je < jend; ++je) {
                uint32_t f;
                const bool joins = meet(in.ix2[je], f);
                if (f == lpr && !last) break;  // the next piece's
                if (joins && lane == f) q = cmul2(in.b, in.d2[je]);
            }
            left = 0;
            const double2 x = make_double2(p.x + q.x, p.y + q.y);
            const bool keep = have && (x.x != 0.0 || x.y != 0.0);
            const uint64_t kept = vote(keep);
            uint32_t before = uint32_t(__popcll(kept & ((uint64_t(1) << lane) - 1))), nb = 0;
            for (uint64_t t = j; t < je; ++t) {
                const uint64_t cc = in.ix2[t];
                uint32_t f;
                if (meet(cc, f)) continue;
                const double2 y = cmul2(in.b, in.d2[t]), z = make_double2(0.0 + y.x, 0.0 + y.y);
                if (z.x == 0.0 && z.y == 0.0) continue;
                if (kFill) {
                    const uint64_t at = pos + uint32_t(__popcll(f < 64 ? kept & ((uint64_t(1) << f) - 1) : kept)) + nb;
                    if (lane == 0 && at < kend) nt_store(cc, z, ixo + at, dout + at);
                    if (lane >= f) ++before;
                }
                ++nb;
            }
            if (kFill && keep && pos + before < kend) nt_store(col, x, ixo + pos + before, dout + pos + before);
            pos += uint32_t(__popcll(kept)) + nb;
            if (last) break;
            i += lpr;
            j = je;
        }
        if (!kFill && lane == 0) counts[rw + row] = pos;
    }
}

// Whether k_spadd_few takes a sum, its lanes per row (a power of two from 4 to 64
// that holds the longer matrix's mean length, or, where the rows cannot be equal,
// what most of them have: mean + 2 sqrt(mean)), its rows per wave (64 or what
// leaves the launch 16 waves per CU, or 256 if rows come in pieces: 16-qubit
// molecule, fill pass, 16 / 64 / 256 waves per CU 612 / 563 / 498 us; 18-qubit ring
// 58 / 49 / 87; 33 entries, 16 qubits 97 / - / 213), and `in` with the longer matrix
// first.
// Rows of up to 64 entries in the mean: sums with as many short entries as rows
// (a diagonal, one Pauli string), where one each is what to expect.  Staged
// tiles / this, count + fill, us: 20 qubits, 4 to 64 random terms 570-900 /
// 500-600; isotropic rings without their zeros, 20, 22, 23, 24 qubits (10.6 to 12.7
// entries in the mean, 32 lanes but for 22) 364 / 323, 1433 / 1134, 3227 / 2268, 6138
// / 4711 (16 lanes: 3373, 7303); Poisson lengths of 7, 14, 22, 35, 20 qubits 265 /
// 250, 417 / 399, 598 / 520, 864 / 798 (the mean rounded up: 363, 517, 521, 728); one
// row in 100 of 600 entries 4360 / 656; but one or two entries per row, which idle
// most of four lanes, 23 qubits 595 / 667 (of the same columns 513 / 666), 670 / 764
// (three 893 / 917, below 2^22 rows equal), and 24 or 100 entries in every other row 432 / 595, 1120 /
// 1700 (a whole number in the mean).  Other sums stay with
// the tiles: rows with two short entries (Z + X) run one at a time here, 20-qubit
// ring 657 / 1290, 0 to 2 each 600 / 900 (and as many as rows, alternately 0 and 2,
// 23 qubits 4780 / 6800).
// Longer rows, which leave the tiles few rows or overflow them: from 128 entries
// per row with one short one, 192 with two.  One / two short entries: 90
// entries 1012 / 1055, 972 / 1280; 128: 784 / 666, 772 / 763; 220: 811 / 535,
// 828 / 578; 400: 1084 / 868, 1097 / 952; 600: 21200 / 685, 21300 / 676.
struct SpFew {
    uint32_t lpr_log2, rpw_log2;
    uint64_t blocks;
    bool pieces;
};
static bool spadd_few(uint64_t nrows, SpAddIn &in, SpFew &f) {
    if (in.nnz1 < in.nnz2) in = SpAddIn{in.b, in.a, in.nnz2, in.nnz1, in.ip2, in.ix2, in.ip1, in.ix1, in.d2, in.d1};
    const double mean = double(in.nnz1) / double(nrows ? nrows : 1);
    const double need = nrows && in.nnz1 % nrows ? mean + 2.0 * std::sqrt(mean) : mean;
    f.lpr_log2 = 2;
    while (f.lpr_log2 < 6 && double(1u << f.lpr_log2) < need) ++f.lpr_log2;
    f.pieces = mean > 64;
    if (f.pieces ? in.nnz2 == 0 || in.nnz2 > 2 * nrows || in.nnz1 / 64 < nrows + in.nnz2
                 : in.nnz2 != nrows || (in.nnz1 / 3 < nrows && nrows >> 22) || need > 64)
        return false;
    f.rpw_log2 = 6;
    const uint64_t waves = f.pieces ? 65536 : 4096;
    while (f.rpw_log2 > 6 - f.lpr_log2 && (nrows >> f.rpw_log2) < waves) --f.rpw_log2;
    f.blocks = (nrows + (uint64_t(4) << f.rpw_log2) - 1) / (uint64_t(4) << f.rpw_log2);
    return true;
}

// Rows per tile: the staged capacity over the mean merged row length, with
// room for rows up to 1/0.85 times the mean.  Lanes per row: enough that the
// tile's rows keep the block's threads busy (a power of two, at most 64).
struct SpTiling {
    uint32_t rows, lpr;
};
static SpTiling spadd_tiling(uint64_t nrows, uint64_t nnz1, uint64_t nnz2, int threads, int cap) {
    const double mean = double(nnz1 + nnz2) / double(nrows ? nrows : 1);
    const double r = mean > 0 ? 0.85 * cap / mean : double(threads);
    const uint32_t rows = r >= threads ? uint32_t(threads) : (r < 1 ? 1u : uint32_t(r));
    uint32_t lpr = 1;
    while (lpr < 64 && lpr * rows < uint32_t(threads)) lpr <<= 1;
    return SpTiling{rows, lpr};
}

__global__ void k_set_zero_u64(uint64_t *p) { *p = 0; }

// indptr of few rows: the counts at ipo[1 ..] become their inclusive sums, by
// one block, in place (the device scan takes three launches and a workspace of
// its own).  What bounds it: latency.  H - e*I, both calls, rings of 8, 12, 14
// qubits 70, 74, 73 -> 46, 46, 62 us.
constexpr uint32_t kScanSmallPer = 16;
__global__ __launch_bounds__(1024) void k_scan_small(uint32_t n, uint64_t *__restrict__ ipo) {
    __shared__ uint64_t waves[16];
    const uint32_t t = threadIdx.x, per = (n + 1023u) / 1024u, at = t * per, lane = t & 63u;
    uint64_t v[kScanSmallPer], sum = 0;
#pragma unroll
    for (uint32_t i = 0; i < kScanSmallPer; ++i) {
        v[i] = i < per && at + i < n ? ipo[1 + at + i] : 0;
        sum += v[i];
    }
    uint64_t incl = sum;
    for (uint32_t o = 1; o < 64; o <<= 1) {
        const uint64_t u = __shfl_up(incl, o);
        if (lane >= o) incl += u;
    }
    if (lane == 63) waves[t / 64] = incl;
    __syncthreads();
    uint64_t run = incl - sum;
    for (uint32_t w = 0; w < t / 64; ++w) run += waves[w];
    if (t == 0) ipo[0] = 0;
#pragma unroll
    for (uint32_t i = 0; i < kScanSmallPer; ++i) {
        run += v[i];
        if (i < per && at + i < n) ipo[1 + at + i] = run;
    }
}

static SpAddIn spadd_in(const double *a, uint64_t nnz1, const uint64_t *ip1, const uint64_t *ix1,
                        const double *d1, const double *b, uint64_t nnz2, const uint64_t *ip2,
                        const uint64_t *ix2, const double *d2) {
    return SpAddIn{make_double2(a[0], a[1]), make_double2(b[0], b[1]), nnz1, nnz2, ip1, ix1, ip2,
                   ix2, reinterpret_cast<const double2 *>(d1), reinterpret_cast<const double2 *>(d2)};
}

int launch_spadd_count(uint64_t nrows, const double *a, uint64_t nnz1, const uint64_t *ip1,
                       const uint64_t *ix1, const double *d1, const double *b, uint64_t nnz2,
                       const uint64_t *ip2, const uint64_t *ix2, const double *d2, uint64_t *ipo,
                       uint64_t *nnz_out, hipStream_t s) {
    SpAddIn in = spadd_in(a, nnz1, ip1, ix1, d1, b, nnz2, ip2, ix2, d2);
    const SpTiling tl = spadd_tiling(nrows, nnz1, nnz2, kSpCountThreads, kSpCountCap);
    SpFew f;
    const bool few = spadd_few(nrows, in, f);
    const uint64_t ntiles = few ? f.blocks : (nrows + tl.rows - 1) / tl.rows;
    if (ntiles > 0x7FFFFFFFull) return fail(QR_ERR_SIZE, "sparse add: too many row tiles");
    // per-row counts, then their inclusive scan into indptr[1..nrows]
    const bool small = nrows <= 1024 * kScanSmallPer;
    size_t tmp_bytes = 0;
    void *tmp = nullptr;
    const size_t cbytes = (size_t(nrows) * sizeof(uint64_t) + 255) & ~size_t(255);
    uint64_t *counts = ipo + 1;
    if (!small) {
        QR_HIP_CHECK(hipcub::DeviceScan::InclusiveSum(nullptr, tmp_bytes, ipo, ipo + 1, nrows, s));
        QR_HIP_CHECK(hipMallocAsync(&tmp, cbytes + tmp_bytes, s));
        counts = static_cast<uint64_t *>(tmp);
        hipLaunchKernelGGL(k_set_zero_u64, dim3(1), dim3(1), 0, s, ipo);
    }
    if (few)
        hipLaunchKernelGGL((f.pieces ? k_spadd_few<false, true> : k_spadd_few<false, false>), dim3(unsigned(ntiles)),
                           dim3(256), 0, s, nrows, f.lpr_log2, f.rpw_log2, in, counts, nullptr, nullptr, nullptr);
    else
        hipLaunchKernelGGL((k_spadd_tile<false, kSpCountThreads, kSpCountCap>), dim3(unsigned(ntiles)),
                           dim3(kSpCountThreads), 0, s, nrows, tl.rows, tl.lpr, in, counts, nullptr, nullptr, nullptr);
    hipError_t e = hipGetLastError();
    if (small) {
        hipLaunchKernelGGL(k_scan_small, dim3(1), dim3(1024), 0, s, uint32_t(nrows), ipo);
        if (e == hipSuccess) e = hipGetLastError();
    } else {
        if (e == hipSuccess)
            e = hipcub::DeviceScan::InclusiveSum(static_cast<unsigned char *>(tmp) + cbytes, tmp_bytes,
                                                 counts, ipo + 1, nrows, s);
        (void)hipFreeAsync(tmp, s);
    }
    if (e != hipSuccess) return hip_fail(e, "sparse add count / scan");
    QR_HIP_CHECK(hipMemcpyAsync(nnz_out, ipo + nrows, sizeof(uint64_t), hipMemcpyDeviceToHost, s));
    QR_HIP_CHECK(hipStreamSynchronize(s));
    return QR_OK;
}

int launch_spadd_fill(uint64_t nrows, const double *a, uint64_t nnz1, const uint64_t *ip1,
                      const uint64_t *ix1, const double *d1, const double *b, uint64_t nnz2,
                      const uint64_t *ip2, const uint64_t *ix2, const double *d2,
                      const uint64_t *ipo, uint64_t *ixo, double *dout, hipStream_t s) {
    SpAddIn in = spadd_in(a, nnz1, ip1, ix1, d1, b, nnz2, ip2, ix2, d2);
    const SpTiling tl = spadd_tiling(nrows, nnz1, nnz2, kSpFillThreads, kSpCap);
    SpFew f;
    const bool few = spadd_few(nrows, in, f);
    const uint64_t ntiles = few ? f.blocks : (nrows + tl.rows - 1) / tl.rows;
    if (ntiles > 0x7FFFFFFFull) return fail(QR_ERR_SIZE, "sparse add: too many row tiles");
    if (few)
        hipLaunchKernelGGL((f.pieces ? k_spadd_few<true, true> : k_spadd_few<true, false>), dim3(unsigned(ntiles)),
                           dim3(256), 0, s, nrows, f.lpr_log2, f.rpw_log2, in, nullptr, ipo, ixo,
                           reinterpret_cast<double2 *>(dout));
    else
        hipLaunchKernelGGL((k_spadd_tile<true, kSpFillThreads, kSpCap>), dim3(unsigned(ntiles)), dim3(kSpFillThreads),
                           0, s, nrows, tl.rows, tl.lpr, in, nullptr, ipo, ixo, reinterpret_cast<double2 *>(dout));
    QR_HIP_CHECK(hipGetLastError());
    return QR_OK;
}

}  // namespace qr
