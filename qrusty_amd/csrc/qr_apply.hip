// qr_apply.hip -- matrix-free Pauli-sum apply and <x|H|x> for gfx950.
//
// y_v[r] = sum_g D_g(r) * x_v[r ^ x_g],  D_g(r) = sum_{t in g} (-1)^popcount(r&z_t) c'_t
//
// This equals the rowwise CSR build followed by the CSR matvec
// (qrusty/src/accel.rs:171-210, 338-370) without materialising the 2^n*G
// entries: D_g(r) is the CSR value of group g in row r, x[r ^ x_g] the gather
// of its column.
//
// Work decomposition (one block = one tile of 2^L consecutive rows of one
// state vector: 256 threads, or 2 or 4 times as many that share the tile's
// groups, see apply_split; at most 40 KB of LDS, so that four blocks share a
// CU and some compute while others wait at a barrier or on their loads):
//  * The tile's slice of x is staged in LDS (LDS-DMA); groups whose x mask is
//    below 2^L gather from LDS, the others ("far" groups) gather the partner
//    tile t ^ (x_g >> L) from global memory (coalesced, permuted inside a
//    line).
//  * Blocks are ordered vector-major, and each XCD receives one contiguous
//    range of tiles of the vector: the far partners of nearby tiles are read
//    through the same L2, and one complex64 vector (128 MiB at 24 qubits)
//    stays resident in the 256 MB MALL while the chip works on it.
//  * Row r = h + l (h = tile base, l < 2^L):  (-1)^popcount(r & z) =
//    (-1)^popcount(h & z) * (-1)^popcount(l & zl), zl = z & (2^L - 1).  The
//    host merges the terms of a group that share zl into "patterns" and cuts
//    the patterns into parts whose zl span at most four dimensions.  Over the
//    tile a part's sum takes at most 16 values, which the block tabulates in
//    LDS (chunk_tables); the index of a row's value is linear in the bits of
//    l, so a thread finds it with a few shifts and XORs of two words of the
//    group's descriptor (ApplyPart) whatever the number of terms.  Summing the
//    signed coefficients per thread instead took 5-6 vector instructions per
//    pattern; molecules of 12 / 16 / 20 / 22 qubits, FP64, one state: 290 / 556
//    / 1633 / 10100 -> 35 / 114 / 890 / 5120 us, 20 qubits and 2000 random terms
//    1590 -> 1100.  What bounds them now (counters): the 20-qubit molecule the
//    LDS, four fifths of its 128 B per cycle (6.7 reads per group and wave), and
//    the vector ALU, 64% busy (34 instructions per group and 4 rows); the
//    28-qubit k-local operator, complex64, the vector ALU, 78% (90 per group
//    and 8 rows, with the tables); the 24-qubit complex64 ring the partners past
//    L2, 7.8 TB/s; small states the chain of descriptor loads, lookups and
//    gathers of each group.
//  * Thread `tid` owns rows l = tid + 256*k.  The gather form on full
//    complex64 tiles owns row pairs instead, l = 2*tid + (k & 1) + 512*(k >>
//    1), so that one 16-byte load gathers both partners of a pair and one
//    16-byte store writes both results; the patterns' low z bits are permuted
//    to match (row bit 0 counts with k).
//  * Partner-staged form (k_apply_staged): when many far groups share a
//    partner tile (their masks agree above the tile), the groups are ordered
//    by partner and each partner tile is loaded into LDS once, double-
//    buffered, instead of being gathered once per group.
//  * Window passes (ApplyWindow; FP64): groups whose partner tiles would be
//    read past L2 are applied in a second pass over tiles made of the low bits
//    and a window of high ones, where their masks stay inside the tile.
//
// Precision modes
//   FP64 : complex128 state (tile 2^10 rows, 4 rows per thread).
//   MIXED: complex64 state (tile 2^11 rows, 8 rows per thread), rounded to
//          complex64 once, when y is written.
// In both, D_g(r), the products and the sum over groups are FP64.  For the
// complex64 state that is also the cheapest arithmetic: FP64 FMAs and
// FP32 -> FP64 conversions issue at the rate of FP32 ones here (packed FP32 is
// off; measured 4.7-5.2 cycles per wave instruction and SIMD, all of them), so
// a row and group takes 2 conversions and 2 FMAs against 2 FMAs and the 3
// additions of a compensated FP32 sum (TwoSum every 4 groups) -- and its error
// is the rounding of y: 3.5e-8 against 4.7e-8 on the 24-qubit ring.
// <x|y> is reduced deterministically: per thread, per block (fixed tree),
// then one pass over the block partials of each vector.
#include "qr_internal.h"

#include <cstdlib>
#include <mutex>
#include <string>
#include <type_traits>

namespace qr {

// 256 threads and at most 40 KB of LDS per block: four blocks per CU (the
// 160 KB of a gfx950 CU).  Measured (24-qubit Heisenberg, 8 states; 28-qubit
// k-local, one state), by threads per block and tile:
//   1024, 2^13 / 2^12 rows (mixed / FP64): 1.80 / 3.75 ms; 252 / 422 ms
//    512, 2^12 / 2^11 rows:                1.75 / 3.66 ms; 237 / 398 ms
//    256, 2^11 / 2^10 rows:                1.64 / 3.47 ms; 228 / 400 ms
// although each halving of the tile adds a far group.  Fewer rows per thread
// on the same tiles (512 threads, 2^11 / 2^10 rows: 4 / 2 rows per thread,
// 72-88 VGPRs, 5-7 waves per SIMD) measured 1.84 / 3.59 ms and 278 / 436 ms
// against 1.63 / 3.50 and 238 / 401 with 256 threads (block partials summed
// in FP64 in both): the per-group work of a thread is shared by fewer rows.
// (All of these before the coefficients were tabulated.)
constexpr int kApplyThreads = 256;
constexpr int kApplyThreadBits = 8;
constexpr size_t kApplyMaxLDS = 40 * 1024;  // LDS of one block
constexpr size_t kApplyFewLDS = 80 * 1024;  // of kFormGatherFew: two blocks per CU
// of an operator with a group that needs more than a chunk's share of it
constexpr size_t kApplyLDSLimit = 160 * 1024;
// dynamic LDS that a launch may ask for without raising the kernel's limit
constexpr size_t kDefaultLDS = 64 * 1024;

// Tile of 2^L rows (x tile in LDS: 16 KB in both precisions at the default
// L; 8 KB for the small complex64 tiles), R rows per thread, and the LDS left
// for one chunk of tables.
//
// Small complex64 tiles (2^10 rows, 4 per thread) serve launches of fewer than
// two 2^11-row tiles per CU, with four thread groups per block (apply_split):
// one state, 2^11-row tiles and two thread groups / small tiles and four:
// molecules 12 / 16 / 18 qubits 64 / 200 / 321 -> 36 / 110 / 183 us.  From two
// tiles per CU on the larger ones win: 20 qubits 804 / 915, random 761 / 1009.
constexpr int kMixedSmallL = 10;
template <bool kMixed, int kL = kMixed ? 11 : 10>
struct ApplyShape {
    static constexpr int L = kL;
    static constexpr int R = (1 << L) / kApplyThreads;
    static constexpr size_t kTile = (size_t(1) << L) * (kMixed ? 8 : 16);
    // LDS for adding up the sums of `split` thread groups (merge_splits)
    static constexpr size_t merge_bytes(int split) { return size_t(split / 2) * R * kApplyThreads * 16; }
    // table bytes of one chunk, in the LDS after the x tile (gather form) or
    // after two tile buffers (partner-staged form); a group of more than
    // kPatSplit patterns is split, one that needs more than a chunk takes a
    // larger chunk of its own
    static constexpr uint32_t kPatSplit = 736, kPatSplitS = 224;
    static constexpr uint32_t kTabChunk = uint32_t(kApplyMaxLDS - kTile - 1024);
    static constexpr uint32_t kTabChunkS = uint32_t(kApplyMaxLDS - 2 * kTile - 1024);
};

template <bool kNarrow>
__device__ __forceinline__ uint32_t parity_of(uint64_t a, uint64_t b) {
    if (kNarrow) return __popc(uint32_t(a) & uint32_t(b)) & 1u;
    return __popcll(a & b) & 1u;
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int off = 32; off > 0; off /= 2) v += __shfl_xor(v, off, 64);
    return v;
}

// x(-1) when bit 31 of `flip` is set: the sign of a double flipped by an XOR
// of its high word.
__device__ __forceinline__ double flip_sign(double a, uint32_t flip) {
    return __hiloint2double(__double2hiint(a) ^ int(flip), __double2loint(a));
}

// Word 3 of a raw (untyped, stride 0) buffer resource on gfx9: 32-bit data
// format; offsets are bounds-checked against num_records bytes.
constexpr int kBufferWord3 = 0x00020000;

// Complex elements as builtin vectors: they load, store and copy across
// address spaces as one 8- or 16-byte access.
typedef float fvec2 __attribute__((ext_vector_type(2)));
typedef float fvec4 __attribute__((ext_vector_type(4)));
typedef double dvec2 __attribute__((ext_vector_type(2)));

typedef __attribute__((address_space(3))) unsigned char lds_byte;

// LDS by absolute byte address.  The tile buffers and tables are aligned to
// their sizes, so places in them are formed with XOR.  Both hold because the
// apply kernels' dynamic LDS begins at address 0: they have no static LDS
// (tests/test_apply_lds.py reads that from the built library).
template <typename T>
__device__ __forceinline__ T lds_load(uint32_t at) {
    return *(const __attribute__((address_space(3))) T *)(at);
}

// Gathers of x[r ^ m] for the R rows of a thread: from the LDS x tile (at
// LDS address xt), or -- for masks above the tile -- from the partner tile in
// global memory, with one uniform base pointer per row block and the
// thread's offset shared.
// With kPairs (complex64, full tiles) the thread's rows k = 2j, 2j+1 are the
// adjacent rows (2 tid, 2 tid + 1) + 2^9 j: their partners r ^ m form one
// aligned pair, read with one 16-byte load.  When bit 0 of m is set, row k's
// partner is xg[k ^ 1]: such groups form classes of their own, whose products
// read the pair crosswise (no data is moved).
template <bool kFar, bool kFull, bool kPairs, int R, typename cT>
__device__ __forceinline__ void gather(uint64_t m, uint32_t tid, uint64_t tile_rows, uint64_t base,
                                       uint32_t xt, const cT *__restrict__ xv, cT (&xg)[R]) {
    const uint64_t mhi = m & ~(tile_rows - 1);
    const uint32_t mlo = uint32_t(m & (tile_rows - 1));
    constexpr uint32_t kS = sizeof(cT);
    if constexpr (kPairs) {
        static_assert(sizeof(cT) == 8 && kFull && R % 2 == 0, "pairs: complex64, full tiles");
        constexpr int kJ = kApplyThreadBits + 1;  // row bit of the pair index j
        const uint32_t tq = tid ^ ((mlo >> 1) & (kApplyThreads - 1));
        fvec4 pr[R / 2];
        if (kFar) {
            const cT *far = xv + (base ^ mhi);
            const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<cT *>(far), 0, int(tile_rows * kS), kBufferWord3);
            const uint32_t jm = mlo >> kJ;
#pragma unroll
            for (int j = 0; j < R / 2; ++j) {
                const uint32_t soff = ((uint32_t(j) ^ jm) << kJ) * kS;
                pr[j] = __builtin_bit_cast(fvec4, __builtin_amdgcn_raw_buffer_load_b128(rs, tq * 2 * kS, soff, 0));
            }
        } else {
            const uint32_t at = xt + tq * 2 * kS + ((mlo >> kJ) << kJ) * kS;
#pragma unroll
            for (int j = 0; j < R / 2; ++j) pr[j] = lds_load<fvec4>(at ^ ((uint32_t(j) << kJ) * kS));
        }
#pragma unroll
        for (int j = 0; j < R / 2; ++j) {
            xg[2 * j] = fvec2{pr[j].x, pr[j].y};
            xg[2 * j + 1] = fvec2{pr[j].z, pr[j].w};
        }
        return;
    }
    const uint32_t tx = tid ^ (mlo & (kApplyThreads - 1));
    const uint32_t mk = mlo >> kApplyThreadBits;
    if (kFar) {
        // the partner tile through a buffer resource: the row block's offset
        // is a scalar, the thread's offset one VGPR shared by the R loads
        const cT *far = xv + (base ^ mhi);
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<cT *>(far), 0, int(tile_rows * kS), kBufferWord3);
#pragma unroll
        for (int k = 0; k < R; ++k) {
            if (!kFull && tid + uint64_t(k) * kApplyThreads >= tile_rows) break;
            const uint32_t soff = ((uint32_t(k) ^ mk) << kApplyThreadBits) * kS;
            if constexpr (sizeof(cT) == 8)
                xg[k] = __builtin_bit_cast(cT, __builtin_amdgcn_raw_buffer_load_b64(rs, tx * kS, soff, 0));
            else
                xg[k] = __builtin_bit_cast(cT, __builtin_amdgcn_raw_buffer_load_b128(rs, tx * kS, soff, 0));
        }
    } else {
        const uint32_t at = xt + tx * kS + (mk << kApplyThreadBits) * kS;
#pragma unroll
        for (int k = 0; k < R; ++k) {
            if (!kFull && tid + uint64_t(k) * kApplyThreads >= tile_rows) break;
            xg[k] = lds_load<cT>(at ^ ((uint32_t(k) << kApplyThreadBits) * kS));
        }
    }
}

// The thread's places in the index words of a part (ApplyPart): nibble shifts
// of its thread bits 0-2 and 3-5, byte shift of its wave.
struct TabView {
    uint32_t sh0, sh1, shw;
};

__device__ __forceinline__ TabView tab_view(uint32_t tid) {
    const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(tid >> 6)));
    return {(tid & 7u) * 4u, ((tid >> 3) & 7u) * 4u, wave * 8u};
}

// LDS address of the thread's value (row index 0) in a part's table of
// elements of 2^kLg bytes; row k's is the same XOR byte k of rc.
template <int kLg>
__device__ __forceinline__ uint32_t tab_place(const TabView &tv, uint32_t w0, uint32_t w1, uint32_t w2,
                                              uint32_t tab) {
    const uint32_t t = ((w0 >> tv.sh0) ^ (w1 >> tv.sh1)) & 15u;
    return ((t << kLg) + (tab << 2)) ^ ((w2 >> tv.shw) & 0xffu);
}

// y += D_g(r) x[r ^ m] for the R rows of a thread, in FP64.  fetch() gathers
// x into xg (row k's partner in xg[k], or in xg[k ^ 1] with kSwap).  D_g is
// read from the chunk's tables: one value per row, or -- groups without a
// row-index bit in their patterns -- one per thread; groups of several parts
// add their parts' values.  kCplx: complex tables; groups with real
// coefficients skip the products with Im D.  next() loads the next group's
// descriptor once this one's LDS reads have returned (scalar loads share
// their counter and return out of order), ahead of the products.
template <bool kFull, bool kCplx, bool kSwap, int R, typename cT, typename Fetch, typename Next>
__device__ __forceinline__ void accumulate(const ApplyGroup &gd, const ApplyPart *__restrict__ part,
                                           uint32_t tid, uint64_t tile_rows, const TabView &tv, cT (&xg)[R],
                                           Fetch fetch, Next next, double (&ar)[R], double (&ai)[R]) {
    constexpr int kLg = 3 + int(kCplx);
    using dT = typename std::conditional<kCplx, dvec2, double>::type;
    fetch();
    dT d[R];
    if (gd.nparts() == 1) {
        const uint32_t at = tab_place<kLg>(tv, gd.w0, gd.w1, gd.w2, gd.tab());
        d[0] = lds_load<dT>(at);
        if (gd.tab_n & kGroupRowvar) {
#pragma unroll
            for (int k = 1; k < R; ++k) d[k] = lds_load<dT>(at ^ uint32_t((gd.rc >> (8 * k)) & 0xffu));
        } else {
#pragma unroll
            for (int k = 1; k < R; ++k) d[k] = d[0];
        }
    } else {
#pragma unroll
        for (int k = 0; k < R; ++k) d[k] = dT(0.0);
        const uint32_t q1 = gd.w0 + gd.nparts();
        for (uint32_t q = gd.w0; q < q1; ++q) {
            const ApplyPart ap = part[q];
            const uint32_t at = tab_place<kLg>(tv, ap.w0, ap.w1, ap.w2, ap.tab);
#pragma unroll
            for (int k = 0; k < R; ++k) d[k] += lds_load<dT>(at ^ uint32_t((ap.rc >> (8 * k)) & 0xffu));
        }
    }
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    next();
    // (keeps the compiler from sinking the load back to its use)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int k = 0; k < R; ++k) {
        if (!kFull && tid + uint64_t(k) * kApplyThreads >= tile_rows) break;
        const cT xb = xg[k ^ int(kSwap)];
        double dr;
        if constexpr (kCplx) dr = d[k].x;
        else dr = d[k];
        ar[k] = fma(dr, double(xb.x), ar[k]);
        ai[k] = fma(dr, double(xb.y), ai[k]);
    }
    if constexpr (kCplx) {
        if (gd.tab_n & kGroupCplx) {
#pragma unroll
            for (int k = 0; k < R; ++k) {
                if (!kFull && tid + uint64_t(k) * kApplyThreads >= tile_rows) break;
                const cT xb = xg[k ^ int(kSwap)];
                ar[k] = fma(-d[k].y, double(xb.y), ar[k]);
                ai[k] = fma(d[k].y, double(xb.x), ai[k]);
            }
        }
    }
}

// Sum of the kSplit thread groups' accumulators, in thread group 0: a fixed
// tree, through LDS (kSplit / 2 x R x 256 values at `area`; the block's other
// uses of it are over).
template <int kSplit, int R>
__device__ __forceinline__ void merge_splits(dvec2 *area, uint32_t tid, uint32_t sub, double (&ar)[R],
                                             double (&ai)[R]) {
#pragma unroll
    for (int h = kSplit / 2; h >= 1; h /= 2) {
        __syncthreads();
        if (sub >= uint32_t(h) && sub < uint32_t(2 * h)) {
#pragma unroll
            for (int k = 0; k < R; ++k)
                area[(uint32_t(sub - h) * R + k) * kApplyThreads + tid] = dvec2{ar[k], ai[k]};
        }
        __syncthreads();
        if (sub < uint32_t(h)) {
#pragma unroll
            for (int k = 0; k < R; ++k) {
                const dvec2 v = area[(sub * R + k) * kApplyThreads + tid];
                ar[k] += v.x;
                ai[k] += v.y;
            }
        }
    }
}

// The end of a tile: y of the thread's rows, and the block's <x|y> partial.  y
// is written once and not read again by the kernel: nontemporal stores, so that
// it does not displace x, which the partner tiles still gather, from the caches.
// row(l) is the state's row of the tile's row l, x(l) its element.  add: y
// and the partial are added to (a window pass after another pass).
template <bool kFull, bool kPairs, int kSplit, int R, typename cT, typename Row, typename X>
__device__ __forceinline__ void finish_tile(uint32_t tid, uint32_t sub, uint64_t tile_rows, bool add, Row row, X x,
                                            cT *__restrict__ yv, double *__restrict__ partials, double *red,
                                            const double (&ar)[R], const double (&ai)[R]) {
    double er = 0.0, ei = 0.0;
    if (kSplit == 1 || sub == 0) {
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const uint64_t l = kPairs ? ((uint64_t(tid) << 1) | uint64_t(k & 1) |
                                         (uint64_t(k >> 1) << (kApplyThreadBits + 1)))
                                      : tid + uint64_t(k) * kApplyThreads;
            if (!kFull && l >= tile_rows) break;
            using eT = decltype(cT{}.x + cT{}.x);
            if (yv) {
                if constexpr (kPairs) {
                    // the pair's two rows in one 16-byte store, at the odd row
                    if (k & 1) {
                        __builtin_nontemporal_store(
                            fvec4{float(ar[k - 1]), float(ai[k - 1]), float(ar[k]), float(ai[k])},
                            reinterpret_cast<fvec4 *>(yv + row(l - 1)));
                    }
                } else {
                    cT *at = yv + row(l);
                    cT was = {0, 0};
                    if (add) was = __builtin_nontemporal_load(at);
                    __builtin_nontemporal_store(cT{eT(ar[k] + was.x), eT(ai[k] + was.y)}, at);
                }
            }
            if (partials) {
                const cT xr = x(l);
                const double xa = xr.x, xb = xr.y;
                er = fma(xa, ar[k], er); er = fma(xb, ai[k], er);
                ei = fma(xa, ai[k], ei); ei = fma(-xb, ar[k], ei);
            }
        }
    }
    if (partials) {
        __syncthreads();  // red shares LDS with the tables
        const double a = wave_sum(er), b = wave_sum(ei);
        if (sub == 0 && (tid & 63) == 0) {
            red[2 * (tid / 64)] = a;
            red[2 * (tid / 64) + 1] = b;
        }
        __syncthreads();
        if (sub == 0 && tid == 0) {
            double s0 = 0.0, s1 = 0.0;
            for (int w = 0; w < kApplyThreads / 64; ++w) { s0 += red[2 * w]; s1 += red[2 * w + 1]; }
            double *at = partials + 2 * uint64_t(blockIdx.x);
            at[0] = add ? at[0] + s0 : s0;
            at[1] = add ? at[1] + s1 : s1;
        }
    }
}

// A_p = sum_t (-1)^popcount(base & z_t) c'_t over the pattern's terms
// [t0, t1), in term order.  The loads of four terms are issued together; the
// sum itself stays sequential.
template <bool kNarrow>
__device__ __forceinline__ double2 pattern_coeff(uint64_t base, uint32_t t0, uint32_t t1,
                                                 const uint64_t *__restrict__ ptz,
                                                 const double2 *__restrict__ ptc) {
    double a_r = 0.0, a_i = 0.0;
    uint32_t t = t0;
    for (; t + 4 <= t1; t += 4) {
        double2 cc[4];
        uint32_t par[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            cc[j] = ptc[t + j];
            par[j] = parity_of<kNarrow>(base, ptz[t + j]);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (par[j]) { a_r -= cc[j].x; a_i -= cc[j].y; }
            else { a_r += cc[j].x; a_i += cc[j].y; }
        }
    }
    for (; t < t1; ++t) {
        const double2 cc = ptc[t];
        if (parity_of<kNarrow>(base, ptz[t])) { a_r -= cc.x; a_i -= cc.y; }
        else { a_r += cc.x; a_i += cc.y; }
    }
    return make_double2(a_r, a_i);
}

// LDS: x tile (gather form) or two tile buffers (partner-staged form) | tables;
// at the end the split's sums take over the tables (gather form) or all of it
// (partner-staged), and the <x|y> partials the first bytes.
__host__ __device__ inline size_t apply_lds_bytes(size_t tiles, uint32_t max_tab, size_t merge) {
    const size_t all = tiles + ((size_t(max_tab) + 15) & ~size_t(15));
    return all > merge + 64 ? all : merge + 64;
}

// One LDS-DMA load: each lane reads the 16 bytes at its `src`, and the wave
// writes them to LDS at lds + lane * 16 (lds: LDS byte address, wave-uniform,
// passed in M0; one wait state between the M0 write and the load).  Written
// as inline asm so that the compiler, which cannot tell the buffer being
// filled from the one being read, does not wait for the load before every
// later LDS read; the caller waits for it (vmcnt) and synchronises the block
// before reading what it wrote.  It has no register result.
// M0 is a reserved register that the compiler may hold a value in across the
// statement, so the asm saves it in an SGPR of its own and restores it after
// the load is issued (the load reads M0 at issue: back-to-back loads with
// different M0 values each land at their own address).
__device__ __forceinline__ void lds_dma16(const void *src, uint32_t lds) {
    uint32_t saved;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %2\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %1, off\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(saved)
        : "v"(src), "s"(lds)
        : "memory");
}

// v of the lane whose number differs in bit `kBit` of the 16 lanes of a DPP
// row: XOR 1 and 2 are quad permutations, XOR 4 and 8 a mirror (XOR 7 of 8
// lanes, 15 of 16) undone on the lower bits.
template <int kBit>
__device__ __forceinline__ double row_xor(double v) {
    auto dpp = [](int w) {
        auto mov = [](int x, auto ctrl) {
            return __builtin_amdgcn_update_dpp(0, x, decltype(ctrl)::value, 0xf, 0xf, true);
        };
        using Xor1 = std::integral_constant<int, 0xB1>;    // quad_perm [1, 0, 3, 2]
        using Xor2 = std::integral_constant<int, 0x4E>;    // quad_perm [2, 3, 0, 1]
        using Xor3 = std::integral_constant<int, 0x1B>;    // quad_perm [3, 2, 1, 0]
        using Xor15 = std::integral_constant<int, 0x140>;  // row_mirror
        using Xor7 = std::integral_constant<int, 0x141>;   // row_half_mirror
        if constexpr (kBit == 1) return mov(w, Xor1{});
        else if constexpr (kBit == 2) return mov(w, Xor2{});
        else if constexpr (kBit == 4) return mov(mov(w, Xor7{}), Xor3{});
        else return mov(mov(w, Xor15{}), Xor7{});
    };
    return __hiloint2double(dpp(__double2hiint(v)), dpp(__double2loint(v)));
}

// Per-chunk LDS tables of a tile, 16 lanes per part: lane c forms
// A_c = sum_t (-1)^popcount(base & z_t) c'_t of the part's pattern of code c,
// and a Walsh-Hadamard transform over the lanes turns the A_c into the
// table's entries, entry e = sum_c (-1)^popcount(e & c) A_c.  Ends with a wait
// for the wave's own global loads and a barrier.
template <bool kNarrow, bool kCplx, uint32_t kThreads>
__device__ __forceinline__ void chunk_tables(const ApplyChunk &ch, uint32_t t, uint64_t base,
                                             const uint32_t *__restrict__ tab,
                                             const ApplyRange *__restrict__ pat,
                                             const uint64_t *__restrict__ ptz,
                                             const double2 *__restrict__ ptc, unsigned char *smem) {
    const uint32_t c = t & 15u;
    // (the lanes of a part stay in the loop together)
    for (uint32_t i = ch.t0 + t / 16u; i < ch.t1; i += kThreads / 16) {
        const ApplyRange pr = pat[16 * uint64_t(i) + c];
        const uint32_t place = tab[i];
        double2 v = pattern_coeff<kNarrow>(base, pr.t0, pr.t1, ptz, ptc);
        auto stage = [&](auto bit_t) {
            constexpr int kBit = decltype(bit_t)::value;
            const double ox = row_xor<kBit>(v.x);
            v.x = ox + ((c & kBit) ? -v.x : v.x);
            if (kCplx) {
                const double oy = row_xor<kBit>(v.y);
                v.y = oy + ((c & kBit) ? -v.y : v.y);
            }
        };
        stage(std::integral_constant<int, 1>{});
        stage(std::integral_constant<int, 2>{});
        stage(std::integral_constant<int, 4>{});
        stage(std::integral_constant<int, 8>{});
        if (c < (place >> 16)) {
            unsigned char *at = smem + 4u * (place & 0xffffu);
            if (!kCplx) reinterpret_cast<double *>(at)[c] = v.x;
            else reinterpret_cast<double2 *>(at)[c] = v;
        }
    }
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): LDS-DMA of the caller's tile
    __syncthreads();
}

// kWin: a window pass (ApplyWindow), whose groups all gather inside the tile;
// win_add: it adds to y and the partials.  kParts: vector v of y is the sum over
// the v-th share of the groups of one state (launch_apply_parts).  nchunk is at
// least 1: the wait for the tile's loads is chunk_tables'.
template <bool kMixed, bool kNarrow, bool kCplx, bool kFull, int kL, int kSplit, bool kWin, bool kParts>
__global__ __launch_bounds__(kApplyThreads * kSplit) void k_apply_tiled(
    uint64_t N, ApplyWindow win, uint32_t ntiles, uint32_t tiles_per_xcd, uint32_t nchunk, uint32_t win_add,
    const ApplyGroup *__restrict__ grp, const ApplyChunk *__restrict__ chunks,
    const ApplyPart *__restrict__ part, const uint32_t *__restrict__ tab,
    const ApplyRange *__restrict__ pat, const uint64_t *__restrict__ ptz,
    const double2 *__restrict__ ptc, const void *__restrict__ xin, void *__restrict__ yout,
    double *__restrict__ partials) {
    using Shape = ApplyShape<kMixed, kL>;
    constexpr int L = Shape::L, R = Shape::R;
    // complex64 full tiles: paired rows (see gather); the patterns are built
    // in the paired-row bit order to match
    constexpr bool kPairs = kMixed && kFull;
    using cT = typename std::conditional<kMixed, fvec2, dvec2>::type;
    extern __shared__ __align__(256) unsigned char smem_raw[];

    const uint32_t tid = threadIdx.x % kApplyThreads;
    const uint32_t sub =
        kSplit == 1 ? 0u : uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x / kApplyThreads)));
    const uint32_t v = blockIdx.x / ntiles;
    uint32_t tile = blockIdx.x % ntiles;
    if (tiles_per_xcd) tile = (tile % 8) * tiles_per_xcd + tile / 8;
    const uint64_t tile_rows = kFull ? (uint64_t(1) << L) : (N < (uint64_t(1) << L) ? N : (uint64_t(1) << L));
    // the tile's row 0, and row l of it
    uint64_t base = uint64_t(tile) * tile_rows;
    if (kWin) {
        const uint32_t mid = win.s - win.f;  // tile index bits below the window
        base = (uint64_t(tile & ((1u << mid) - 1u)) << win.f) | (uint64_t(tile >> mid) << (win.s + L - win.f));
    }
    auto row = [&](uint64_t l) {
        return kWin ? base + ((l & ((1u << win.f) - 1u)) | ((l >> win.f) << win.s)) : base + l;
    };
    const cT *__restrict__ xv = reinterpret_cast<const cT *>(xin) + uint64_t(kParts ? 0u : v) * N;
    // the thread group's share of the groups: every `stride`-th from `share` on
    const uint32_t share = kParts ? v * kSplit + sub : sub;
    const uint32_t stride = kParts ? gridDim.x / ntiles * kSplit : uint32_t(kSplit);

    cT *xt = reinterpret_cast<cT *>(smem_raw);
    const uint32_t lds0 = uint32_t(uintptr_t((lds_byte *)smem_raw));
    const TabView tv = tab_view(tid);

    // the tile: straight into LDS, 16 bytes per lane, in flight while the
    // first chunk's tables are formed
    if constexpr (kFull) {
        constexpr uint32_t kThreads = kApplyThreads * kSplit, kPer = 16 / sizeof(cT);
        const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x / 64)));
#pragma unroll
        for (uint32_t i = 0; i < (uint32_t(Shape::kTile) - 1) / (16 * kThreads) + 1; ++i) {
            const uint32_t off = (i * kThreads + wave * 64u) * 16u;
            if (Shape::kTile % (16u * kThreads) != 0 && off >= Shape::kTile) break;
            lds_dma16(xv + row((off / 16u + threadIdx.x % 64u) * kPer), lds0 + off);
        }
    } else {
        for (uint64_t i = threadIdx.x; i < tile_rows; i += kApplyThreads * kSplit) xt[i] = xv[row(i)];
    }

    double ar[R], ai[R];
#pragma unroll
    for (int k = 0; k < R; ++k) ar[k] = ai[k] = 0.0;
    cT xg[R];
    for (uint32_t c = 0; c < nchunk; ++c) {
        const ApplyChunk ch = chunks[c];
        if (c) __syncthreads();  // the previous chunk's tables are no longer read
        chunk_tables<kNarrow, kCplx, kApplyThreads * kSplit>(ch, threadIdx.x, base, tab, pat, ptz, ptc,
                                                             smem_raw);
        auto run_class = [&](auto far_t, auto swap_t, int cls) {
            constexpr bool kFar = decltype(far_t)::value, kSwap = decltype(swap_t)::value;
            const uint32_t g1 = ch.cg[cls + 1];
            // (in the order of the chunk)
            uint32_t g = ch.cg[cls];
            if constexpr (kParts) g += (share - (ch.cg[cls] - ch.cg[0])) & (stride - 1);
            else if constexpr (kSplit > 1) g += (share - (ch.cg[cls] - ch.cg[0])) % kSplit;
            if (g >= g1) return;
            ApplyGroup nx = grp[g];
            do {
                const ApplyGroup gd = nx;
                // all descriptor fields in SGPRs before the gathers are issued,
                // so that no later scalar-load wait also waits for them
                asm volatile("" ::"s"(gd.m), "s"(gd.w0), "s"(gd.w1), "s"(gd.w2), "s"(gd.tab_n), "s"(gd.rc));
                g += stride;
                const auto fetch = [&]() {
                    gather<kFar, kFull, kPairs, R>(gd.m, tid, tile_rows, base, lds0, xv, xg);
                };
                const auto next = [&]() { nx = grp[g < g1 ? g : g1 - 1]; };
                accumulate<kFull, kCplx, kSwap, R>(gd, part, tid, tile_rows, tv, xg, fetch, next, ar, ai);
            } while (g < g1);
        };
        using F = std::false_type;
        using T = std::true_type;
        run_class(F{}, F{}, 0);
        if constexpr (kPairs) run_class(F{}, T{}, 1);
        if constexpr (!kWin) {
            run_class(T{}, F{}, 2);
            if constexpr (kPairs) run_class(T{}, T{}, 3);
        }
    }
    // the sums are added up where the tables were, so that <x|y> takes x from the
    // tile (y and energy, read again / this, us: 26 qubits, 1, 8 groups 569 / 512, 689
    // / 571, rings of 23, 24 qubits 205 / 192, 376 / 359; 574 for the 8 groups before
    // there were two thread groups)
    if (kSplit > 1) merge_splits<kSplit, R>(reinterpret_cast<dvec2 *>(smem_raw + Shape::kTile), tid, sub, ar, ai);
    const auto x = [&](uint64_t l) { return xt[l]; };
    finish_tile<kFull, kPairs, kSplit, R, cT>(tid, sub, tile_rows, kWin && win_add, row, x,
                                              yout ? reinterpret_cast<cT *>(yout) + uint64_t(v) * N : nullptr,
                                              partials, reinterpret_cast<double *>(smem_raw), ar, ai);
}

// Partner-staged form of k_apply_tiled (full tiles only).  Instead of one
// tile of x in LDS and far gathers from global memory, two tile buffers take
// the partner tiles t ^ hi in turn, one per run of groups sharing hi (hi = 0:
// the tile itself), so a partner tile is read once per chunk however many
// groups use it.  The load of run r + 1 (LDS-DMA: global memory straight into
// LDS, no registers) is in flight while run r is computed.
// Eight rows per thread and complex tables take 128 VGPRs, and no more: one above
// halves the blocks of two thread groups per CU (random, complex coefficients, 23
// qubits, 1000 terms 4360 / 8790 us, 24 qubits, 300 terms 3200 / 5015).
template <bool kMixed, bool kNarrow, bool kCplx, int kL, int kSplit, bool kParts>
__global__ __launch_bounds__(kApplyThreads * kSplit, kL == 11 ? 4 : 1) void k_apply_staged(
    uint64_t N, uint32_t ntiles, uint32_t tiles_per_xcd, uint32_t nchunk, uint32_t nrun,
    const ApplyGroup *__restrict__ grp,
    const ApplyChunk *__restrict__ chunks, const ApplyRun *__restrict__ runs,
    const ApplyPart *__restrict__ part, const uint32_t *__restrict__ tab,
    const ApplyRange *__restrict__ pat, const uint64_t *__restrict__ ptz,
    const double2 *__restrict__ ptc, const void *__restrict__ xin, void *__restrict__ yout,
    double *__restrict__ partials) {
    using Shape = ApplyShape<kMixed, kL>;
    constexpr int L = Shape::L, R = Shape::R;
    using cT = typename std::conditional<kMixed, fvec2, dvec2>::type;
    constexpr uint64_t tile_rows = uint64_t(1) << L;
    constexpr uint32_t kThreads = kApplyThreads * kSplit;
    constexpr uint32_t kStageTileBytes = uint32_t(Shape::kTile);  // one stage buffer: one tile
    constexpr uint32_t kLoads = (kStageTileBytes - 1) / (16u * kThreads) + 1;  // 16-byte loads per thread
    static_assert(tile_rows * sizeof(cT) == kStageTileBytes, "a tile fills one stage buffer");
    static_assert(kStageTileBytes % 1024 == 0, "tile must split into the waves' 16-byte loads");
    extern __shared__ __align__(256) unsigned char smem_raw[];

    const uint32_t tid = threadIdx.x % kApplyThreads;
    const uint32_t wave = uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x / 64)));
    const uint32_t sub = kSplit == 1 ? 0u : wave / (kApplyThreads / 64);
    const uint32_t v = blockIdx.x / ntiles;
    uint32_t tile = blockIdx.x % ntiles;
    if (tiles_per_xcd) tile = (tile % 8) * tiles_per_xcd + tile / 8;
    const uint64_t base = uint64_t(tile) * tile_rows;
    const cT *__restrict__ xv = reinterpret_cast<const cT *>(xin) + uint64_t(kParts ? 0u : v) * N;
    // the thread group's share of the groups: every `stride`-th from `share` on
    const uint32_t share = kParts ? v * kSplit + sub : sub;
    const uint32_t stride = kParts ? gridDim.x / ntiles * kSplit : uint32_t(kSplit);

    const uint32_t lds0 = uint32_t(uintptr_t((lds_byte *)smem_raw));
    const TabView tv = tab_view(tid);

    // partner tile base ^ hi into buffer b: each wave fills 1 KB per load,
    // lane i the 16 bytes at i * 16
    auto stage = [&](uint64_t hi, uint32_t b) {
        const unsigned char *src = reinterpret_cast<const unsigned char *>(xv + (base ^ hi));
#pragma unroll
        for (uint32_t j = 0; j < kLoads; ++j) {
            const uint32_t off = (j * kThreads + wave * 64u) * 16u;
            if (kStageTileBytes % (16u * kThreads) != 0 && off >= kStageTileBytes) break;
            lds_dma16(src + off + (threadIdx.x % 64u) * 16u, lds0 + b * kStageTileBytes + off);
        }
    };

    double ar[R], ai[R];
#pragma unroll
    for (int k = 0; k < R; ++k) ar[k] = ai[k] = 0.0;
    cT xg[R];
    if (nrun) stage(runs[0].hi, 0);
    uint32_t r = 0, g = share;
    const uint32_t glast = nrun ? runs[nrun - 1].g1 - 1 : 0;
    ApplyGroup nx = grp[g < glast ? g : glast];
    for (uint32_t c = 0; c < nchunk; ++c) {
        const ApplyChunk ch = chunks[c];
        if (c) __syncthreads();  // the previous chunk's tables are no longer read
        chunk_tables<kNarrow, kCplx, kThreads>(ch, threadIdx.x, base, tab, pat, ptz, ptc, smem_raw);
        for (; r < ch.r1; ++r) {
            // run r's tile has landed (each wave waits for its own loads, the
            // barrier for all of them), and no wave still reads run r - 1's
            // buffer, which the next load overwrites
            __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
            __syncthreads();
            if (r + 1 < nrun) stage(runs[r + 1].hi, (r + 1) & 1u);
            // the thread group's share of the run's groups, gathering from that tile
            const uint32_t g1 = runs[r].g1, xt = lds0 + (r & 1u) * kStageTileBytes;
            while (g < g1) {
                const ApplyGroup gd = nx;
                asm volatile("" ::"s"(gd.m), "s"(gd.w0), "s"(gd.w1), "s"(gd.w2), "s"(gd.tab_n), "s"(gd.rc));
                g += stride;
                const auto fetch = [&]() {
                    gather<false, true, false, R>(gd.m, tid, tile_rows, base, xt, xv, xg);
                };
                const auto next = [&]() { nx = grp[g < glast ? g : glast]; };
                accumulate<true, kCplx, false, R>(gd, part, tid, tile_rows, tv, xg, fetch, next, ar, ai);
            }
        }
    }
    if (kSplit > 1) merge_splits<kSplit, R>(reinterpret_cast<dvec2 *>(smem_raw), tid, sub, ar, ai);
    const auto row = [base](uint64_t l) { return base + l; };
    // (the buffers hold partner tiles)
    const auto x = [&](uint64_t l) { return xv[base + l]; };
    finish_tile<true, false, kSplit, R, cT>(tid, sub, tile_rows, false, row, x,
                                            yout ? reinterpret_cast<cT *>(yout) + uint64_t(v) * N : nullptr,
                                            partials, reinterpret_cast<double *>(smem_raw), ar, ai);
}

// out[2v], out[2v+1] = sum of the ntiles block partials of vector v
__global__ __launch_bounds__(256) void k_reduce_partials(uint32_t ntiles,
                                                         const double *__restrict__ partials,
                                                         double *__restrict__ out) {
    const uint32_t v = blockIdx.x;
    double a = 0.0, b = 0.0;
    for (uint32_t i = threadIdx.x; i < ntiles; i += 256) {
        a += partials[2 * (uint64_t(v) * ntiles + i)];
        b += partials[2 * (uint64_t(v) * ntiles + i) + 1];
    }
    __shared__ double ra[256], rb[256];
    ra[threadIdx.x] = a;
    rb[threadIdx.x] = b;
    __syncthreads();
    for (int s = 128; s > 0; s /= 2) {
        if (int(threadIdx.x) < s) {
            ra[threadIdx.x] += ra[threadIdx.x + s];
            rb[threadIdx.x] += rb[threadIdx.x + s];
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) { out[2 * v] = ra[0]; out[2 * v + 1] = rb[0]; }
}

// y = the sum of its parts y_p (launch_apply_parts), in order
__global__ __launch_bounds__(256) void k_sum_parts(uint32_t n, uint32_t parts, const dvec2 *__restrict__ from,
                                                   dvec2 *__restrict__ y) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= n) return;
    dvec2 v = from[i];
    for (uint32_t p = 1; p < parts; ++p) v += from[uint64_t(p) * n + i];
    y[i] = v;
}

template <bool kMixed, bool kNarrow, int kL, int kSplit, bool kWin = false, bool kParts = false>
static int launch_tiled(const qr_op *op, DeviceTables *t, int slot, uint32_t nvec, const void *d_x,
                        void *d_y, double *partials, uint32_t ntiles, hipStream_t s, bool few = false,
                        bool add = false) {
    using Shape = ApplyShape<kMixed, kL>;
    const uint64_t N = uint64_t(1) << op->nq;
    const uint64_t tile_rows = N < (uint64_t(1) << Shape::L) ? N : (uint64_t(1) << Shape::L);
    const DeviceTables::Patterns &pt = t->pat[slot];
    size_t shmem = Shape::kTile + apply_lds_bytes(0, pt.max_tab, Shape::merge_bytes(kSplit));
    if (few && shmem < kApplyFewLDS) shmem = kApplyFewLDS;
    if (shmem > kApplyLDSLimit) return fail(QR_ERR_SIZE, "apply: LDS stage too large");
    const uint32_t tpx = (ntiles % 8 == 0) ? ntiles / 8 : 0;
    const bool full = tile_rows == (uint64_t(1) << Shape::L);
    auto pick = [&](auto cplx_t) {
        constexpr bool kC = decltype(cplx_t)::value;
        return full ? k_apply_tiled<kMixed, kNarrow, kC, true, kL, kSplit, kWin, kParts>
                    : k_apply_tiled<kMixed, kNarrow, kC, false, kL, kSplit, false, false>;
    };
    auto kern = pt.cplx ? pick(std::true_type{}) : pick(std::false_type{});
    if ((kWin || kParts) && !full) return fail(QR_ERR_ARG, "apply: partial tiles");
    if (shmem > kDefaultLDS)
        QR_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, int(shmem)));
    const uint64_t nblocks = uint64_t(ntiles) * nvec;
    if (nblocks > 0x7FFFFFFFull) return fail(QR_ERR_SIZE, "apply grid too large");
    hipLaunchKernelGGL(kern, dim3(unsigned(nblocks)), dim3(kApplyThreads * kSplit), shmem, s, N, pt.win, ntiles,
                       tpx, pt.nchunk, uint32_t(add), pt.grp, pt.chunk, pt.part, pt.tab, pt.pat,
                       pt.ptz, pt.ptc, d_x, d_y, partials);
    QR_HIP_CHECK(hipGetLastError());
    return QR_OK;
}

template <bool kMixed, bool kNarrow, int kL, int kSplit, bool kParts = false>
static int launch_staged(const qr_op *op, DeviceTables *t, int slot, uint32_t nvec, const void *d_x,
                         void *d_y, double *partials, uint32_t ntiles, hipStream_t s) {
    using Shape = ApplyShape<kMixed, kL>;
    const uint64_t N = uint64_t(1) << op->nq;
    const DeviceTables::Patterns &pt = t->pat[slot];
    const size_t shmem = apply_lds_bytes(2 * Shape::kTile, pt.max_tab, Shape::merge_bytes(kSplit));
    if (shmem > kApplyLDSLimit) return fail(QR_ERR_SIZE, "apply: LDS stage too large");
    const uint32_t tpx = (ntiles % 8 == 0) ? ntiles / 8 : 0;
    auto kern = pt.cplx ? k_apply_staged<kMixed, kNarrow, true, kL, kSplit, kParts>
                        : k_apply_staged<kMixed, kNarrow, false, kL, kSplit, kParts>;
    if (shmem > kDefaultLDS)
        QR_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                         hipFuncAttributeMaxDynamicSharedMemorySize, int(shmem)));
    const uint64_t nblocks = uint64_t(ntiles) * nvec;
    if (nblocks > 0x7FFFFFFFull) return fail(QR_ERR_SIZE, "apply grid too large");
    hipLaunchKernelGGL(kern, dim3(unsigned(nblocks)), dim3(kApplyThreads * kSplit), shmem, s, N, ntiles, tpx,
                       pt.nchunk, pt.nrun, pt.grp, pt.chunk, pt.run, pt.part, pt.tab, pt.pat, pt.ptz, pt.ptc, d_x, d_y, partials);
    QR_HIP_CHECK(hipGetLastError());
    return QR_OK;
}

// Which form applies the operator (of the state's size, not of the number of
// states, so that every call finds the same tables).  F groups reach outside
// the tile, on D partner tiles, P of them past an L2 (as in choose_windows).
constexpr int kFormGather = 0;       // F gathers from memory
constexpr int kFormStaged = 1;       // D partner tiles through LDS
constexpr int kFormStagedDense = 2;  // the same with F >= 8 D
constexpr int kFormGatherFew = 3;    // gathers, two blocks per CU
constexpr int kFormStagedFew = 4;    // staged, two thread groups per block
constexpr int kFormGatherNear = 5;   // FP64, more than 8 groups, F = 0
// Measured (us, one state, gather / partner-staged):
//   FP64: reference's molecules (F/D 9..), 16 / 20 / 22 qubits 134 / 113,
//     1360 / 928, 7750 / 5050; k-local 24 qubits, 3000 terms (F/D 3.6) 7784 /
//     7436, 300 terms, two states (1.4) 4140 / 3340, 20 qubits 459 / 400;
//     random 20 qubits, 2000 terms (2.3) 1123 / 1104; below 2^20 rows, where x
//     stays in L2, gathers win up to F/D 8: 18 qubits, 100 terms 50 / 60,
//     k-local 16 qubits 28 / 33.  Operators with window passes keep only
//     partners that the L2 holds: 24-qubit ring 300 / 321.  So do those with 5 to 12
//     partners, many of them in L2, for half of the groups or more: random
//     bonds, y / y and energy, 24 qubits, 14, 12 groups 210 / 270 against 275 / 285,
//     200 / 259 against 256 / 277, 25 qubits, 12 415 / 496 against 482 / 502, k-local,
//     23 qubits, 12 114 / 162 against 134 / 179; but k-local, 24 qubits, 21 groups, 10
//     of them far, 337 / 397 against 332 / 379, 36 groups, 23 partners 611 / 660
//     against 594 / 659, 4 groups, 3 partners, two states 221 / 303 against 204 / 300.
//   complex64 (2^11-row tiles): molecule 20 qubits 804 / 883, random 20 qubits
//     762 / 840, k-local 24 qubits, 3000 terms 4940 / 5160, ring 24 qubits 183
//     / 199; a state past the 256 MB MALL: k-local 28 qubits 236 / 229 ms.
//   small complex64 tiles: gathers in all cases, within 5% at the worst.
// Where most partners lie past L2 (random operators), and hardly any group
// shares its partner, each group is a pass over x, and what counts is that the
// blocks find each other's partners in L2: masks ascend, so those of one step
// lie in a region as large as the tiles that the XCD works on, and neighbouring
// masks go to the same region.  Four blocks of 256 threads per CU make that 2 MB
// of the 4 MB L2, and once the blocks have drifted apart by a region every
// partner comes from the MALL or HBM; two make it 1 MB, which held in all cases.
// FP64, four states or one, gathers from four blocks per CU / staged / this, us:
// 24 qubits, 1000, 1500, 3000 terms 34400 / 34200 / 17100, 49300 / 48800 / 23200,
// 102800 / 96200 / 41300; 23 qubits, 300, 1000 4640 / 4650 / 3350, 14600 / 14900 /
// 6950, four states 68200 / 68900 / 27800; 22 qubits, 300 1790 / 1840 / 1170, four
// states 8890 / 9310 / 4710; 21 qubits (two blocks of 512 threads, as 20), 300
// 447 / 442 / 406, four states 3320 / 3260 / 1790; 25 qubits, 1000 59300 / 70500 /
// 46700.  With few partners the tile itself, which gathers load for groups
// inside it, counts: staged wins, 20 qubits, 8, 30 terms 24 / 17, 52 / 35; 21
// qubits, 100 terms 222 / 212 (but 20 qubits and 100 terms, two blocks, 71 / 82); one
// term, 19 qubits, four states 16 / 12.  Complex64 gains from the staged form,
// from 2^23 rows on with two thread groups per block (gathers / staged, one
// thread group / two): 22 qubits, 300 and 1000 terms 630 / 588 / 730, 2200 / 1800
// / 2250, four states 3750 / 2260 / 2780, 12100 / 6840 / 8750; 23 qubits, 300 terms
// 1970 / 1890 / 1475; 24 qubits, 300, 1000, 3000 terms 4680 / 4710 / 3220, 15300 /
// 8570 / 10200, 44100 / 23500 / 27300; 25 qubits, 1000 34500 / 34500 / 23100; but
// 21 qubits, 300 terms 236 / 287 (x in L2).
// The environment variable QR_APPLY_FORM (1 gather, 2 staged) overrides the
// choice, for tests and measurement.
static int apply_form(const qr_op *op, int kind, int L, const PatternShape &win_shape) {
    const char *e = getenv("QR_APPLY_FORM");
    if (e && atoi(e) == 1) return kFormGather;
    int form = op->form[kind].load(std::memory_order_relaxed) - 1;
    if (form < 0) {
        // gx ascends, so groups with equal bits above the tile are adjacent
        uint64_t far = 0, distinct = 0, past = 0, prev = 0;
        const int near = kind == 0 ? 17 : 18;
        for (uint64_t g = 0; g < op->G; ++g) {
            const uint64_t hi = op->gx[g] >> L;
            if (!hi) continue;
            ++far;
            if (distinct == 0 || hi != prev) {
                ++distinct;
                past += (op->gx[g] >> near) != 0;
            }
            prev = hi;
        }
        std::vector<ApplyWindow> wins;
        std::vector<uint8_t> pass;
        // (then the partners left are mostly in L2)
        const bool windows = win_shape.L && choose_windows(op, win_shape.L, wins, pass);
        const bool dense = far >= 8 * distinct;
        const bool scattered = 4 * past >= 3 * distinct, lone = scattered && 4 * far < 5 * distinct;
        const int state_log2 = int(op->nq) + (kind == 0 ? 4 : 3);
        bool staged = far > 0 && kind != 2 && !windows, few = false;
        if (kind == 0) {
            few = staged && lone && distinct >= 64 && state_log2 >= 24;
            const bool some = distinct >= 5 && distinct <= 12 && 2 * far >= op->G;
            staged = staged && !few &&
                     (dense || (state_log2 >= 26 && !some) || (state_log2 >= 24 && (scattered || 2 * far >= 3 * distinct)) ||
                      (far == op->G && 4 * far < 5 * distinct && distinct <= 16));
        } else {
            staged = staged && ((state_log2 >= 28 && 2 * far >= 3 * distinct) ||
                                (state_log2 >= 25 && scattered && distinct >= 64));
            few = staged && lone && distinct >= 64 && state_log2 >= 26;
        }
        form = few       ? (kind == 0 ? kFormGatherFew : kFormStagedFew)
               : staged  ? (dense ? kFormStagedDense : kFormStaged)
               : kind == 0 && far == 0 && op->G > 8 ? kFormGatherNear : kFormGather;
        op->form[kind].store(form + 1, std::memory_order_relaxed);
    }
    if (e && atoi(e) == 2) return form == kFormStagedDense || form == kFormStagedFew ? form : kFormStaged;
    return form;
}

// One memory pool per device for the per-launch <x|y> workspaces.  Its
// release threshold keeps freed blocks in the pool, so that after the first
// launch taking a buffer costs no device allocation.
static std::mutex g_pool_mu;
static hipMemPool_t g_pool[kMaxDevices];

static int partials_pool(hipMemPool_t *out) {
    int dev = 0;
    QR_HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(QR_ERR_ARG, "device index out of range");
    std::lock_guard<std::mutex> lock(g_pool_mu);
    if (!g_pool[dev]) {
        hipMemPoolProps props = {};
        props.allocType = hipMemAllocationTypePinned;
        props.location.type = hipMemLocationTypeDevice;
        props.location.id = dev;
        hipMemPool_t p;
        QR_HIP_CHECK(hipMemPoolCreate(&p, &props));
        uint64_t keep = ~uint64_t(0);
        QR_HIP_CHECK(hipMemPoolSetAttribute(p, hipMemPoolAttrReleaseThreshold, &keep));
        g_pool[dev] = p;
    }
    *out = g_pool[dev];
    return QR_OK;
}

// Workspace of the allocation-free entry point (qr_pauli_apply_noalloc): the
// <x|y> block partials, 2 doubles per (tile, vector), in a file-scope device
// array of 4 MiB that each device holds until the process ends.  Every call
// on one device shares it and it keeps the last call's contents; each block
// overwrites its own two slots, so nothing needs clearing.  In host code the
// array's name is no device address: its address on each device comes from
// hipGetSymbolAddress, taken once per device with that device current.
constexpr size_t kScratchDoubles = size_t(1) << 19;
static __device__ __align__(256) double scratch[kScratchDoubles];
static std::mutex g_scratch_mu;
static double *g_scratch[kMaxDevices];

static int scratch_partials(double **out) {
    int dev = 0;
    QR_HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(QR_ERR_ARG, "device index out of range");
    std::lock_guard<std::mutex> lock(g_scratch_mu);
    if (!g_scratch[dev]) {
        void *p = nullptr;
        QR_HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
        if (!p) return fail(QR_ERR_HIP, "hipGetSymbolAddress(scratch) returned no address");
        g_scratch[dev] = static_cast<double *>(p);
    }
    *out = g_scratch[dev];
    return QR_OK;
}

// Compute units of the current device (queried once per device).
static int apply_cus(int *out) {
    static std::mutex mu;
    static int cache[kMaxDevices];
    int dev = 0;
    QR_HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(QR_ERR_ARG, "device index out of range");
    std::lock_guard<std::mutex> lock(mu);
    if (!cache[dev]) {
        int cus = 0;
        QR_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        cache[dev] = cus > 0 ? cus : 1;
    }
    *out = cache[dev];
    return QR_OK;
}

// One way of applying an operator: tile size, form, and the pattern-table
// slot that holds its tables (2 * kind + staged; kind 0: FP64, 1: complex64,
// 2: small complex64 tiles).
struct ApplyPlan {
    int L = 0, tiles_log2 = 0, slot = 0, form = kFormGather;
    bool small = false, staged = false, single = false;  // single: one group
    PatternShape shape = {}, win_shape = {};
    int elem_log2 = 4;
};

template <bool kMixed, int kL>
static ApplyPlan make_plan(const qr_op *op, int kind) {
    using Shape = ApplyShape<kMixed, kL>;
    ApplyPlan p;
    p.L = int(op->nq) < kL ? int(op->nq) : kL;
    p.tiles_log2 = int(op->nq) - p.L;
    p.single = op->G == 1;
    p.elem_log2 = kMixed ? 3 : 4;
    if (!kMixed && p.L == kL)
        p.win_shape = {p.L, kApplyThreadBits, Shape::kPatSplit, Shape::kTabChunk,
                       uint32_t(Shape::kTile), false, false, {}};
    p.form = p.L == kL ? apply_form(op, kind, p.L, p.win_shape) : kFormGather;
    const bool staged = p.staged =
        p.form == kFormStaged || p.form == kFormStagedDense || p.form == kFormStagedFew;
    // the gather form on full complex64 tiles runs the paired-row layout
    const bool pairs = kMixed && !staged && p.L == kL;
    p.shape = {p.L, kApplyThreadBits, staged ? Shape::kPatSplitS : Shape::kPatSplit,
               staged ? Shape::kTabChunkS : Shape::kTabChunk,
               uint32_t(staged ? 2 * Shape::kTile : Shape::kTile), staged, pairs, {}};
    p.small = kind == 2;
    p.slot = 2 * kind + (staged ? 1 : 0);
    return p;
}

// Thread groups of 256 per block.  Several share a tile's groups (each takes
// every split-th), so that a launch of few tiles still fills the CUs' wave
// slots: the loop over the groups is a chain of scalar loads, table lookups
// and gathers, which only other waves hide.  Measured (us, split 1 / 2 / 4):
// FP64 molecules, 12 qubits 86 / 50 / 35, 16: 272 / 161 / 113, 18 (256 tiles):
// 613 / 371 / 235, 20 (1024 tiles, staged, F/D 9): 1007 / 928 / 989, 22: 6020
// / 5050 / 5570; k-local 20 qubits, 3000 terms (staged, F/D 5): 400 / 486 /
// 716 (one term, 19 qubits, four states 12 / 13 / 23); ring 24 qubits (gather)
// 320 / 300 / 358, a diagonal, 26 qubits 722 / 854; all groups inside the tile, y /
// y and energy, split 1 against 2: 24 qubits, 12, 24 groups 84 / 141 against 96 / 176,
// 130 / 187 against 144 / 229, 26 qubits, 16 414 / 522 against 470 / 665, but 24 qubits,
// 6 90 / 147 against 81 / 157, and below 2^22 rows equal; gathers with two blocks per
// CU, random, 300 terms, 21 qubits 491 / 406, 22 qubits 1170 / 1670.  Complex64,
// 2^11-row tiles: molecule 20 qubits (512 tiles) 1085 / 804, k-local 24 qubits
// (8192 tiles) 4940 / 5250; 2^10-row tiles: molecule 18 qubits (256 tiles) 439 /
// 256 / 183, random 18 qubits, 3 states (768 tiles) 47 / 36 / 41.
static int apply_split(const ApplyPlan &p, bool mixed, uint64_t blocks, int cus) {
    if (!mixed && p.form == kFormStaged) return 1;
    if (p.form == kFormGatherFew) return p.tiles_log2 <= 11 ? 2 : 1;
    if (p.form == kFormGatherNear && p.tiles_log2 >= 12) return 1;
    if ((!mixed || p.small) && blocks <= uint64_t(2) * cus) return 4;
    if (!mixed || p.form == kFormStagedFew) return p.single ? 1 : 2;
    return p.small || blocks < uint64_t(4) * cus ? 2 : 1;
}

int apply_tables(const qr_op *op, DeviceTables *t) {
    const ApplyPlan plan = make_plan<false, ApplyShape<false>::L>(op, 0);
    return device_patterns(op, t, plan.slot, plan.shape, plan.win_shape, false);
}

// FP64 applies of one state of few tiles and many groups, for a caller with
// memory for the sums: a tile's blocks take a share of the groups each and write
// what they add to y, which k_sum_parts sums.  In few blocks such an apply is a
// chain over the groups, 0.08-0.1 us each, which a batch of few operators ends up
// waiting for.  Measured, batches of one random operator (build and y, us), y from
// the entries in the tile builder's registers / whole applies / shares of 64 blocks
// in all: 12 qubits, 1000, 2000, 3500 terms 67, 85, 115 / 128, 222, 324 / 58, 89,
// 119; 13 qubits, 5000 323 / 686 / 308; 14 qubits, 500, 2000 114, 323 / 102, 418 /
// 69, 262; 15 qubits, 300, 2000 173, 676 / 94, 571 / 80, 463.  32, 64, 128 and 256
// blocks: 64 operators of 8 to 14 qubits 760, 746, 774, 789, 32 of 11 to 14 2650,
// 2605, 2680, 2930, but one of 15 qubits and 1000 terms 301, 245, 221, 207.
constexpr uint32_t kPartsBlocks = 64, kPartsGroups = 32;

uint32_t apply_parts(const qr_op *op) {
    constexpr int L = ApplyShape<false>::L;
    if (int(op->nq) < L || op->nq > 32) return 1;
    const uint64_t tiles = uint64_t(1) << (op->nq - L);
    uint32_t parts = 1;
    while (2 * parts * tiles <= kPartsBlocks && 2 * parts * kPartsGroups <= op->G) parts *= 2;
    return parts;
}

int launch_apply_parts(const qr_op *op, DeviceTables *t, uint32_t parts, const void *d_x, void *d_y, void *d_sums,
                       hipStream_t s) {
    constexpr int L = ApplyShape<false>::L;
    const ApplyPlan plan = make_plan<false, L>(op, 0);
    int rc = device_patterns(op, t, plan.slot, plan.shape, plan.win_shape, true);
    if (rc) return rc;
    const uint32_t n = 1u << op->nq, ntiles = n >> L;
    // (no window passes: the states are far below their least size)
    rc = plan.staged
             ? launch_staged<false, true, L, 4, true>(op, t, plan.slot, parts, d_x, d_sums, nullptr, ntiles, s)
             : launch_tiled<false, true, L, 4, false, true>(op, t, plan.slot, parts, d_x, d_sums, nullptr, ntiles, s);
    if (rc) return rc;
    hipLaunchKernelGGL(k_sum_parts, dim3((n + 255) / 256), dim3(256), 0, s, n, parts,
                       static_cast<const dvec2 *>(d_sums), static_cast<dvec2 *>(d_y));
    QR_HIP_CHECK(hipGetLastError());
    return QR_OK;
}

int launch_pauli_apply(const qr_op *op, DeviceTables *t, int32_t precision, uint32_t nvec,
                       const void *d_x, void *d_y, double *d_expect, hipStream_t s,
                       bool noalloc) {
    // QR_APPLY_WIDE=1 runs the 64-bit-mask instances on any operator, so that
    // the tests can check them without a state of more than 32 qubits
    const char *wide_env = getenv("QR_APPLY_WIDE");
    const bool force_wide = wide_env && atoi(wide_env) == 1;
    const bool mixed = precision == QR_PREC_MIXED, narrow = op->nq <= 32 && !force_wide;
    const uint64_t N = uint64_t(1) << op->nq;
    if (nvec == 0) return fail(QR_ERR_SIZE, "apply: nvec == 0");
    int rc, cus = 0;
    if ((rc = apply_cus(&cus))) return rc;
    ApplyPlan plan;
    if (!mixed) {
        plan = make_plan<false, ApplyShape<false>::L>(op, 0);
    } else {
        // small complex64 tiles when the default ones give fewer than two
        // blocks per CU; QR_APPLY_SMALL (0 never, 1 always where the state
        // has more rows than a small tile) overrides the choice, for tests
        // and measurement
        const bool can_small = int(op->nq) > kMixedSmallL;
        bool small = can_small && (N >> ApplyShape<true>::L) * nvec < uint64_t(2) * uint64_t(cus);
        const char *small_env = getenv("QR_APPLY_SMALL");
        if (small_env) small = can_small && atoi(small_env) == 1;
        plan = small ? make_plan<true, kMixedSmallL>(op, 2) : make_plan<true, ApplyShape<true>::L>(op, 1);
        // without allocation only uploaded tables can serve: those of the
        // other tile size when this one's are not on the device
        if (noalloc && can_small) {
            const ApplyPlan other = small ? make_plan<true, ApplyShape<true>::L>(op, 1)
                                          : make_plan<true, kMixedSmallL>(op, 2);
            if (!tables_ready(op, t, plan.slot, plan.L) && tables_ready(op, t, other.slot, other.L))
                plan = other;
        }
    }
    rc = device_patterns(op, t, plan.slot, plan.shape, plan.win_shape, noalloc);
    if (rc) return rc;
    const int L = plan.L;
    if ((N >> L) * uint64_t(nvec) > 0x7FFFFFFFull)
        return fail(QR_ERR_SIZE, "apply: state too large for one launch");
    const uint32_t ntiles = uint32_t(N >> L);
    // <x|y> block partials: a buffer of this launch's own, taken from the
    // device's pool and given back after the reduction, both in stream order,
    // so launches on one operator from several streams never share one
    double *partials = nullptr;
    if (d_expect && noalloc) {
        const uint64_t need = uint64_t(ntiles) * nvec * 2;
        if (need > kScratchDoubles)
            return fail(QR_ERR_SIZE, "apply_noalloc: <x|H|x> of " + std::to_string(nvec) +
                                         " vectors of " + std::to_string(ntiles) +
                                         " tiles needs " + std::to_string(need * 8) +
                                         " bytes of partials; the scratch array holds " +
                                         std::to_string(kScratchDoubles * 8));
        if ((rc = scratch_partials(&partials))) return rc;
    } else if (d_expect) {
        hipMemPool_t pool;
        if ((rc = partials_pool(&pool))) return rc;
        QR_HIP_CHECK(hipMallocFromPoolAsync(reinterpret_cast<void **>(&partials),
                                            size_t(ntiles) * nvec * 2 * sizeof(double), pool, s));
    }
    // QR_APPLY_SPLIT (1, 2, 4) overrides the number of thread groups, for
    // tests and measurement
    const char *split_env = getenv("QR_APPLY_SPLIT");
    const int split = split_env ? atoi(split_env) : apply_split(plan, mixed, uint64_t(ntiles) * nvec, cus);
    const uint32_t nwin = t->pat[plan.slot].nwin;
    auto launch = [&](auto mixed_t, auto l_t, auto split_t) {
        constexpr bool kMixed = decltype(mixed_t)::value;
        constexpr int kL = decltype(l_t)::value, kSplit = decltype(split_t)::value;
        // all states in one launch; with window passes up to 128 MB of them
        // at a time through all passes, so that the later ones find x and y in
        // the 256 MB MALL
        const uint64_t some = (uint64_t(1) << 27) / (N << plan.elem_log2);
        const uint32_t step = nwin ? uint32_t(some ? some : 1) : nvec;
        for (uint32_t v = 0; v < nvec; v += step) {
            const uint32_t nv = nvec - v < step ? nvec - v : step;
            const size_t off = size_t(v) * (N << plan.elem_log2);
            const void *x = static_cast<const unsigned char *>(d_x) + off;
            void *y = d_y ? static_cast<unsigned char *>(d_y) + off : nullptr;
            double *e = partials ? partials + 2 * uint64_t(ntiles) * v : nullptr;
            // (window passes may have taken every group: then the first of
            // them writes y)
            const bool rows_pass = t->pat[plan.slot].nchunk > 0, few = plan.form == kFormGatherFew;
            int r = QR_OK;
            if (rows_pass && plan.staged)
                r = narrow ? launch_staged<kMixed, true, kL, kSplit>(op, t, plan.slot, nv, x, y, e, ntiles, s)
                           : launch_staged<kMixed, false, kL, kSplit>(op, t, plan.slot, nv, x, y, e, ntiles, s);
            else if (rows_pass)
                r = narrow ? launch_tiled<kMixed, true, kL, kSplit>(op, t, plan.slot, nv, x, y, e, ntiles, s, few)
                           : launch_tiled<kMixed, false, kL, kSplit>(op, t, plan.slot, nv, x, y, e, ntiles, s, few);
            if constexpr (!kMixed)
                for (uint32_t k = 0; !r && k < nwin; ++k) {
                    const int sl = plan.slot + kApplySlots * int(k + 1);
                    const bool add = rows_pass || k > 0;
                    r = narrow ? launch_tiled<false, true, kL, 1, true>(op, t, sl, nv, x, y, e, ntiles, s, false, add)
                               : launch_tiled<false, false, kL, 1, true>(op, t, sl, nv, x, y, e, ntiles, s, false, add);
                }
            if (r) return r;
        }
        return int(QR_OK);
    };
    auto launch_split = [&](auto mixed_t, auto l_t) {
        // (2^11-row tiles: four thread groups would not fit the registers)
        constexpr int kMost = decltype(l_t)::value == kMixedSmallL ? 4 : 2;
        if (split >= 4 && kMost == 4) return launch(mixed_t, l_t, std::integral_constant<int, kMost>{});
        if (split >= 2) return launch(mixed_t, l_t, std::integral_constant<int, 2>{});
        return launch(mixed_t, l_t, std::integral_constant<int, 1>{});
    };
    using MixedL = std::integral_constant<int, ApplyShape<true>::L>;
    using SmallL = std::integral_constant<int, kMixedSmallL>;
    using Fp64L = std::integral_constant<int, ApplyShape<false>::L>;
    if (!mixed) rc = launch_split(std::false_type{}, Fp64L{});
    else if (plan.small) rc = launch_split(std::true_type{}, SmallL{});
    else rc = launch_split(std::true_type{}, MixedL{});
    if (!rc && d_expect) {
        hipLaunchKernelGGL(k_reduce_partials, dim3(nvec), dim3(256), 0, s, ntiles, partials,
                           d_expect);
        const hipError_t e = hipGetLastError();
        if (e != hipSuccess) rc = hip_fail(e, "k_reduce_partials");
    }
    if (partials && !noalloc) {
        const hipError_t e = hipFreeAsync(partials, s);
        if (!rc && e != hipSuccess) rc = hip_fail(e, "hipFreeAsync(partials)");
    }
    if (rc) return rc;
    return QR_OK;
}

}  // namespace qr
