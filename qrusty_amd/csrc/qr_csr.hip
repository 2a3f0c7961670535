// qr_csr.hip -- CSR build and CSR x vector kernels for gfx950 (CDNA4, wave64).
//
// CSR build (replaces accel::rowwise::make_row / make_unsafe_vectors_chunked,
// qrusty/src/accel.rs:171-210, 267-336).  The reference builds each row by
// emitting T (col, val) pairs, stable-sorting them by column and folding equal
// columns.  Here the work is split by *output entry*: one thread produces the
// entry of (row r, group j), where the groups are the distinct x masks sorted
// ascending and each group's terms are stored in input order.  Nothing is
// sorted on the device:
//   column   = r ^ x_j
//   position = r*G + rank_r(j), rank_r(j) = j + sum_{(b, s) in list_j, r_b=1} s
//              (the trie identity documented in qr_api.cpp: build_rank_lists)
//   value    = fold over the group's terms, in input order, of
//              (-1)^popcount(r & z_t) * c'_t  (first value, then +)
// which is exactly the reference's stable-sort-then-fold result, so indices
// and values are bit-identical.  The kernel is bound by HBM writes (24 B per
// nnz).  Rows are staged in LDS by the tile builder (qr_tile.h) and copied out
// coalesced; an operator with more than kWordMaxG groups (kSubMaxG past 32
// qubits) is built as sub-operators, subtrees of the mask trie that fill a
// contiguous segment of every row.
//
// CSR matvec (replaces accel::rowwise::spmat_dot_densevec, accel.rs:338-370):
// a power-of-two team of lanes per row streams the row's indices/values with
// non-temporal loads, gathers x, accumulates in FP64 with FMAs and reduces the
// team with cross-lane shuffles.
#include "qr_internal.h"
#include "qr_mv.h"
#include "qr_tile.h"

#include <algorithm>
#include <mutex>
#include <type_traits>

namespace qr {

// Tile of a block: each of the 8 XCDs (blocks go to them round-robin) builds
// one contiguous range of tiles, so that the lines at the ends of
// neighbouring rows, which two blocks write parts of, meet in one L2, and an
// XCD touches an eighth of the output's pages.  Launch order / this one (ms,
// two output buffers each; their place moves the rate by up to 20%): 20 qubits
// and 2000 random terms 10.5, 8.6 / 7.9, 7.4; 300 terms 1.34, 1.11 / 1.25,
// 1.08; 24-qubit ring 1.79, 1.52 / 1.76, 1.46; 20-qubit molecule 13.3, 11.8 /
// 11.0, 10.2.  Windows of 8 times 8 to 512 tiles lie between.  Grids that are
// no multiple of 8 (row ranges) have it too: 17 qubits, 100004 rows, 1100, 1300,
// 1900 terms in launch order / this 616, 708, 977 / 464, 560, 816 us.
__device__ __forceinline__ uint32_t xcd_tile() {
    const uint32_t x = blockIdx.x % 8u, n = gridDim.x;  // n % 8 ranges are one longer
    return x * (n / 8u) + min(x, n % 8u) + blockIdx.x / 8u;
}

// LDS-staged build: one block per tile of the shared tile builder
// (qr_tile.h), without the fused matvec; the heavy-group instances of
// fold_tiles run 2^op.fold_log2 consecutive tiles per block, folding the
// heavy groups once for all of them.
template <int kChunks, int kMode>
__global__ __launch_bounds__(kStageThreads) void k_csr_build_staged(TileOp op) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    if constexpr (fold_tiles<kChunks, kMode>()) {
        const uint32_t tile_log2 = 10u - op.jw_log2 + 4u;
        const uint32_t k = 1u << op.fold_log2;
        for (uint32_t s = 0; s < k; ++s) {
            const uint64_t tile = uint64_t(xcd_tile()) * k + s;
            if ((((op.row_begin >> tile_log2) + tile) << tile_log2) >= op.row_end) break;
            build_tile_staged<false, kChunks, false, kMode>(op, tile, smem_raw, s);
        }
    } else {
        build_tile_staged<false, kChunks, false, kMode>(op, xcd_tile(), smem_raw);
    }
}

// The sign-word builder (operators of at most 32 qubits): one group per thread
// and few vector instructions per term and row.  Thread layout as in qr_tile.h
// (kT = RS rows x JW lanes, the rows of a tile in M = 2^m_log2 batches of RS),
// but
//  * kReal, for operators whose coefficients c' are all real and whose groups
//    have few terms past kWordHold (molecular and spin Hamiltonians): a lane
//    holds its group's terms.  The sign of a term over the tile's M rows is one
//    32-bit word, the parity of r & z for batch m in bit 31 - m (the parity is
//    linear in r: the fixed bits give all or none, each of the five batch bits
//    an alternating pattern), shifted up once per batch; its top bit goes
//    straight into the coefficient's sign bit: a shift, a bit-field insert and
//    an addition per term, against mask, count, compare, selects and two
//    additions.  (The imaginary part of a real coefficient is a signed zero,
//    and a sum of signed zeros is -0 only if all are: one word per group, the
//    AND of its terms'.)  Terms past those held come from memory;
//  * otherwise every term is loaded once per four batches, whose rows differ
//    in two bits and so in two sign flips, and added to four sums;
//  * absent terms are -0.0, which every sum absorbs unchanged, so all lanes
//    run the same additions;
//  * a lane's first slot comes from a table by row bit (word_rank), all its
//    loads at once, where a walk along its rank list is a chain of them that a
//    tile of 32 rows did not hide (20-qubit molecule 11.5 -> 10.2 ms, 16 qubits
//    and 24069 groups 7.3 -> 5.9);
//  * a row's slot moves by one addition per batch (what the bits that the step
//    flips add, qr_tile.h);
//  * 64 VGPRs: two 1024-thread blocks per CU, one copying out while the other
//    computes, and two stages per block, one barrier per batch;
//  * M is chosen so that small operators still fill the chip.
// Groups of many terms are folded by a pass of their own at the start of the
// tile, one thread per (group, row), their terms in LDS.  The additions are
// the same, in the same order, as build_tile_staged's, so the values are
// bit-identical.  Operators of more than kWordMaxG groups are built as
// sub-operators of at most that many (kSub), consecutive blocks building the same
// rows (launch_build_words).
// What bounds it: the stores (5.2 or 6.5 TB/s of 24 B per entry, by the place
// of the output in memory; fills reach 6.65), and from about five terms per
// group on the additions and the loads of the terms.  The two-group-chunk
// builder that it replaced / this one, us: molecules of 12 / 16 / 18 / 20
// qubits 139 / 510 / 4030 / 28100 -> 20 / 290 / 1820-2430 / 10200-12500; rings
// of 14 / 24 qubits 24.5 / 2160 -> 7.6 / 1480-1780; one-term groups, 12 qubits
// (195 groups) 29 -> 7.9, 20 qubits (1999) 9000-9400 -> 7400-8900, 18 qubits
// (4948) 7000 -> 4500-5600, 16 qubits (24069) 10010 -> 6200; terms of weight 1
// to 4, 16 qubits (332 groups of 3.0 terms) 196 -> 104, 20 qubits (610 of 3.3)
// 6350 -> 2900, 18 qubits (1208 of 6.6) 8790 -> 2580.  Holding four complex
// terms per lane instead of loading them for every four batches: 600 groups of
// 4 terms 688 against 775, but of 8 3620 against 1060, and a wave waits for
// its longest group.
constexpr int kWordMaxLog2 = 5;   // batches per tile (log2)
constexpr uint32_t kWordLDS = 80 * 1024;  // of one block: two per CU

// Sign words of the batch bits: bit b of m set <=> the bits of kSignWord[b]
__device__ __forceinline__ uint32_t sign_word(uint32_t parity, uint32_t zm) {
    uint32_t w = 0u - (parity & 1u);
    w ^= (zm & 1u) ? 0x55555555u : 0u;
    w ^= (zm & 2u) ? 0x33333333u : 0u;
    w ^= (zm & 4u) ? 0x0F0F0F0Fu : 0u;
    w ^= (zm & 8u) ? 0x00FF00FFu : 0u;
    w ^= (zm & 16u) ? 0x0000FFFFu : 0u;
    return w;
}

// |c| with the sign in bit 31 of w
__device__ __forceinline__ double with_sign(double c, uint32_t w) {
    return __hiloint2double(int((uint32_t(__double2hiint(c)) & 0x7fffffffu) | (w & 0x80000000u)), __double2loint(c));
}
__device__ __forceinline__ uint32_t sign_of(double c) { return uint32_t(__double2hiint(c)) & 0x80000000u; }

__device__ __forceinline__ double flip(double c, uint32_t sign) {
    return __hiloint2double(__double2hiint(c) ^ int(sign), __double2loint(c));
}

// A heavy group's term in LDS, a broadcast read or two for a wave: the real
// form's 16 bytes (re, z and the sign of im), the other's double2 and z apart.
struct RealTerm {
    double re;
    uint32_t z, im;
};
template <bool kReal>
struct HeavyTerms {
    unsigned char *at;
    uint32_t most;  // terms that fit
    __device__ HeavyTerms(unsigned char *a, uint32_t bytes) : at(a), most(bytes / (kReal ? 16u : 20u)) {}
    __device__ uint32_t *z() const { return reinterpret_cast<uint32_t *>(at + 16u * most); }
    __device__ void put(uint32_t i, const WordTerm &t) const {
        if constexpr (kReal) {
            reinterpret_cast<RealTerm *>(at)[i] = RealTerm{t.re, t.z, sign_of(t.im)};
        } else {
            reinterpret_cast<double2 *>(at)[i] = make_double2(t.re, t.im);
            z()[i] = t.z;
        }
    }
    __device__ WordTerm get(uint32_t i) const {
        if constexpr (kReal) {
            const RealTerm t = reinterpret_cast<const RealTerm *>(at)[i];
            return WordTerm{t.re, __hiloint2double(int(t.im), 0), t.z, 0};
        } else {
            const double2 c = reinterpret_cast<const double2 *>(at)[i];
            return WordTerm{c.x, c.y, z()[i], 0};
        }
    }
};

// v plus, in term order, the terms [t, t1) in row r, four loaded ahead of
// their additions.
template <bool kReal>
__device__ __forceinline__ double2 fold_words(double2 v, const HeavyTerms<kReal> &terms, uint32_t t, uint32_t t1,
                                              uint32_t r) {
    uint32_t im = sign_of(v.y);
    auto add = [&](const WordTerm &e) {
        const uint32_t s = uint32_t(__popc(r & e.z)) << 31;
        v.x = v.x + flip(e.re, s);
        if (kReal) im &= sign_of(e.im) ^ s;
        else v.y = v.y + flip(e.im, s);
    };
    constexpr uint32_t kF = 4;
    for (; t + kF <= t1; t += kF) {
        WordTerm e[kF];
#pragma unroll
        for (uint32_t u = 0; u < kF; ++u) e[u] = terms.get(t + u);
#pragma unroll
        for (uint32_t u = 0; u < kF; ++u) add(e[u]);
    }
    for (; t < t1; ++t) add(terms.get(t));
    if (kReal) v.y = __hiloint2double(int(im), 0);
    return v;
}

// What the builder runs on: the operator's tables, the sub-operators of this
// launch (one: the whole operator, if !kSub), and its outputs (indptr null:
// not this launch).
struct WordOp {
    const WordLeaf *leaves;
    const WordGroup *groups;
    const int32_t *rank;
    const uint64_t *tz, *ttz;  // terms, and the tail table (qr_op::ttz, ttc)
    const double2 *tc, *ttc;
    const uint32_t *ptr;       // heavy groups' terms
    const WordTerm *terms;
    uint64_t *indptr, *indices;
    double2 *data;
    uint64_t row_begin, row_end;
    uint32_t G, nq, nleaves, ntail, jw_log2, m_log2;
};

// LDS of a block: two stages, whose place the heavy groups' terms take first
// (in turns of that size), and those groups' values, as many as leave two blocks
// to a CU (all of them: the launch takes fewer batches per tile until they fit).
struct WordLds {
    uint32_t nheavy, hv_at, total;
    __host__ __device__ WordLds(uint32_t g, uint32_t rs_log2, uint32_t tile_log2, uint32_t hcnt, const uint32_t *ptr) {
        const uint32_t stage = (((g << rs_log2) + 1u) & ~1u) * 48u, each = 16u << tile_log2;
        const uint32_t fit = (kWordLDS - stage) / each;
        nheavy = hcnt < fit ? hcnt : fit;
        hv_at = stage;
        if (nheavy) {
            const uint32_t room = kWordLDS - nheavy * each, n = ptr[nheavy] - ptr[0];
            const uint32_t want = n < room / 20u ? (20u * n + 15u) & ~15u : room;
            if (want > hv_at) hv_at = want;
        }
        total = hv_at + nheavy * each;
    }
};

template <bool kReal, bool kSub, int kT>
__global__ __launch_bounds__(kT, 8) void k_csr_build_words(WordOp op) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    const uint32_t block = xcd_tile(), tile = kSub ? block / op.nleaves : block;
    const WordLeaf &lf = op.leaves[kSub ? block - tile * op.nleaves : 0u];
    const uint32_t G = lf.g, s0 = lf.s0, hcnt = lf.hcnt, at = lf.at, jw_log2 = op.jw_log2;
    const uint32_t rs_log2 = kSub ? 0u : uint32_t(__builtin_ctz(kT)) - jw_log2;
    const uint32_t m_log2 = op.m_log2, tile_log2 = rs_log2 + m_log2, M = 1u << m_log2;
    const uint32_t tid = threadIdx.x;
    const uint32_t lane = kSub ? tid : tid & ((1u << jw_log2) - 1u);
    const uint32_t ro = kSub ? 0u : tid >> jw_log2;
    const uint64_t row_begin = op.row_begin, row_end = op.row_end;
    const uint64_t tile_base = ((row_begin >> tile_log2) + tile) << tile_log2;
    const uint32_t rfix = uint32_t(tile_base) | ro;  // at most 32 bits of row
    const uint32_t batch_pad = ((G << rs_log2) + 1u) & ~1u;
    const uint32_t stage_b = batch_pad * 24u;
    const WordLds lds(G, rs_log2, tile_log2, hcnt, op.ptr + at);
    const uint32_t nheavy = lds.nheavy;
    double2 *hv = reinterpret_cast<double2 *>(smem_raw + lds.hv_at);

    if (op.indptr && (!kSub || block == tile * op.nleaves)) {
        const uint64_t r0 = max(row_begin, tile_base), r1 = min(row_end, tile_base + (1ull << tile_log2));
        const uint64_t g = op.G;
        for (uint64_t r = r0 + tid; r < r1 + (r1 == row_end); r += kT) op.indptr[r - row_begin] = r * g;
    }

    // heavy groups first, before the lanes' own terms take registers: their
    // terms into LDS, then one thread per (group, row)
    if (nheavy) {
        const auto hptr = as_global(op.ptr) + at;
        const HeavyTerms<kReal> terms(smem_raw, lds.hv_at);
        const uint32_t h0 = hptr[0], nt = hptr[nheavy] - h0;
        for (uint32_t i = tid; i < nheavy << tile_log2; i += kT) hv[i] = make_double2(-0.0, -0.0);
        for (uint32_t t0 = 0; t0 < nt; t0 += terms.most) {
            const uint32_t t1 = min(t0 + terms.most, nt);
            if (t0) __syncthreads();  // the terms before
            for (uint32_t i = tid; i < t1 - t0; i += kT) terms.put(i, op.terms[h0 + t0 + i]);
            __syncthreads();
            for (uint32_t i = tid; i < nheavy << tile_log2; i += kT) {
                const uint32_t g = i >> tile_log2, r = uint32_t(tile_base) + (i & ((1u << tile_log2) - 1u));
                const uint32_t a = max(hptr[g] - h0, t0), e = min(hptr[g + 1] - h0, t1);
                if (a < e) hv[i] = fold_words<kReal>(hv[i], terms, a - t0, e - t0, r);
            }
        }
        // (the barrier after the lanes' setup, which overlaps the long groups)
    }

    // place of the lane's group in row rfix, and its change when the batch
    // index goes from m to m + 1 with t = ctz(m + 1): what bit t adds minus
    // what the bits below, which turn off, did
    int32_t slot = int32_t(ro * G + lane);
    int32_t step[kWordMaxLog2] = {0, 0, 0, 0, 0};
    // the same of the sub-operator's first entry
    int32_t off = int32_t(s0), ostep[kWordMaxLog2] = {0, 0, 0, 0, 0};
    if (kSub) {
        int32_t below = 0;
#pragma unroll
        for (uint32_t b = 0; b < 32; ++b) {
            const int32_t v = lf.off[b];
            if (b >= m_log2) off += (rfix >> b) & 1u ? v : 0;
            if (b < uint32_t(kWordMaxLog2)) ostep[b] = v - below;
            below += v;
        }
    }
    const bool valid = lane < G;
    int32_t hs = -1;
    uint32_t xj = 0, n = 0, tf = 0, wi = 0xffffffffu;
    uint32_t w[kWordHold];
    double c[kWordHold];
#pragma unroll
    for (int u = 0; u < int(kWordHold); ++u) {
        w[u] = 0xffffffffu;  // -0.0
        c[u] = 0.0;
    }
    const auto gtz = as_global(op.tz), gttz = as_global(op.ttz);
    const auto gtc = as_global(reinterpret_cast<const dvec2 *>(op.tc));
    const auto gttc = as_global(reinterpret_cast<const dvec2 *>(op.ttc));
    // term u of the lane's group: those past the second from the tail table
    // (coalesced) as far as it goes
    auto load = [&](uint32_t u) {
        const bool tail = u >= 2 && u - 2 < op.ntail;
        const uint32_t i = tail ? (u - 2) * op.G + s0 + lane : tf + u;
        const double2 cc = ld2((tail ? gttc : gtc) + i);
        return WordTerm{cc.x, cc.y, uint32_t(tail ? gttz[i] : gtz[i]), 0};
    };
    if (valid) {
        const auto rank = as_global(op.rank) + s0 + lane;
        int32_t below = 0;
#pragma unroll
        for (uint32_t k = 0; k < uint32_t(kWordMaxLog2); ++k) {
            const uint32_t b = rs_log2 + k;
            const int32_t v = k < m_log2 && b < op.nq ? rank[uint64_t(b) * op.G] : 0;
            step[k] = v - below;
            below += v;
        }
        for (uint32_t b = 0; b < rs_log2 && b < op.nq; ++b) slot += (ro >> b) & 1u ? rank[uint64_t(b) * op.G] : 0;
        for (uint32_t b = tile_log2; b < op.nq; ++b)
            if ((uint32_t(tile_base) >> b) & 1u) slot += rank[uint64_t(b) * op.G];
        const WordGroup gr = op.groups[s0 + lane];
        xj = gr.x;
        tf = gr.tf;
        hs = gr.heavy < int32_t(nheavy) ? gr.heavy : -1;
        if (hs < 0) {
            n = gr.n;
            if constexpr (kReal) {
#pragma unroll
                for (int u = 0; u < int(kWordHold); ++u) {
                    if (uint32_t(u) >= n) break;
                    const WordTerm t = load(uint32_t(u));
                    const uint32_t s = sign_word(__popc(rfix & t.z), (t.z >> rs_log2) & (M - 1u));
                    w[u] = s ^ (sign_of(t.re) ? 0xffffffffu : 0u);
                    wi &= s ^ (sign_of(t.im) ? 0xffffffffu : 0u);
                    c[u] = t.re;
                }
            }
        }
    }
    if (nheavy) __syncthreads();
    // the wave's longest group, in registers and past them
    const bool more2 = __any(n > 2), more4 = __any(n > 4), past = __any(n > kWordHold);

    // the batch's entries, in LDS: written at the lane's slot, copied out by
    // consecutive threads (a batch has at most kT of them)
    const uint32_t stage_entries = G << rs_log2;
    const bool whole = tile_base >= row_begin && tile_base + (uint64_t(M) << rs_log2) <= row_end;
    // output place of the batch's first row (before row_begin: not used)
    uint64_t dst = (tile_base - row_begin) * op.G;
    if (kSub) dst += uint64_t(int64_t(off));
    const uint64_t dst_step = uint64_t(op.G) << rs_log2;
    const auto indices = as_global(op.indices);
    const auto data = as_global(reinterpret_cast<dvec2 *>(op.data));
    auto batch = [&](uint32_t m, uint32_t buf, double2 e) {
        uint64_t *si = reinterpret_cast<uint64_t *>(smem_raw + buf * stage_b);
        double2 *sd = reinterpret_cast<double2 *>(si + batch_pad);
        const uint32_t r = rfix + (m << rs_log2);
        if (valid && (whole || (uint64_t(r) >= row_begin && uint64_t(r) < row_end))) {
            if constexpr (kReal) {
                // term-order fold: first value, then + (accel.rs:191-208)
                e.x = with_sign(c[0], w[0]);
                e.x = e.x + with_sign(c[1], w[1]);
                if (more2) {
                    e.x = e.x + with_sign(c[2], w[2]);
                    e.x = e.x + with_sign(c[3], w[3]);
                }
                if (more4) {
                    e.x = e.x + with_sign(c[4], w[4]);
                    e.x = e.x + with_sign(c[5], w[5]);
                }
                uint32_t im = wi;
                if (past) {
                    for (uint32_t u = kWordHold; u < n; ++u) {
                        const WordTerm t = load(u);
                        const uint32_t sg = uint32_t(__popc(r & t.z)) << 31;
                        e.x = e.x + flip(t.re, sg);
                        im &= sign_of(t.im) ^ sg;
                    }
                }
                e.y = __hiloint2double(int(im & 0x80000000u), 0);
            }
            if (hs >= 0) e = hv[(uint32_t(hs) << tile_log2) | (m << rs_log2) | ro];
            si[slot] = r ^ xj;
            sd[slot] = e;
        }
#pragma unroll
        for (int u = 0; u < int(kWordHold); ++u) w[u] <<= 1;
        wi <<= 1;
        __syncthreads();
        bool mine = tid < stage_entries;
        if (!whole) {
            const uint64_t b0 = tile_base + (uint64_t(m) << rs_log2);
            const uint64_t row = b0 + (kSub ? 0u : tid / G);
            mine = mine && row >= row_begin && row < row_end;
        }
        if (mine) {
            indices[dst + tid] = si[tid];
            const double2 dv = sd[tid];
            data[dst + tid] = dvec2{dv.x, dv.y};
        }
    };
    auto advance = [&](int t) {
        slot += step[t];
        dst += dst_step;
        if (kSub) dst += uint64_t(int64_t(ostep[t]));
    };
    // !kReal: the lane's group in the rows of four batches, each term loaded
    // once for the four and two in flight (-0.0, the absent term, first: every
    // sum absorbs it unchanged)
    double2 e4[4] = {};
    auto fold4 = [&](uint32_t m) {
#pragma unroll
        for (int k = 0; k < 4; ++k) e4[k] = make_double2(-0.0, -0.0);
        const uint32_t r = rfix + (m << rs_log2);
        auto add = [&](const WordTerm &t) {
            const uint32_t s0 = uint32_t(__popc(r & t.z)) << 31;
            const uint32_t za = (t.z >> rs_log2) << 31, zb = (t.z >> (rs_log2 + 1u)) << 31;
            const uint32_t sg[4] = {s0, s0 ^ za, s0 ^ zb, s0 ^ za ^ zb};
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                e4[k].x = e4[k].x + flip(t.re, sg[k]);
                e4[k].y = e4[k].y + flip(t.im, sg[k]);
            }
        };
        for (uint32_t u = 0; u < n; u += 2) {
            WordTerm t0 = load(u), t1{-0.0, -0.0, 0, 0};
            if (u + 1 < n) t1 = load(u + 1);
            add(t0);
            add(t1);
        }
    };
#pragma unroll 1
    for (uint32_t m = 0; m < M; m += 4) {  // M is at least 4
        if constexpr (!kReal) fold4(m);
        batch(m, 0, e4[0]);
        advance(0);
        batch(m + 1, 1, e4[1]);
        advance(1);
        batch(m + 2, 0, e4[2]);
        advance(0);
        batch(m + 3, 1, e4[3]);
        const uint32_t t = uint32_t(__builtin_ctz(m + 4u));  // 2 to 5 (the end)
        if (t == 2) advance(2);
        else if (t == 3) advance(3);
        else advance(4);
    }
}

__global__ __launch_bounds__(256) void k_indptr(uint64_t row_begin, uint64_t nrows, uint64_t G,
                                                uint64_t *__restrict__ indptr) {
    uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x;
    if (i <= nrows) indptr[i] = (row_begin + i) * G;
}

// Builds by k_csr_build_words: the whole operator, or its sub-operators, in one
// launch with the threads that the largest needs, or in one for each number of
// threads.  One launch writes every row from end to end, while its lines are in L2;
// several write it in pieces, whose ends leave the caches in between.  But it idles
// the threads that small sub-operators don't need, which counts where the lanes load
// their terms again; so one (word_joint) for the real form and up to 4 terms per
// group, where it takes at most twice the threads.  Several / one, us: molecules of
// 18, 20, 22 qubits (4 to 6 GB) 1249 / 1085, 928 / 822, 1330 / 1197; random, 17
// qubits, 1025 groups (488 + 537) 837 / 592 (638 by the builder before this one), 18
// qubits, 2086 736 / 589; 880 + 220 groups of 1, 3 (complex), 6 terms 798 / 662, 795
// / 730, 812 / 693; 200 + 150, 900, 210 of 4 complex terms 1173 / 954; but 900 + 300
// of 8 1063 / 1260, 1000 + 60 of 6 853 / 1055; 1000, 60, 120, 240 of 1 (2.3 times the
// threads) 985 / 1079.
static int launch_build_words(const qr_op *op, const DeviceTables *t, uint64_t row_begin, uint64_t row_end,
                              uint64_t *d_indptr, uint64_t *d_indices, double *d_data, hipStream_t s) {
    const uint32_t G = uint32_t(op->G);
    auto run = [&](auto sub_t, auto threads_t, uint32_t jw, size_t first, size_t last) {
        constexpr bool kSub = decltype(sub_t)::value;
        constexpr int kT = decltype(threads_t)::value;
        const uint32_t nl = uint32_t(last - first), rs_log2 = kSub ? 0u : uint32_t(__builtin_ctz(kT)) - jw;
        // batches per tile: as many as the sign words of the real form have, and
        // as many where the tile folds heavy groups; half of that for the rest,
        // which loads its terms again anyway (20 qubits, 2000 terms 7.5 / 7.4
        // ms; weights 1 to 4, 2000 terms 2.9 / 3.5), and for one or two groups, whose
        // tiles are the longest (24 and 25 qubits 187 / 166, 211 / 186 us); fewer where
        // the launch would have under four blocks per CU
        uint32_t ml = (op->word_real && G > 2) || t->nheavy ? kWordMaxLog2 : kWordMaxLog2 - 1;
        while (ml > 2 && nl * ((row_end - row_begin) >> (rs_log2 + ml)) < 1024) --ml;
        // and as few as the LDS holds all heavy groups' values for (by 8 batches
        // it does: a heavy group has 4 times the mean of terms, so they are at
        // most a quarter of the operator's, and kMaxHeavy).  The lanes of a group
        // that does not fit load its terms for every row: 32 batches whether they
        // fit or not / this, us: 24 qubits, 8 groups, one of 64, 300 terms 4230 /
        // 644, 20900 / 1270, with complex coefficients 8270 / 1270; 23 qubits, 12
        // groups, two of 200 13800 / 935; 21 qubits, 64 groups, 15 of 100 11060 /
        // 1045; 20 qubits, 200 groups, 40 of 100 7640 / 1490.
        auto all_fit = [&]() {
            for (size_t k = first; k < last; ++k) {
                const WordLeaf &lf = op->word_leaves[k];
                if (WordLds(lf.g, rs_log2, rs_log2 + ml, lf.hcnt, op->word_ptr.data() + lf.at).nheavy < lf.hcnt)
                    return false;
            }
            return true;
        };
        while (ml > 2 && !all_fit()) --ml;
        const uint32_t tl = rs_log2 + ml;
        const uint64_t nt = nl * (((row_end - 1) >> tl) - (row_begin >> tl) + 1);
        if (nt > 0x7FFFFFFFull) return fail(QR_ERR_SIZE, "CSR build grid too large");
        uint32_t shmem = 0;
        for (size_t k = first; k < last; ++k) {
            const WordLeaf &lf = op->word_leaves[k];
            shmem = std::max(shmem, WordLds(lf.g, rs_log2, tl, lf.hcnt, op->word_ptr.data() + lf.at).total);
        }
        const WordOp args{t->word_leaves + first, t->word_groups, t->word_rank, t->tz, t->ttz, t->tc, t->ttc,
                          t->word_ptr, t->word_terms, d_indptr, d_indices, reinterpret_cast<double2 *>(d_data),
                          row_begin, row_end, G, uint32_t(op->nq), nl, t->ntail, jw, ml};
        d_indptr = nullptr;  // by the first launch
        auto kern = op->word_real ? k_csr_build_words<true, kSub, kT> : k_csr_build_words<false, kSub, kT>;
        if (shmem > 64 * 1024)
            QR_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, int(shmem)));
        hipLaunchKernelGGL(kern, dim3(unsigned(nt)), dim3(kT), shmem, s, args);
        QR_HIP_CHECK(hipGetLastError());
        return int(QR_OK);
    };
    using T = std::true_type;
    using F = std::false_type;
    using T256 = std::integral_constant<int, 256>;
    using T512 = std::integral_constant<int, 512>;
    using T1024 = std::integral_constant<int, 1024>;
    const auto &lv = op->word_leaves;
    if (lv.size() == 1) return run(F{}, T1024{}, stage_jw_log2(G), 0, 1);
    auto to = [&](uint32_t most) {
        size_t k = 0;
        while (k < lv.size() && lv[k].g <= most) ++k;
        return k;
    };
    size_t a = to(256), b = to(512);
    const size_t c = lv.size();
    if (op->word_joint) {
        uint32_t most = 0;
        for (const auto &l : lv) most = std::max(most, l.g);
        a = most <= 256 ? c : 0;
        b = most <= 512 ? c : 0;
    }
    int rc = QR_OK;
    if (a && (rc = run(T{}, T256{}, 0, 0, a))) return rc;
    if (b > a && (rc = run(T{}, T512{}, 0, a, b))) return rc;
    if (c > b) rc = run(T{}, T1024{}, 0, b, c);
    return rc;
}

int launch_csr_indptr(const qr_op *op, uint64_t row_begin, uint64_t nrows, uint64_t *d_indptr, hipStream_t s) {
    const uint64_t nb = (nrows + 1 + 255) / 256;
    hipLaunchKernelGGL(k_indptr, dim3(unsigned(nb)), dim3(256), 0, s, row_begin, nrows, op->G, d_indptr);
    QR_HIP_CHECK(hipGetLastError());
    return QR_OK;
}

int launch_csr_build(const qr_op *op, DeviceTables *t, uint64_t row_begin, uint64_t row_end,
                     uint64_t *d_indptr, uint64_t *d_indices, double *d_data, hipStream_t s) {
    const uint64_t nrows = row_end - row_begin;
    if (op->G > 0x7FFFFFFFull) return fail(QR_ERR_SIZE, "too many groups");
    const uint32_t G = uint32_t(op->G);
    int rc;
    bool words = false;
    if (nrows && (rc = word_tables(op, t, s, &words))) return rc;
    if (words) return launch_build_words(op, t, row_begin, row_end, d_indptr, d_indices, d_data, s);
    // wider masks, and captures that come before any build of the operator: the
    // shared tile builder
    if (d_indptr && (rc = launch_csr_indptr(op, row_begin, nrows, d_indptr, s))) return rc;
    if (nrows == 0) return QR_OK;
    if (!op->leaves.empty()) {
        // one sub-operator per subtree of the mask trie, each <= kSubMaxG
        // groups with one row per batch (JW = 1024): the fast 1- and 2-chunk
        // kernels, each writing its contiguous segment of every row
        const uint32_t jw = 10, tl2 = 4;
        const uint64_t nt = ((row_end - 1) >> tl2) - (row_begin >> tl2) + 1;
        if (nt > 0x7FFFFFFFull) return fail(QR_ERR_SIZE, "CSR build grid too large");
        for (size_t k = 0; k < op->leaves.size(); ++k) {
            const auto &lf = op->leaves[k];
            const uint32_t g = lf.s1 - lf.s0, nch = (g + 1023) >> 10;
            uint32_t dbuf = 0;
            const uint32_t nh = heavy_fit(lf.hcnt, jw);
            // (sub-operators keep one stage: the second would cost them tiles
            // per heavy fold; 20-qubit molecule, when it was built here, 14.12
            // -> 14.38 ms)
            const size_t sb = stage_bytes(g, jw, &dbuf);
            const uint32_t fl = fold_tiles_log2(true, sb, heavy_bytes(nh, jw), nt);
            const size_t shmem = sb + (heavy_bytes(nh, jw) << fl);
            TileOp top{t->gx + lf.s0, t->gterm + lf.s0, t->tz, t->tc, t->rl_ptr + lf.s0, t->rl,
                       d_indices, reinterpret_cast<double2 *>(d_data), nullptr, nullptr, nullptr,
                       row_begin, row_end, g, jw, nch, dbuf,
                       nh ? t->leaf_heavy + lf.hoff : nullptr, nh, lf.s0, lf.depth, G,
                       t->ntail ? t->ttz + lf.s0 : nullptr, t->ntail ? t->ttc + lf.s0 : nullptr, t->ntail, fl};
            auto kst = nh ? (nch <= 1 ? k_csr_build_staged<1, kTileSubHeavy> : k_csr_build_staged<2, kTileSubHeavy>)
                          : (nch <= 1 ? k_csr_build_staged<1, kTileSub> : k_csr_build_staged<2, kTileSub>);
            QR_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kst),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, int(shmem)));
            hipLaunchKernelGGL(kst, dim3(unsigned(((nt - 1) >> fl) + 1)), dim3(kStageThreads), shmem, s, top);
            QR_HIP_CHECK(hipGetLastError());
        }
        return QR_OK;
    }
    // G <= kSubMaxG: one or two group chunks per thread.  Operators of 129 to
    // 1024 groups run two chunks on half the lanes per row (twice the rows per
    // batch): measured 6-14% faster at G = 150, 417, 690, 880 and 990; one
    // chunk stays faster at G = 25 and 60, and four chunks on 512 lanes were
    // 22% slower than two on 1024 at G = 1996 (one block per CU instead of two).
    uint32_t jw = stage_jw_log2(G);
    if (jw == 8 || jw == 9 || (jw == 10 && G <= 1024)) jw -= 1;
    const uint32_t nch = (G + (1u << jw) - 1) >> jw;
    const uint32_t tl2 = 10 - jw + 4;
    const uint64_t nt = ((row_end - 1) >> tl2) - (row_begin >> tl2) + 1;
    if (nt > 0x7FFFFFFFull) return fail(QR_ERR_SIZE, "CSR build grid too large");
    uint32_t dbuf = 0;
    const uint32_t nh = heavy_fit(t->nheavy, jw);
    const size_t sb = nh ? heavy_stage(nch >= 2, G, jw, heavy_bytes(nh, jw), &dbuf) : stage_bytes(G, jw, &dbuf);
    const uint32_t fl = fold_tiles_log2(nch >= 2, sb, heavy_bytes(nh, jw), nt);
    const size_t shmem = sb + (heavy_bytes(nh, jw) << fl);
    TileOp top{t->gx, t->gterm, t->tz, t->tc, t->rl_ptr, t->rl, d_indices,
               reinterpret_cast<double2 *>(d_data), nullptr, nullptr, nullptr,
               row_begin, row_end, G, jw, nch, dbuf, t->heavy, nh, 0, 0, G, t->ttz, t->ttc, t->ntail, fl};
    auto kst = nh ? (nch <= 1 ? k_csr_build_staged<1, kTileHeavy> : k_csr_build_staged<2, kTileHeavy>)
                  : (nch <= 1 ? k_csr_build_staged<1, kTilePlain> : k_csr_build_staged<2, kTilePlain>);
    QR_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void *>(kst),
                                     hipFuncAttributeMaxDynamicSharedMemorySize, int(shmem)));
    hipLaunchKernelGGL(kst, dim3(unsigned(((nt - 1) >> fl) + 1)), dim3(kStageThreads), shmem, s, top);
    QR_HIP_CHECK(hipGetLastError());
    return QR_OK;
}

// ---------------------------------------------------------------------------
// CSR x vector
// ---------------------------------------------------------------------------
// Entries outside [0, nnz) and columns >= ncols are skipped, so a malformed
// CSR handed in through SpMat.new_unchecked cannot read out of bounds.
//
// LPR lanes share a row, so a wave covers 64/LPR consecutive rows.  For the
// Pauli CSR, rows that differ only in their low bits gather x at columns that
// differ only in those bits, i.e. from the same cache lines, so a wave's
// gathers coalesce.  Blocks are handed to the 8 XCDs round-robin; the block
// index is remapped so that each XCD works on one contiguous range of rows
// and its L2 sees the neighbouring rows' x lines.
// Plain stream loads: nontemporal ones lose in the rows that come here (150
// entries: 3%, 60: 8%, 25 -- the 24-qubit Heisenberg CSR: 13%).
template <int LPR>
__global__ __launch_bounds__(256) void k_csr_matvec(uint64_t nrows, uint64_t ncols, uint64_t nnz,
                                                    uint32_t nblocks_xcd,
                                                    const uint64_t *__restrict__ indptr,
                                                    const uint64_t *__restrict__ indices,
                                                    const double2 *__restrict__ data,
                                                    const double2 *__restrict__ x,
                                                    double2 *__restrict__ y) {
    uint32_t b = blockIdx.x;
    if (nblocks_xcd) b = (b % 8) * nblocks_xcd + b / 8;
    const uint64_t gid = uint64_t(b) * 256 + threadIdx.x;
    const uint64_t row = gid / LPR;
    const int lane = int(threadIdx.x % LPR);
    double2 acc = make_double2(0.0, 0.0);
    if (row < nrows) {
        const uint64_t k0 = min(indptr[row], nnz), k1 = min(indptr[row + 1], nnz);
        uint64_t k = k0 + lane;
        // eight independent entries in flight per lane (measured best of 2, 4, 8);
        // full chunks of U * LPR entries for all lanes of the row together, so
        // that no lane of a row loops while another takes the tail
        constexpr int U = 8;
        for (; k - lane + U * LPR <= k1; k += U * LPR) {
            uint64_t c[U];
            double2 a[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                c[u] = indices[k + u * LPR];
                const dvec2 av = *reinterpret_cast<const dvec2 *>(data + k + u * LPR);
                a[u] = make_double2(av.x, av.y);
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                double2 bx = make_double2(0.0, 0.0);
                if (c[u] < ncols) bx = x[c[u]];
                acc.x = fma(a[u].x, bx.x, acc.x);
                acc.x = fma(-a[u].y, bx.y, acc.x);
                acc.y = fma(a[u].x, bx.y, acc.y);
                acc.y = fma(a[u].y, bx.x, acc.y);
            }
        }
        if (k < k1) {
            // the fewer than U entries left (all of a short row): predicated,
            // with every load issued before the first is used
            uint64_t c[U];
            double2 a[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                c[u] = ~uint64_t(0);
                a[u] = make_double2(0.0, 0.0);
                if (k + u * LPR < k1) {
                    c[u] = indices[k + u * LPR];
                    const dvec2 av = *reinterpret_cast<const dvec2 *>(data + k + u * LPR);
                    a[u] = make_double2(av.x, av.y);
                }
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (c[u] < ncols) {
                    const double2 bx = x[c[u]];
                    acc.x = fma(a[u].x, bx.x, acc.x);
                    acc.x = fma(-a[u].y, bx.y, acc.x);
                    acc.y = fma(a[u].x, bx.y, acc.y);
                    acc.y = fma(a[u].y, bx.x, acc.y);
                }
            }
        }
    }
#pragma unroll
    for (int off = LPR / 2; off > 0; off /= 2) {
        acc.x += __shfl_xor(acc.x, off, LPR);
        acc.y += __shfl_xor(acc.y, off, LPR);
    }
    if (row < nrows && lane == 0) y[row] = acc;
}

// Rows of 8 to 64 entries on average (128 past the MALL): a wave takes 8
// consecutive rows, whose entries are contiguous, streams them in whole lines (U
// loads of 64 consecutive entries, nontemporal: the x lines keep the caches), and
// reads them back from LDS in the gather layout of qr_mv.h: lane (s, t) takes the
// entries s, s + 8, ... of row t, so that the 8 rows that read one x line do so
// in one instruction.  Waves whose rows do not fit that (a general CSR) read them
// from memory in the same per-lane order, kD entries per lane in flight; the sums
// are bit-identical to k_csr_matvec<8>.
// What bounds it: memory, 6.2 TB/s with the x lines read again past L2 (the
// 24-qubit ring: 10.1 GB of CSR, 12.8 GB fetched).
// Matrices past the MALL's 256 MB.  Two rows per 8-lane slot, loaded straight to
// the gather layout / this, us: rings of 20, 23, 24 qubits 118 / 96, 1122 / 948,
// 2460 / 2056; terms of weight 1 to 4, 23 qubits (29 entries) 1385 / 1140; random
// operators of 20 entries, 23 qubits 1044 / 938, 31, 22 qubits 731 / 676; 24, 22
// qubits 547 / 564, where x comes past L2 for every entry; and for
// k_csr_matvec<8> / this, 35, 48, 64 entries, 22 qubits 836 / 754, 1077 / 1073,
// 1439 / 1373; terms of weight 1 to 4 (45 and 57 entries) 1060 / 835, 1318 /
// 1076; for 2 and 4 lanes per row / this, 8, 10, 24 qubits 949 / 867, 1190 /
// 1020, 12, 15, 23 qubits 668 / 544, 839 / 703, but 6, 24 qubits 710 / 789.
// Rows of uneven length (as many lanes per row / this): isotropic rings without
// their zeros, 23, 24, 26 qubits (12.5 to 14 entries in the mean) 727 / 611, 1494
// / 1284, 6690 / 5490; Poisson lengths of 20, 28, 40, 50, 20 to 21 qubits 164 /
// 133, 431 / 329, 267 / 226, 331 / 283; half of the rows 3 and half 40 long 150 /
// 125; one row in 100 of 600 entries, the others 15, 328 / 194 (with one entry per
// lane in flight for the waves that do not fit 422); half 30 and half 90 long,
// the one kind measured slower, 171 / 180.
// Rows of 65 to 128 run blocks of two waves (three blocks' LDS per CU), only in
// matrices of equal rows and 2^25 entries on: 70, 96, 22 qubits 1666 / 1489, 2123
// / 2150, 110, 128, 21 qubits 1309 / 1170, 1442 / 1346, weights 1 to 4, 82 and 110
// entries 1681 / 1525, 2205 / 2115; where the MALL holds the matrix 28 / 33 (100
// entries, 16 qubits).
// Where the MALL holds the matrix the streams gain little, and only equal rows
// of 11 to 63 entries run here: 19 qubits, 12, 20 entries 46 / 46, 58 / 58; random
// operators, 17 qubits, 16, 30, 44, 56 entries 13.7 / 11.3, 21.3 / 18.7, 28.8 / 27.1,
// 34.7 / 36, 16 qubits, 44, 56 entries 15.8 / 13.2, 18.7 / 17.6; but 64, 16 and 17
// qubits 17.5 / 20, 36.4 / 40.8, 8 and 10 entries, 20 and 19 qubits 58 / 65, 41 /
// 44, Poisson lengths of 12, 50, 19 and 17 qubits 42 / 49, 40 / 44.
// U: loads per lane; rows of up to 8 U entries.
constexpr uint64_t kMallBytes = uint64_t(1) << 28;
constexpr uint64_t kShortLongNnz = uint64_t(1) << 25;
template <uint32_t U, uint32_t kWaves = 4>
__global__ __launch_bounds__(64 * kWaves, U <= 3 ? 8 : 1) void k_csr_matvec_short(uint64_t nrows, uint64_t ncols, uint64_t nnz,
                                                          uint32_t nblocks_xcd,
                                                          const uint64_t *__restrict__ indptr,
                                                          const uint64_t *__restrict__ indices,
                                                          const double2 *__restrict__ data,
                                                          const double2 *__restrict__ x,
                                                          double2 *__restrict__ y) {
    constexpr uint32_t kFit = 64 * U;  // entries of a wave's rows
    // entries per lane in flight where the rows do not fit: 8 take 92 VGPRs, which
    // cost U = 4 a wave per SIMD (25 and 29 equal entries, 22 qubits, 4 / 8: 515 /
    // 526, 572 / 581 us; one row in 100 of 600 entries, the others 18, 236 / 213)
    constexpr uint32_t kD = U <= 4 ? 4 : 8;
    __shared__ uint64_t s_idx[kWaves][kFit];
    __shared__ dvec2 s_dat[kWaves][kFit];
    uint32_t b = blockIdx.x;
    if (nblocks_xcd) b = (b % 8) * nblocks_xcd + b / 8;
    const uint32_t wave = threadIdx.x / 64, l = threadIdx.x % 64, ls = l / 8, lt = l % 8;
    const uint64_t r0 = (uint64_t(b) * kWaves + wave) * 8;
    if (r0 >= nrows) return;
    const uint64_t rl = r0 + (l < 8 ? l : 8);
    const uint64_t pl = min(indptr[rl < nrows ? rl : nrows], nnz);  // lane j <= 8: where row r0 + j begins
    const uint64_t first = readlane_u64(pl, 0), end = readlane_u64(pl, 8);
    const uint64_t row = r0 + lt, k0 = __shfl(pl, int(lt)), k1 = __shfl(pl, int(lt) + 1);
    double2 acc = make_double2(0.0, 0.0);
    auto add = [&](dvec2 a, double2 bx) {
        acc.x = fma(a.x, bx.x, acc.x);
        acc.x = fma(-a.y, bx.y, acc.x);
        acc.y = fma(a.x, bx.y, acc.y);
        acc.y = fma(a.y, bx.x, acc.y);
    };
    if (__all(k0 <= k1 && first <= k0 && k1 <= end && end - first <= kFit)) {
        const uint32_t at = uint32_t(k0 - first), len = uint32_t(k1 - k0);
        // U loads and U gathers per lane, none behind a branch
        const uint64_t top = end > first ? end - 1 : first ? first - 1 : 0;
        uint64_t c[U];
        dvec2 a[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            // (lanes past the rows repeat their last entry: the entries there
            // would be fetched twice)
            const uint64_t k = min(first + l + 64 * u, top);
            c[u] = __builtin_nontemporal_load(indices + k);
            a[u] = __builtin_nontemporal_load(reinterpret_cast<const dvec2 *>(data + k));
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            s_idx[wave][l + 64 * u] = c[u];
            s_dat[wave][l + 64 * u] = a[u];
        }
        // LDS writes of other lanes visible to this wave's reads below
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        double2 bx[U];
        bool ok[U];
#pragma unroll
        for (uint32_t u = 0; u < U; ++u) {
            const uint32_t p = ls + 8 * u;
            c[u] = s_idx[wave][(at + p) % kFit];
            a[u] = s_dat[wave][(at + p) % kFit];
            ok[u] = p < len && c[u] < ncols;
            bx[u] = x[ok[u] ? c[u] : 0];
        }
#pragma unroll
        for (uint32_t u = 0; u < U; ++u)
            if (ok[u]) add(a[u], bx[u]);
        for (uint32_t p = ls + 8 * U; p < len; p += 8) {
            const uint64_t cc = s_idx[wave][at + p];
            if (cc < ncols) add(s_dat[wave][at + p], x[cc]);
        }
    } else {
        // kD entries per lane in flight
        for (uint64_t k = k0 + ls; k < k1; k += 8 * kD) {
            uint64_t c[kD];
            dvec2 a[kD];
            double2 bx[kD];
#pragma unroll
            for (uint32_t u = 0; u < kD; ++u) {
                c[u] = ~uint64_t(0);
                a[u] = dvec2{0.0, 0.0};
                if (k + 8 * u < k1) {
                    c[u] = indices[k + 8 * u];
                    a[u] = *reinterpret_cast<const dvec2 *>(data + k + 8 * u);
                }
            }
#pragma unroll
            for (uint32_t u = 0; u < kD; ++u) {
                bx[u] = make_double2(0.0, 0.0);
                if (c[u] < ncols) bx[u] = x[c[u]];
            }
#pragma unroll
            for (uint32_t u = 0; u < kD; ++u)
                if (c[u] < ncols) add(a[u], bx[u]);
        }
    }
#pragma unroll
    for (int off = 32; off >= 8; off /= 2) {
        acc.x += __shfl_xor(acc.x, off);
        acc.y += __shfl_xor(acc.y, off);
    }
    if (ls == 0 && row < nrows) y[row] = acc;
}

// k_csr_matvec_staged (the walker of qr_mv.h over a general CSR): which band
// of x the resident waves read.  In a column-sorted row, chunk c
// covers about the same band of x in every row (1/31 of x, 0.5 MB, for the
// 2000-term CSR), so waves working on the same chunk index read the same
// band, and the XCD's 4 MB L2 serves them.  Blocks start whenever a slot
// frees, and in steady state the resident ones are spread evenly over their
// rows: block i (in launch order on its XCD, of K resident per XCD) starts
// about i/K of a block's lifetime after block 0.  So block i starts its rows
// at chunk i*n/K (mod n, for n chunks) and wraps around: a block then sits at
// the same chunk index as the others when it runs.  Measured on the
// 2000-term CSR: 10.20 ms without the offset, 9.68 ms with it (K = 96, the
// residency on MI355X; 48: 10.99 ms, 192: 10.23 ms), 8.97 ms with every
// gather served from L2 (a timing-only build); a persistent grid (one
// resident set of blocks looping over the rows, all starting at chunk 0)
// took 10.29 ms, its waves drifting apart.  The summation order depends only
// on the block index, so results are reproducible.
// One block per 32 rows; block index remapped so that each XCD works on one
// contiguous range of rows (blocks go to the 8 XCDs round-robin).
template <int C>
__global__ __launch_bounds__(256) void k_csr_matvec_staged(uint64_t nrows, uint64_t ncols, uint64_t nnz,
                                                           uint32_t nblocks_xcd, uint32_t k_res,
                                                           const uint64_t *__restrict__ indptr,
                                                           const uint64_t *__restrict__ indices,
                                                           const double2 *__restrict__ data,
                                                           const double2 *__restrict__ x,
                                                           double2 *__restrict__ y) {
    using S = MvStagedShape<C>;
    extern __shared__ __align__(16) unsigned char mv_lds[];
    uint32_t b = blockIdx.x;
    if (nblocks_xcd) b = (b % 8) * nblocks_xcd + b / 8;
    const int wave = int(threadIdx.x / 64);
    uint64_t *s_idx = reinterpret_cast<uint64_t *>(mv_lds + size_t(wave) * S::kWaveBytes);
    dvec2 *s_dat = reinterpret_cast<dvec2 *>(s_idx + S::kRows * S::kIdxStride);
    // row bounds clamped to [0, nnz), so that a malformed indptr cannot read out
    // of bounds
    auto bounds = [indptr, nnz](uint64_t r, uint64_t *k0, uint64_t *len) {
        const uint64_t a = min(indptr[r], nnz), e = min(indptr[r + 1], nnz);
        *k0 = a;
        *len = e > a ? e - a : 0;
    };
    mv_staged_rows<C>((uint64_t(b) * 4 + uint64_t(wave)) * S::kRows, nrows, ncols, bounds, indices,
                      data, x, y, s_idx, s_dat, blockIdx.x / 8, k_res);
}

// Blocks of k_csr_matvec_staged resident at once on the current device (per
// device, computed once).
static int mv_staged_resident(int *out) {
    static std::mutex mu;
    static int cache[kMaxDevices];
    int dev = 0;
    QR_HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(QR_ERR_ARG, "device index out of range");
    std::lock_guard<std::mutex> lock(mu);
    if (!cache[dev]) {
        int per_cu = 0, cus = 0;
        QR_HIP_CHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(
            &per_cu, reinterpret_cast<const void *>(k_csr_matvec_staged<kMvStagedChunk>), 256,
            4 * MvStagedShape<kMvStagedChunk>::kWaveBytes));
        QR_HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
        cache[dev] = std::max(1, per_cu) * std::max(1, cus);
    }
    *out = cache[dev];
    return QR_OK;
}

int launch_csr_matvec(uint64_t nrows, uint64_t ncols, uint64_t nnz, const uint64_t *d_indptr,
                      const uint64_t *d_indices, const double *d_data, const double *d_x,
                      double *d_y, hipStream_t s) {
    const uint64_t avg = nrows ? nnz / nrows : 0;
    if (avg >= kMvStagedMinRow) {
        using Sh = MvStagedShape<kMvStagedChunk>;
        int resident = 0;
        if (int rc = mv_staged_resident(&resident)) return rc;
        const uint32_t k_res = uint32_t(std::max(1, resident / 8));  // per XCD
        const uint64_t nb = ((nrows + Sh::kRows - 1) / Sh::kRows + 3) / 4;
        if (nb > 0x7FFFFFFFull) return fail(QR_ERR_SIZE, "CSR matvec grid too large");
        const uint32_t nbx = (nb % 8 == 0) ? uint32_t(nb / 8) : 0;
        hipLaunchKernelGGL(k_csr_matvec_staged<kMvStagedChunk>, dim3(unsigned(nb)), dim3(256),
                           4 * Sh::kWaveBytes, s, nrows, ncols, nnz, nbx, k_res, d_indptr, d_indices,
                           reinterpret_cast<const double2 *>(d_data),
                           reinterpret_cast<const double2 *>(d_x), reinterpret_cast<double2 *>(d_y));
        QR_HIP_CHECK(hipGetLastError());
        return QR_OK;
    }
    // ~4+ entries per lane, at most 8 lanes per row (8 rows per wave; 4 and 16
    // to 32 lanes per row measured slower at G = 2000, and 16 no faster at
    // G = 25)
    int lpr = 1;
    while (lpr < 8 && uint64_t(lpr) * 4 <= avg) lpr *= 2;
    const uint64_t threads = nrows * uint64_t(lpr);
    const uint64_t nblocks = (threads + 255) / 256;
    if (nblocks > 0x7FFFFFFFull) return fail(QR_ERR_SIZE, "CSR matvec grid too large");
    const uint32_t nbx = (nblocks % 8 == 0) ? uint32_t(nblocks / 8) : 0;
    auto x = reinterpret_cast<const double2 *>(d_x);
    auto data = reinterpret_cast<const double2 *>(d_data);
    auto y = reinterpret_cast<double2 *>(d_y);
    const dim3 grid(static_cast<unsigned>(nblocks)), block(256);
    const bool equal = nnz % nrows == 0, in_mall = nnz * 24 <= kMallBytes;
    if (ncols && avg >= 8 && (in_mall ? equal && avg >= 11 && avg < 64
                                      : avg <= 64 || (avg <= 128 && equal && nnz >= kShortLongNnz))) {
        // a wave's eight rows are to fit, with an eighth to spare where they
        // cannot be equal
        const uint64_t need = equal ? avg : avg + avg / 8 + 1;
        const uint32_t waves = need > 64 ? 2 : 4;  // (the LDS of three blocks per CU)
        const uint64_t nb = (nrows + 8 * waves - 1) / (8 * waves);
        if (nb > 0x7FFFFFFFull) return fail(QR_ERR_SIZE, "CSR matvec grid too large");
        const uint32_t nbx_short = (nb % 8 == 0) ? uint32_t(nb / 8) : 0;
        auto kern = need <= 8    ? k_csr_matvec_short<1>
                    : need <= 16 ? k_csr_matvec_short<2>
                    : need <= 24 ? k_csr_matvec_short<3>
                    : need <= 32 ? k_csr_matvec_short<4>
                    : need <= 48 ? k_csr_matvec_short<6>
                    : need <= 64 ? k_csr_matvec_short<8>
                    : need <= 96 ? k_csr_matvec_short<12, 2>
                                 : k_csr_matvec_short<16, 2>;
        hipLaunchKernelGGL(kern, dim3(unsigned(nb)), dim3(64 * waves), 0, s, nrows, ncols, nnz, nbx_short, d_indptr,
                           d_indices, data, x, y);
        QR_HIP_CHECK(hipGetLastError());
        return QR_OK;
    }
    auto kern = lpr == 1 ? k_csr_matvec<1> : lpr == 2 ? k_csr_matvec<2> : lpr == 4 ? k_csr_matvec<4> : k_csr_matvec<8>;
    hipLaunchKernelGGL(kern, grid, block, 0, s, nrows, ncols, nnz, nbx, d_indptr, d_indices, data, x, y);
    QR_HIP_CHECK(hipGetLastError());
    return QR_OK;
}

}  // namespace qr
