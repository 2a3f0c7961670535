// qr_api.cpp -- host side of libqrhip: labels, operators, modes, C ABI glue.
//
// Mirrors the reference's host logic (qrusty/src/lib.rs:117-585 and
// accel.rs:141-157) and prepares the device tables the HIP kernels read:
//   * terms grouped by x mask (a stable sort, so a group's terms keep their
//     input order, which is the order make_row folds them in, accel.rs:188-208);
//   * per-group "rank lists" that give each group's position in the ascending
//     column order of any row r without sorting (see build_rank_lists).
#include "qr_internal.h"

#include <algorithm>
#include <cstring>
#include <numeric>
#include <utility>

namespace qr {

static thread_local std::string g_last_error;

int fail(int code, const std::string &msg) {
    g_last_error = msg;
    return code;
}

int hip_fail(hipError_t e, const char *what) {
    return fail(QR_ERR_HIP, std::string("HIP error in ") + what + ": " + hipGetErrorString(e));
}

// Label grammar of qrusty/src/lib.rs:127: ^([+-]?)1?([ij]?)([IXYZ]+)$.
// Qubit q is label[len-1-q] (lib.rs:144); x bit for X|Y and z bit for Y|Z
// (lib.rs:80-91); phase = (base_phase + #Y) mod 4 (lib.rs:179-181).
static int parse_label(const char *s, uint32_t *nq, uint32_t *base_phase, uint32_t *ny,
                       uint64_t *x, uint64_t *z) {
    if (!s) return fail(QR_ERR_ARG, "null label");
    const char *p = s;
    bool neg = false, imag = false;
    if (*p == '+' || *p == '-') { neg = (*p == '-'); ++p; }
    if (*p == '1') ++p;
    if (*p == 'i' || *p == 'j') { imag = true; ++p; }
    size_t n = std::strlen(p);
    if (n == 0) return fail(QR_ERR_LABEL, "error: malformed label");
    bool known = true;
    for (size_t k = 0; k < n; ++k)
        known &= (p[k] == 'I') | (p[k] == 'X') | (p[k] == 'Y') | (p[k] == 'Z');
    if (!known) return fail(QR_ERR_LABEL, "error: malformed label");
    if (n > 63) return fail(QR_ERR_SIZE, "Pauli labels of more than 63 qubits are not supported");
    uint64_t xm = 0, zm = 0;
    for (size_t k = 0; k < n; ++k) {
        const char c = p[k];
        xm = 2 * xm | uint64_t((c == 'X') | (c == 'Y'));
        zm = 2 * zm | uint64_t((c == 'Y') | (c == 'Z'));
    }
    const uint32_t y = uint32_t(__builtin_popcountll(xm & zm));
    *nq = uint32_t(n);
    *base_phase = (imag ? 1u : 0u) + (neg ? 2u : 0u);
    *ny = y;
    *x = xm;
    *z = zm;
    return QR_OK;
}

// Rank lists.  Sort the G distinct masks ascending (the column order of row 0)
// and view them as a binary trie, splitting at the highest differing bit.
// Row r orders its columns r ^ x ascending, which is the same trie with the
// two children of every node splitting at bit b swapped when bit b of r is
// set.  A group at sorted position j therefore sits at
//     rank_r(j) = j + sum over the splitting nodes on its path with r_b = 1 of
//                 (+size of right child if j is in the left child,
//                  -size of left child  if j is in the right child).
// Each (bit, sigma) pair is one RankEntry; a path has at most min(n, G-1) of them.
static void build_rank_lists(const std::vector<uint64_t> &gx, std::vector<uint32_t> &ptr,
                             std::vector<RankEntry> &out) {
    const uint32_t G = uint32_t(gx.size());
    ptr.assign(size_t(G) + 1, 0);
    out.clear();
    RankEntry path[64];
    auto walk = [&](auto &self, uint32_t lo, uint32_t hi, int depth) -> void {
        if (hi - lo <= 1) {
            out.insert(out.end(), path, path + depth);
            ptr[hi] = uint32_t(out.size());
            return;
        }
        const uint64_t diff = gx[lo] ^ gx[hi - 1];
        const int b = 63 - __builtin_clzll(diff);
        const uint64_t bit = uint64_t(1) << b;
        // sorted and sharing all bits above b: first index with bit b set
        const uint32_t m = uint32_t(std::partition_point(gx.begin() + lo, gx.begin() + hi,
                                                         [bit](uint64_t v) { return (v & bit) == 0; }) -
                                    gx.begin());
        path[depth] = {b, int32_t(hi - m)};
        self(self, lo, m, depth + 1);
        path[depth] = {b, -int32_t(m - lo)};
        self(self, m, hi, depth + 1);
    };
    walk(walk, 0, G, 0);
}

static void free_patterns(DeviceTables::Patterns &pt);

void free_tables(DeviceTables &t) {
    if (t.apart)
        for (void *p : {(void *)t.gx, (void *)t.gterm, (void *)t.tz, (void *)t.tc, (void *)t.rl_ptr, (void *)t.rl,
                        (void *)t.gkind})
            if (p) (void)hipFree(p);
    if (t.mem) (void)hipFree(t.mem);
    if (t.word_mem) (void)hipFree(t.word_mem);
    for (auto &pt : t.pat) free_patterns(pt);
    t = DeviceTables{};
}

// A part under construction: patterns whose zl span at most kPartRank
// dimensions.  basis[j]: the zl that raised the rank to j + 1; red: the same
// span in echelon form, leading bits descending, comb[i] = red[i]'s
// coordinates in the basis.
struct PartBuild {
    uint64_t basis[kPartRank] = {}, red[kPartRank] = {};
    uint32_t comb[kPartRank] = {};
    int rank = 0;
    uint32_t n = 0;
    size_t pats[1 << kPartRank];
    uint32_t code[1 << kPartRank];  // coordinates of each pattern's zl
    // v minus its component in the span; the component's coordinates in *c
    uint64_t reduce(uint64_t v, uint32_t *c) const {
        *c = 0;
        for (int i = 0; i < rank; ++i)
            if ((v >> (63 - __builtin_clzll(red[i]))) & 1) {
                v ^= red[i];
                *c ^= comb[i];
            }
        return v;
    }
    bool add(size_t p, uint64_t zl) {
        uint32_t c;
        const uint64_t rest = reduce(zl, &c);
        if (rest) {
            if (rank == kPartRank) return false;
            basis[rank] = zl;
            c ^= 1u << rank;  // rest in the basis
            int at = rank;
            while (at > 0 && red[at - 1] < rest) {
                red[at] = red[at - 1];
                comb[at] = comb[at - 1];
                --at;
            }
            red[at] = rest;
            comb[at] = c;
            c = 1u << rank;  // zl in the basis
            ++rank;
        }
        pats[n] = p;
        code[n++] = c;
        return true;
    }
    // table index bits of row bit i
    uint32_t col(int i) const {
        uint32_t c = 0;
        for (int j = 0; j < rank; ++j) c |= uint32_t((basis[j] >> i) & 1) << j;
        return c;
    }
};

// Patterns: inside a tile of 2^L rows (fixed high bits h, low bits l), term t
// of group g contributes (-1)^popcount(h & z_t) * c'_t * (-1)^popcount(l & zl_t)
// with zl_t = z_t & (2^L - 1).  Terms of a group that share zl_t therefore
// merge, per tile, into one coefficient.  A group's patterns, by ascending zl,
// go to the first part whose span holds their zl, else to the last part while
// its rank is below kPartRank, else to a new one; the kernel tabulates each
// part per tile (ApplyPart) and a row looks its value up.  Ascending zl keeps
// the patterns of neighbouring bits together: the diagonal of a spin ring (two
// patterns per bit) takes one part per three or four bits.  Terms keep input
// order inside a pattern.  With `pairs` the low bits are taken in the
// paired-row order (pair_row_bits).
void build_patterns(const qr_op *op, const PatternShape &shape, const std::vector<uint8_t> &pass, uint8_t id,
                    HostPatterns &out) {
    const int L = shape.L, tb = shape.tb;
    const bool staged = shape.staged, pairs = shape.pairs;
    const uint64_t mask = L >= 64 ? ~uint64_t(0) : ((uint64_t(1) << L) - 1);
    // a mask's bits in the tile's row order (window passes: bits [0, f) and
    // [s, s + L - f); the others are not part of the tile)
    const ApplyWindow win = shape.win;
    auto tile_bits = [&](uint64_t v) {
        if (!win.s) return v & mask;
        const uint64_t low = (uint64_t(1) << win.f) - 1;
        return ((v & low) | ((v >> win.s) << win.f)) & mask;
    };
    out = HostPatterns{};
    ApplyChunk cur{};
    uint32_t cur_bytes = 0;  // table bytes of the chunk
    std::vector<uint8_t> gcls;  // class of each group of the chunk, without the far bit
    for (uint64_t g = 0; g < op->G; ++g) {
        if (!pass.empty() && pass[g] != id) continue;
        for (uint32_t i = op->gterm[g]; i < op->gterm[g + 1]; ++i) out.cplx = out.cplx || op->tc[2 * i + 1] != 0.0;
    }
    const int lg = out.cplx ? 4 : 3;  // log2 bytes of a table entry
    const uint64_t far_mask = ~mask;
    // closes the chunk: its groups are reordered by class, or (staged) by
    // partner tile and then class
    auto close_chunk = [&]() {
        const uint32_t g0 = cur.cg[0], g1 = uint32_t(out.grp.size()), n = g1 - g0;
        cur.t1 = uint32_t(out.tab.size());
        cur.r0 = cur.r1 = uint32_t(out.run.size());
        if (n) {
            std::vector<uint32_t> order(n);
            std::iota(order.begin(), order.end(), 0u);
            const std::vector<ApplyGroup> was(out.grp.begin() + g0, out.grp.end());
            auto cls = [&](uint32_t i) { return ((was[i].m & far_mask) ? 2u : 0u) | gcls[i]; };
            auto hi = [&](uint32_t i) { return was[i].m & far_mask; };
            if (!staged)
                std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) { return cls(a) < cls(b); });
            else
                std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) { return hi(a) > hi(b); });
            for (uint32_t i = 0; i < n; ++i) out.grp[g0 + i] = was[order[i]];
            if (!staged) {
                uint32_t c = 0;
                for (uint32_t i = 0; i <= n; ++i) {
                    const uint32_t cg = i < n ? cls(order[i]) : uint32_t(kApplyClasses);
                    while (c <= cg && c <= uint32_t(kApplyClasses)) cur.cg[c++] = g0 + i;
                }
            } else {
                for (uint32_t i = 0; i < n; ++i) {
                    if (i + 1 < n && hi(order[i + 1]) == hi(order[i])) continue;
                    ApplyRun r{};
                    r.hi = hi(order[i]);
                    r.g1 = g0 + i + 1;
                    out.run.push_back(r);
                }
                cur.r1 = uint32_t(out.run.size());
                for (uint32_t c = 0; c <= uint32_t(kApplyClasses); ++c) cur.cg[c] = g0;
                cur.cg[kApplyClasses] = g1;
            }
            out.chunk.push_back(cur);
            out.max_tab = std::max(out.max_tab, cur_bytes);
        }
        cur = ApplyChunk{};
        cur.cg[0] = g1;
        cur.t0 = uint32_t(out.tab.size());
        cur_bytes = 0;
        gcls.clear();
    };
    if (pass.empty()) {
        out.grp.reserve(op->G);
        out.tab.reserve(op->G);
        out.pat.reserve(16 * op->G);
        out.ptz.reserve(op->T);
        out.ptc.reserve(2 * op->T);
    }
    std::vector<std::pair<uint64_t, uint32_t>> zt;  // a group's (zl, term)
    std::vector<size_t> heads;                      // first term of each pattern
    std::vector<PartBuild> parts;
    std::vector<uint32_t> where;
    for (uint64_t k = 0; k < op->G; ++k) {
        const uint64_t g = staged ? op->G - 1 - k : k;
        if (!pass.empty() && pass[g] != id) continue;
        // window passes keep the mask in the tile's row order
        const uint64_t gm = win.s ? tile_bits(op->gx[g]) : op->gx[g];
        zt.clear();
        for (uint32_t i = op->gterm[g]; i < op->gterm[g + 1]; ++i)
            zt.emplace_back(pairs ? pair_row_bits(tile_bits(op->tz[i]), tb) : tile_bits(op->tz[i]), i);
        std::sort(zt.begin(), zt.end());
        heads.clear();
        for (size_t i = 0; i < zt.size(); ++i)
            if (i == 0 || zt[i].first != zt[i - 1].first) heads.push_back(i);
        heads.push_back(zt.size());
        const size_t npat = heads.size() - 1;
        for (size_t s0 = 0; s0 < npat; s0 += shape.psplit) {
            const size_t s1 = std::min(npat, s0 + shape.psplit);
            parts.clear();
            for (size_t s = s0; s < s1; ++s) {
                const uint64_t zl = zt[heads[s]].first;
                bool placed = false;
                uint32_t c;
                for (size_t k = 0; k < parts.size() && !placed; ++k)
                    if (k + 1 == parts.size() || parts[k].reduce(zl, &c) == 0) placed = parts[k].add(s, zl);
                if (!placed) {
                    parts.emplace_back();
                    parts.back().add(s, zl);
                }
            }
            bool real = true;
            for (size_t i = heads[s0]; i < heads[s1]; ++i) real = real && op->tc[2 * zt[i].second + 1] == 0.0;
            // each table aligned to its size
            auto place = [&](uint32_t at, std::vector<uint32_t> *where) {
                for (const PartBuild &p : parts) {
                    const uint32_t size = 1u << (p.rank + lg);
                    at = (at + size - 1) & ~(size - 1);
                    if (where) where->push_back(at);
                    at += size;
                }
                return at;
            };
            if (place(cur_bytes, nullptr) > shape.tcap) close_chunk();
            where.clear();
            cur_bytes = place(cur_bytes, &where);
            ApplyGroup a{};
            a.m = gm;
            bool rowvar = false;
            for (size_t k = 0; k < parts.size(); ++k) {
                const PartBuild &p = parts[k];
                // index of the bits [bit0, bit0 + nbits) = v
                auto span = [&p](int bit0, int nbits, uint32_t *to) {
                    to[0] = 0;
                    for (int i = 0; i < nbits; ++i) {
                        const uint32_t c = p.col(bit0 + i);
                        for (uint32_t v = 0; v < 1u << i; ++v) to[v | 1u << i] = to[v] ^ c;
                    }
                };
                uint32_t s0[8], s1[8], s2[4], sr[8];
                span(0, 3, s0);
                span(3, 3, s1);
                span(6, 2, s2);
                span(tb, 3, sr);
                ApplyPart ap{};
                for (uint32_t v = 0; v < 8; ++v) {
                    ap.w0 |= s0[v] << (4 * v);
                    ap.w1 |= s1[v] << (4 * v);
                    ap.rc |= uint64_t(sr[v] << lg) << (8 * v);
                }
                for (uint32_t v = 0; v < 4; ++v) ap.w2 |= (s2[v] << lg) << (8 * v);
                ap.tab = (shape.tab0 + where[k]) / 4;
                rowvar = rowvar || ap.rc;
                if (parts.size() == 1) {
                    a.w0 = ap.w0;
                    a.w1 = ap.w1;
                    a.w2 = ap.w2;
                    a.rc = ap.rc;
                    a.tab_n = ap.tab | (1u << 16);
                } else {
                    if (k == 0) {
                        a.w0 = uint32_t(out.part.size());
                        a.tab_n = uint32_t(parts.size()) << 16;
                    }
                    out.part.push_back(ap);
                }
                size_t by_code[16];
                std::fill(by_code, by_code + 16, npat);
                for (uint32_t i = 0; i < p.n; ++i) by_code[p.code[i]] = p.pats[i];
                for (uint32_t c = 0; c < 16; ++c) {
                    ApplyRange pr{uint32_t(out.ptz.size()), 0};
                    for (size_t q = by_code[c] < npat ? heads[by_code[c]] : 0;
                         by_code[c] < npat && q < heads[by_code[c] + 1]; ++q) {
                        const uint32_t t = zt[q].second;
                        out.ptz.push_back(op->tz[t]);
                        out.ptc.push_back(op->tc[2 * t]);
                        out.ptc.push_back(op->tc[2 * t + 1]);
                    }
                    pr.t1 = uint32_t(out.ptz.size());
                    out.pat.push_back(pr);
                }
                out.tab.push_back(ap.tab | (1u << (16 + p.rank)));
            }
            a.tab_n |= (rowvar ? kGroupRowvar : 0u) | (real ? 0u : kGroupCplx);
            gcls.push_back(uint8_t(pairs ? a.m & 1 : 0));
            out.grp.push_back(a);
        }
    }
    close_chunk();
}

// Arrays that go to the device in one allocation and, up to kStageBytes, one
// copy: each allocation and each copy of its own costs 10-20 us, which a small
// operator's dozen tables made the larger part of its first call.
class TableSet {
    static constexpr size_t kStageBytes = size_t(32) << 20;
    struct Piece {
        void **dst;
        const void *src;
        size_t bytes, at;
    };
    std::vector<Piece> pieces_;
    size_t total_ = 0;

  public:
    template <typename T>
    void add(T **dst, const void *src, size_t n) {
        pieces_.push_back({reinterpret_cast<void **>(dst), src, n * sizeof(T), total_});
        total_ += (std::max<size_t>(n, 1) * sizeof(T) + 255) & ~size_t(255);
    }
    template <typename T>
    void add(T **dst, const std::vector<T> &src) { add(dst, src.data(), src.size()); }
    int upload(void **mem) const {
        if (!total_) return QR_OK;
        QR_HIP_CHECK(hipMalloc(mem, total_));
        unsigned char *base = static_cast<unsigned char *>(*mem);
        if (total_ <= kStageBytes) {
            std::vector<unsigned char> host(total_);
            for (const Piece &p : pieces_)
                if (p.bytes) std::memcpy(host.data() + p.at, p.src, p.bytes);
            QR_HIP_CHECK(hipMemcpy(base, host.data(), total_, hipMemcpyHostToDevice));
        } else {
            for (const Piece &p : pieces_)
                if (p.bytes) QR_HIP_CHECK(hipMemcpy(base + p.at, p.src, p.bytes, hipMemcpyHostToDevice));
        }
        for (const Piece &p : pieces_) *p.dst = base + p.at;
        return QR_OK;
    }
};

// The sign-word builder's tables; `rank` holds one of them until the upload.
static void add_words(const qr_op *op, DeviceTables &t, TableSet &set, std::vector<int32_t> &rank) {
    // rank lists by bit, without the sub-operators' ancestors
    rank.resize(uint64_t(op->nq) * op->G);
    for (const auto &lf : op->word_leaves) {
        uint32_t depth = 0;
        for (int32_t v : lf.off) depth += v != 0;
        for (uint32_t g = lf.s0; g < lf.s0 + lf.g; ++g)
            for (uint32_t e = op->rl_ptr[g] + depth; e < op->rl_ptr[g + 1]; ++e)
                rank[uint64_t(op->rl[e].bit) * op->G + g] = op->rl[e].sigma;
    }
    set.add(&t.word_leaves, op->word_leaves);
    set.add(&t.word_groups, op->word_groups);
    set.add(&t.word_rank, rank);
    set.add(&t.word_ptr, op->word_ptr);
    set.add(&t.word_terms, op->word_terms);
}

// with_base: also the tables that qr_group.hip builds on the device;
// with_words: also the sign-word builder's, in the same copy
int upload_tables(const qr_op *op, DeviceTables &t, bool with_base, bool with_words) {
    TableSet set;
    if (with_base) {
        set.add(&t.gx, op->gx);
        set.add(&t.gterm, op->gterm);
        set.add(&t.tz, op->tz);
        set.add(&t.tc, op->tc.data(), op->T);
        set.add(&t.rl_ptr, op->rl_ptr);
        set.add(&t.rl, op->rl);
        set.add(&t.gkind, op->gkind);
    }
    if (!op->heavy.empty()) set.add(&t.heavy, op->heavy);
    if (!op->leaf_heavy.empty()) set.add(&t.leaf_heavy, op->leaf_heavy);
    std::vector<int32_t> rank;
    with_words = with_words && !op->word_leaves.empty();
    if (with_words) add_words(op, t, set, rank);
    if (op->ntail) {
        set.add(&t.ttz, op->ttz);
        set.add(&t.ttc, op->ttc.data(), op->ttz.size());
    }
    t.apart = !with_base;
    if (int rc = set.upload(&t.mem)) return rc;
    t.nheavy = uint32_t(op->heavy.size());
    t.ntail = op->ntail;
    t.words = with_words;
    return QR_OK;
}

int word_tables(const qr_op *op, DeviceTables *t, hipStream_t s, bool *have) {
    std::lock_guard<std::mutex> lock(op->mu);
    *have = t->words;
    if (t->words || op->word_leaves.empty()) return QR_OK;
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &st) != hipSuccess) {
        (void)hipGetLastError();
        return QR_OK;
    }
    if (st != hipStreamCaptureStatusNone) return QR_OK;
    TableSet set;
    std::vector<int32_t> rank;
    add_words(op, *t, set, rank);
    if (int rc = set.upload(&t->word_mem)) return rc;
    *have = t->words = true;
    return QR_OK;
}

int device_tables(const qr_op *op, DeviceTables **out, bool noalloc, bool with_words) {
    int dev = 0;
    QR_HIP_CHECK(hipGetDevice(&dev));
    if (dev < 0 || dev >= kMaxDevices) return fail(QR_ERR_ARG, "device index out of range");
    std::lock_guard<std::mutex> lock(op->mu);
    DeviceTables &t = op->dev[dev];
    if (!t.ready && noalloc)
        return fail(QR_ERR_ARG, "apply_noalloc: the operator's tables are not on this device "
                                "(one qr_pauli_apply of it on this device uploads them)");
    if (!t.ready) {
        if (int rc = upload_tables(op, t, true, with_words)) {
            free_tables(t);
            return rc;
        }
        t.ready = true;
    }
    *out = &t;
    return QR_OK;
}

bool tables_ready(const qr_op *op, const DeviceTables *t, int slot, int L) {
    std::lock_guard<std::mutex> lock(op->mu);
    return t->pat[slot].L == L;
}

// Which groups run in window passes.  In the pass over tiles of consecutive
// rows, every distinct value of the mask bits above the tile is a partner
// tile that each tile reads; those whose mask stays within about 2^17
// complex128 rows find it in the XCD's 4 MB L2, the others read it past L2,
// at the 6.2-7 TB/s that HBM and the MALL deliver (L2: 31 TB/s).  A window
// pass reads x once, and y once and writes it once more, whatever the number
// of masks it holds: three streams of the state.  So the windows [s, s + w)
// that save the most partner streams are taken in turn while they save at
// least kWindowMinSaved (a partner stream is saved when all groups that share
// it move).  Up to the MALL's 256 MB that is done if together they save half
// of the partners past L2 (the return value): nearest-neighbour rings and
// chains, whose masks are a few adjacent bits.  Measured, one state / 8 states,
// without and with: 24-qubit ring 432 -> 301 us / 3.49 -> 2.91 ms, 22 qubits
// 107 -> 78 / 697 -> 633 us; k-local and molecular operators, where windows
// save a sixth of the partners, lost 1-5% with them.  For states past the
// MALL every partner is read from HBM: k-local, 28 qubits and 1000 terms 94
// -> 80 ms, 26 qubits and 3000 terms 35.2 -> 33.9.
// FP64 only: y goes through memory from pass to pass, which keeps a sum of
// doubles and would round the running sum of a complex64 state once per pass.
constexpr uint32_t kWindowMinSaved = 5;
constexpr int kWindowMinStateLog2 = 25, kMallLog2 = 28;  // bytes of one state
bool choose_windows(const qr_op *op, int L, std::vector<ApplyWindow> &wins,
                    std::vector<uint8_t> &pass) {
    wins.clear();
    pass.assign(op->G, 0);
    const int n = int(op->nq), state_log2 = n + 4;
    const bool past_mall = state_log2 > kMallLog2;
    if (state_log2 < kWindowMinStateLog2) return false;
    const int f = 3;  // 128-byte segments
    const int w = L - f, near = 17;
    // gx ascends: the groups of one partner are adjacent
    struct Partner { uint64_t g0, g1, bits; };
    std::vector<Partner> far;
    for (uint64_t g = 0; g < op->G;) {
        uint64_t e = g, bits = 0;
        while (e < op->G && (op->gx[e] >> L) == (op->gx[g] >> L)) bits |= op->gx[e++];
        if (op->gx[e - 1] >> near) far.push_back({g, e, bits});
        g = e;
    }
    while (int(wins.size()) < kMaxWindows) {
        uint32_t best = 0;
        int best_s = 0;
        auto inside = [&](const Partner &p, int s) {
            const uint64_t tile = ((uint64_t(1) << f) - 1) | (((uint64_t(1) << w) - 1) << s);
            return pass[p.g0] == 0 && (p.bits & ~tile) == 0;
        };
        for (int s = n - w; s >= f + 1; --s) {
            uint32_t saved = 0;
            for (const Partner &p : far) saved += inside(p, s) ? 1u : 0u;
            if (saved > best) {
                best = saved;
                best_s = s;
            }
        }
        if (best < kWindowMinSaved) break;
        wins.push_back({uint32_t(f), uint32_t(best_s)});
        for (const Partner &p : far)
            if (inside(p, best_s))
                for (uint64_t g = p.g0; g < p.g1; ++g) pass[g] = uint8_t(wins.size());
    }
    size_t moved = 0;
    for (const Partner &p : far) moved += pass[p.g0] != 0;
    const bool most = !wins.empty() && 2 * moved >= far.size();
    if (!most && !past_mall) {
        wins.clear();
        pass.assign(op->G, 0);
    }
    return most;
}

static int upload_patterns(DeviceTables::Patterns &pt, const HostPatterns &hp, const PatternShape &shape) {
    TableSet set;
    set.add(&pt.grp, hp.grp);
    set.add(&pt.chunk, hp.chunk);
    if (shape.staged) set.add(&pt.run, hp.run);
    set.add(&pt.part, hp.part);
    set.add(&pt.tab, hp.tab);
    set.add(&pt.pat, hp.pat);
    set.add(&pt.ptz, hp.ptz);
    set.add(&pt.ptc, hp.ptc.data(), hp.ptz.size());
    if (int rc = set.upload(&pt.mem)) return rc;
    pt.nchunk = uint32_t(hp.chunk.size());
    pt.nrun = uint32_t(hp.run.size());
    pt.max_tab = hp.max_tab;
    pt.cplx = hp.cplx;
    pt.win = shape.win;
    return QR_OK;
}

static void free_patterns(DeviceTables::Patterns &pt) {
    if (pt.mem) (void)hipFree(pt.mem);
    pt = DeviceTables::Patterns{};
}

int device_patterns(const qr_op *op, DeviceTables *t, int slot, const PatternShape &shape,
                    const PatternShape &win_shape, bool noalloc) {
    std::lock_guard<std::mutex> lock(op->mu);
    DeviceTables::Patterns &pt = t->pat[slot];
    if (pt.L == shape.L) return QR_OK;
    if (noalloc)
        return fail(QR_ERR_ARG, "apply_noalloc: the operator's apply tables for this precision "
                                "are not on this device (one qr_pauli_apply of it with this "
                                "precision on this device uploads them)");
    for (int k = 0; k <= kMaxWindows; ++k) free_patterns(t->pat[slot + kApplySlots * k]);
    std::vector<ApplyWindow> wins;
    std::vector<uint8_t> pass;
    if (win_shape.L) choose_windows(op, win_shape.L, wins, pass);
    HostPatterns hp;
    int rc;
    for (size_t k = 0; k < wins.size(); ++k) {
        PatternShape ws = win_shape;
        ws.win = wins[k];
        build_patterns(op, ws, pass, uint8_t(k + 1), hp);
        DeviceTables::Patterns &pw = t->pat[slot + kApplySlots * int(k + 1)];
        if ((rc = upload_patterns(pw, hp, ws))) return rc;
        pw.L = ws.L;
    }
    build_patterns(op, shape, pass, 0, hp);
    if ((rc = upload_patterns(pt, hp, shape))) return rc;
    pt.nwin = uint32_t(wins.size());
    pt.L = shape.L;
    return QR_OK;
}

// The parts of an operator derived from its grouped tables (gx, gterm):
// the sub-operators (subtrees of at most kSubMaxG groups) and heavy groups.
void finish_op(qr_op *op) {
    // subtrees of at most `most` groups, split where build_rank_lists splits
    auto cut = [op](uint32_t most, std::vector<qr_op::SubLeaf> &leaves) {
        if (op->G <= most) return;
        struct Node { uint32_t lo, hi, depth; };
        std::vector<Node> stack{{0, uint32_t(op->G), 0}};
        while (!stack.empty()) {
            const Node nd = stack.back();
            stack.pop_back();
            if (nd.hi - nd.lo <= most) {
                leaves.push_back({nd.lo, nd.hi, nd.depth, 0, 0});
                continue;
            }
            const uint64_t bit = uint64_t(1) << (63 - __builtin_clzll(op->gx[nd.lo] ^ op->gx[nd.hi - 1]));
            const uint32_t m = uint32_t(std::partition_point(op->gx.begin() + nd.lo,
                                                             op->gx.begin() + nd.hi,
                                                             [bit](uint64_t v) { return (v & bit) == 0; }) -
                                        op->gx.begin());
            stack.push_back({m, nd.hi, nd.depth + 1});
            stack.push_back({nd.lo, m, nd.depth + 1});
        }
    };
    cut(kSubMaxG, op->leaves);
    // heavy groups: at least 8 terms and 4x the mean, the largest kMaxHeavy
    {
        const double mean = double(op->T) / double(op->G);
        std::vector<std::pair<uint32_t, uint32_t>> cand;  // (terms, group)
        for (uint64_t g = 0; g < op->G; ++g) {
            const uint32_t n = op->gterm[g + 1] - op->gterm[g];
            if (n >= 8 && double(n) >= 4.0 * mean) cand.emplace_back(n, uint32_t(g));
        }
        std::sort(cand.begin(), cand.end(), [](const auto &a, const auto &b) {
            return a.first != b.first ? a.first > b.first : a.second < b.second;
        });
        if (cand.size() > kMaxHeavy) cand.resize(kMaxHeavy);
        for (const auto &c : cand) op->heavy.push_back(c.second);
        std::sort(op->heavy.begin(), op->heavy.end());
        // each sub-operator's heavy groups, in its own (leaf-local) indices
        auto split = [op](std::vector<qr_op::SubLeaf> &leaves, std::vector<uint32_t> &heavy) {
            for (auto &lf : leaves) {
                lf.hoff = uint32_t(heavy.size());
                for (uint32_t g : op->heavy)
                    if (g >= lf.s0 && g < lf.s1) heavy.push_back(g - lf.s0);
                lf.hcnt = uint32_t(heavy.size()) - lf.hoff;
            }
        };
        split(op->leaves, op->leaf_heavy);
    }
    // the form of the sign-word builder: terms past those it holds are loaded
    // again for every row, so they have to be few
    bool real = true;
    for (uint64_t i = 0; i < op->T; ++i) real = real && op->tc[2 * i + 1] == 0.0;
    uint64_t past = 0;
    for (uint64_t g = 0; g < op->G; ++g) {
        const uint64_t n = op->gterm[g + 1] - op->gterm[g];
        if (n > kWordHold && !std::binary_search(op->heavy.begin(), op->heavy.end(), uint32_t(g)))
            past += n - kWordHold;
    }
    op->word_real = real && 16 * past <= op->G;
    if (op->nq <= 32) {
        std::vector<qr_op::SubLeaf> leaves;
        cut(kWordMaxG, leaves);
        if (leaves.empty()) leaves.push_back({0, uint32_t(op->G), 0, 0, 0});
        auto threads = [](const auto &l) { return l.s1 - l.s0 <= 256 ? 256u : l.s1 - l.s0 <= 512 ? 512u : 1024u; };
        uint64_t most = 0, sum = 0;
        for (const auto &l : leaves) {
            most = std::max<uint64_t>(most, threads(l));
            sum += threads(l);
        }
        op->word_joint = most * leaves.size() <= 2 * sum && (op->word_real || op->T <= 4 * op->G);
        if (!op->word_joint)
            std::stable_sort(leaves.begin(), leaves.end(),
                             [&](const auto &a, const auto &b) { return threads(a) < threads(b); });
        op->word_groups.resize(op->G);
        for (const auto &l : leaves) {
            WordLeaf lf{l.s0, l.s1 - l.s0, 0, uint32_t(op->word_ptr.size()), {}};
            for (uint32_t e = op->rl_ptr[l.s0]; e < op->rl_ptr[l.s0] + l.depth; ++e) lf.off[op->rl[e].bit] = op->rl[e].sigma;
            for (uint32_t g = l.s0; g < l.s1; ++g) {
                const uint32_t t0 = op->gterm[g], t1 = op->gterm[g + 1];
                op->word_groups[g] = {uint32_t(op->gx[g]), t0, t1 - t0, -1};
                if (!std::binary_search(op->heavy.begin(), op->heavy.end(), g)) continue;
                op->word_groups[g].heavy = int32_t(lf.hcnt++);
                op->word_ptr.push_back(uint32_t(op->word_terms.size()));
                for (uint32_t i = t0; i < t1; ++i)
                    op->word_terms.push_back({op->tc[2 * i], op->tc[2 * i + 1], uint32_t(op->tz[i]), 0});
            }
            op->word_ptr.push_back(uint32_t(op->word_terms.size()));
            op->word_leaves.push_back(lf);
        }
    }
    // tail table: operators with heavy groups, whose other groups also run
    // past two terms (the molecular Hamiltonians: 4 and 6), and those of many
    // terms per group
    if (!op->heavy.empty() || op->T >= 2 * op->G) {
        uint32_t nt = 0;
        for (uint64_t g = 0; g < op->G; ++g) {
            const uint32_t n = op->gterm[g + 1] - op->gterm[g];
            if (n > 2 && !std::binary_search(op->heavy.begin(), op->heavy.end(), uint32_t(g)))
                nt = std::max(nt, n - 2);
        }
        nt = std::min(nt, kMaxTail);
        while (nt && uint64_t(nt) * op->G > kMaxTailSlots) --nt;
        op->ntail = nt;
        op->ttz.assign(uint64_t(nt) * op->G, 0);
        op->ttc.assign(2 * uint64_t(nt) * op->G, 0.0);
        for (uint64_t g = 0; g < op->G; ++g) {
            const uint32_t t0 = op->gterm[g], n = op->gterm[g + 1] - t0;
            for (uint32_t u = 0; u < nt && u + 2 < n; ++u) {
                const uint64_t slot = uint64_t(u) * op->G + g;
                op->ttz[slot] = op->tz[t0 + 2 + u];
                op->ttc[2 * slot] = op->tc[2 * (t0 + 2 + u)];
                op->ttc[2 * slot + 1] = op->tc[2 * (t0 + 2 + u) + 1];
            }
        }
    }
}

}  // namespace qr

using namespace qr;

extern "C" {

const char *qr_last_error(void) { return g_last_error.c_str(); }

int qr_abi_version(void) { return QRHIP_ABI_VERSION; }

int qr_device_alloc(uint64_t bytes, void **d_out) {
    if (!d_out) return fail(QR_ERR_ARG, "null argument");
    *d_out = nullptr;
    if (bytes == 0) return QR_OK;
    const hipError_t e = hipMalloc(d_out, bytes);
    if (e == hipErrorOutOfMemory) return fail(QR_ERR_NOMEM, "device out of memory");
    if (e != hipSuccess) return hip_fail(e, "hipMalloc");
    return QR_OK;
}

int qr_device_free(void *d_ptr) {
    if (d_ptr) QR_HIP_CHECK(hipFree(d_ptr));
    return QR_OK;
}

int qr_copy_to_device(void *d_dst, const void *src, uint64_t bytes, void *stream) {
    if (bytes == 0) return QR_OK;
    if (!d_dst || !src) return fail(QR_ERR_ARG, "null argument");
    QR_HIP_CHECK(hipMemcpyAsync(d_dst, src, bytes, hipMemcpyHostToDevice, (hipStream_t)stream));
    return QR_OK;
}

int qr_copy_to_host(void *dst, const void *d_src, uint64_t bytes, void *stream) {
    if (bytes == 0) return QR_OK;
    if (!dst || !d_src) return fail(QR_ERR_ARG, "null argument");
    QR_HIP_CHECK(hipMemcpyAsync(dst, d_src, bytes, hipMemcpyDeviceToHost, (hipStream_t)stream));
    QR_HIP_CHECK(hipStreamSynchronize((hipStream_t)stream));
    return QR_OK;
}

int qr_pauli_parse(const char *label, uint32_t *num_qubits, uint32_t *base_phase,
                   uint32_t *phase, uint64_t *x_mask, uint64_t *z_mask) {
    uint32_t nq, bp, ny;
    uint64_t x, z;
    int rc = parse_label(label, &nq, &bp, &ny, &x, &z);
    if (rc) return rc;
    if (num_qubits) *num_qubits = nq;
    if (base_phase) *base_phase = bp;
    if (phase) *phase = (bp + ny) % 4;
    if (x_mask) *x_mask = x;
    if (z_mask) *z_mask = z;
    return QR_OK;
}

int qr_op_create(const char *const *labels, const double *coeffs, uint64_t num_terms,
                 int32_t phase_convention, qr_op **out) {
#pragma clang fp contract(off)
    if (!out) return fail(QR_ERR_ARG, "null output pointer");
    *out = nullptr;
    if (num_terms == 0)
        return fail(QR_ERR_TERMS, "SparsePauliOp::new: at least one pauli must be supplied");
    if (!labels || !coeffs) return fail(QR_ERR_ARG, "null labels or coefficients");
    if (phase_convention != QR_PHASE_ROWWISE && phase_convention != QR_PHASE_KRON)
        return fail(QR_ERR_ARG, "unknown phase convention");
    if (num_terms > 0xFFFFFFF0ull) return fail(QR_ERR_SIZE, "too many terms");
    qr_op *op = new (std::nothrow) qr_op;
    if (!op) return fail(QR_ERR_NOMEM, "out of host memory");
    const uint64_t T = num_terms;
    op->T = T;
    op->x.resize(T);
    op->z.resize(T);
    op->cp.resize(2 * T);
    // M[p] of accel.rs:147-152, multiplied as num-complex does:
    // (a.re*b.re - a.im*b.im, a.re*b.im + a.im*b.re) with a = M[p], b = c.
    static const double M[4][2] = {{1.0, 0.0}, {0.0, -1.0}, {-1.0, 0.0}, {0.0, 1.0}};
    for (uint64_t t = 0; t < T; ++t) {
        uint32_t nq, bp, ny;
        int rc = parse_label(labels[t], &nq, &bp, &ny, &op->x[t], &op->z[t]);
        if (rc) { delete op; return rc; }
        if (t == 0) op->nq = nq;
        else if (nq != op->nq) {
            delete op;
            return fail(QR_ERR_TERMS,
                        "SparsePauliOp::new: all supplied paulis must have the same #qubits");
        }
        uint32_t p = phase_convention == QR_PHASE_ROWWISE ? (bp + ny) % 4 : (ny + 4 - bp) % 4;
        op->cp[2 * t] = M[p][0] * coeffs[2 * t] - M[p][1] * coeffs[2 * t + 1];
        op->cp[2 * t + 1] = M[p][0] * coeffs[2 * t + 1] + M[p][1] * coeffs[2 * t];
    }
    // group by x, input order inside a group
    std::vector<std::pair<uint64_t, uint32_t>> order(T);
    for (uint64_t t = 0; t < T; ++t) order[t] = {op->x[t], uint32_t(t)};
    std::sort(order.begin(), order.end());
    op->tz.resize(T);
    op->tc.resize(2 * T);
    for (uint64_t i = 0; i < T; ++i) {
        const uint32_t t = order[i].second;
        if (i == 0 || op->x[t] != op->gx.back()) {
            op->gx.push_back(op->x[t]);
            op->gterm.push_back(uint32_t(i));
        }
        op->tz[i] = op->z[t];
        op->tc[2 * i] = op->cp[2 * t];
        op->tc[2 * i + 1] = op->cp[2 * t + 1];
    }
    op->gterm.push_back(uint32_t(T));
    op->G = op->gx.size();
    op->gkind.resize(op->G);
    for (uint64_t g = 0; g < op->G; ++g) {
        bool real = true, imag = true;
        for (uint32_t i = op->gterm[g]; i < op->gterm[g + 1]; ++i) {
            if (op->tc[2 * i + 1] != 0.0) real = false;
            if (op->tc[2 * i] != 0.0) imag = false;
        }
        op->gkind[g] = real ? 1 : (imag ? 2 : 0);
    }
    build_rank_lists(op->gx, op->rl_ptr, op->rl);
    finish_op(op);
    *out = op;
    return QR_OK;
}

int qr_op_create_device(const char *const *labels, const double *coeffs, uint64_t num_terms,
                        int32_t phase_convention, void *stream, qr_op **out) {
    if (!out) return fail(QR_ERR_ARG, "null output pointer");
    *out = nullptr;
    if (num_terms == 0)
        return fail(QR_ERR_TERMS, "SparsePauliOp::new: at least one pauli must be supplied");
    if (!labels || !coeffs) return fail(QR_ERR_ARG, "null labels or coefficients");
    if (phase_convention != QR_PHASE_ROWWISE && phase_convention != QR_PHASE_KRON)
        return fail(QR_ERR_ARG, "unknown phase convention");
    if (num_terms > 0xFFFFFFF0ull) return fail(QR_ERR_SIZE, "too many terms");
    return group_terms_device(labels, coeffs, num_terms, phase_convention, (hipStream_t)stream, out);
}

int qr_op_tables(const qr_op *op, uint64_t *gx, uint32_t *gterm, uint64_t *tz, double *tc,
                 uint8_t *gkind, uint32_t *rl_ptr, int32_t *rl, uint64_t *num_rank_entries) {
    if (!op) return fail(QR_ERR_ARG, "null operator");
    if (gx) std::copy(op->gx.begin(), op->gx.end(), gx);
    if (gterm) std::copy(op->gterm.begin(), op->gterm.end(), gterm);
    if (tz) std::copy(op->tz.begin(), op->tz.end(), tz);
    if (tc) std::copy(op->tc.begin(), op->tc.end(), tc);
    if (gkind) std::copy(op->gkind.begin(), op->gkind.end(), gkind);
    if (rl_ptr) std::copy(op->rl_ptr.begin(), op->rl_ptr.end(), rl_ptr);
    if (rl)
        for (size_t e = 0; e < op->rl.size(); ++e) {
            rl[2 * e] = op->rl[e].bit;
            rl[2 * e + 1] = op->rl[e].sigma;
        }
    if (num_rank_entries) *num_rank_entries = op->rl.size();
    return QR_OK;
}

int qr_op_destroy(qr_op *op) {
    if (!op) return QR_OK;
    int cur = 0;
    bool have = hipGetDevice(&cur) == hipSuccess;
    for (int d = 0; d < kMaxDevices; ++d) {
        if (!op->dev[d].ready && !op->dev[d].gx) continue;
        if (hipSetDevice(d) == hipSuccess) free_tables(op->dev[d]);
    }
    if (have) (void)hipSetDevice(cur);
    delete op;
    return QR_OK;
}

int qr_op_info(const qr_op *op, uint32_t *num_qubits, uint64_t *num_terms, uint64_t *num_groups,
               uint64_t *nnz) {
    if (!op) return fail(QR_ERR_ARG, "null operator");
    if (num_qubits) *num_qubits = op->nq;
    if (num_terms) *num_terms = op->T;
    if (num_groups) *num_groups = op->G;
    if (nnz) {
        unsigned __int128 v = (unsigned __int128)op->G << op->nq;
        *nnz = (v >> 64) ? 0 : uint64_t(v);
    }
    return QR_OK;
}

int qr_op_terms(const qr_op *op, uint64_t *x, uint64_t *z, double *coeff) {
    if (!op) return fail(QR_ERR_ARG, "null operator");
    if (x) std::memcpy(x, op->x.data(), op->T * sizeof(uint64_t));
    if (z) std::memcpy(z, op->z.data(), op->T * sizeof(uint64_t));
    if (coeff) std::memcpy(coeff, op->cp.data(), 2 * op->T * sizeof(double));
    return QR_OK;
}

int qr_op_row_layout(const qr_op *op, uint64_t row, uint64_t *cols, uint32_t *groups) {
    if (!op) return fail(QR_ERR_ARG, "null operator");
    if (op->nq < 64 && (row >> op->nq) != 0) return fail(QR_ERR_ARG, "row out of range");
    for (uint64_t j = 0; j < op->G; ++j) {
        int64_t rank = int64_t(j);
        for (uint32_t e = op->rl_ptr[j]; e < op->rl_ptr[j + 1]; ++e)
            if ((row >> op->rl[e].bit) & 1) rank += op->rl[e].sigma;
        if (rank < 0 || uint64_t(rank) >= op->G)
            return fail(QR_ERR_ARG, "internal error: rank out of range");
        if (cols) cols[rank] = row ^ op->gx[j];
        if (groups) groups[rank] = uint32_t(j);
    }
    return QR_OK;
}

int qr_mode_parse(const char *mode, int32_t *kind, uint64_t *step, int32_t *phase_convention) {
    if (!mode) return fail(QR_ERR_ARG, "null mode");
    std::string m(mode);
    int32_t k = -1;
    uint64_t st = 0;
    auto find_step = [&](const char *key) -> int {
        // unanchored search like Regex::is_match(r"<key>/(\d+)") (lib.rs:283-288)
        size_t klen = std::strlen(key);
        for (size_t pos = m.find(key); pos != std::string::npos; pos = m.find(key, pos + 1)) {
            size_t d = pos + klen;
            if (d < m.size() && m[d] == '/' && d + 1 < m.size() && m[d + 1] >= '0' && m[d + 1] <= '9') {
                uint64_t v = 0;
                bool overflow = false;
                for (size_t i = d + 1; i < m.size() && m[i] >= '0' && m[i] <= '9'; ++i) {
                    if (v > (UINT64_MAX - 9) / 10) overflow = true;
                    v = v * 10 + uint64_t(m[i] - '0');
                }
                st = overflow ? 0 : v;
                return 1;
            }
        }
        return 0;
    };
    if (m.empty()) k = QR_MODE_DEFAULT;
    else if (m == "Binary") k = QR_MODE_BINARY;
    else if (m == "Accel") k = QR_MODE_ACCEL;
    else if (m == "Rowwise") k = QR_MODE_ROWWISE;
    else if (m == "RowwiseUnsafe") k = QR_MODE_ROWWISE_UNSAFE;
    else if (find_step("RowwiseUnsafeChunked")) k = QR_MODE_ROWWISE_UNSAFE_CHUNKED;
    else if (m == "Reduce") k = QR_MODE_REDUCE;
    else if (m == "Rayon") k = QR_MODE_RAYON;
    else if (find_step("RayonChunked")) k = QR_MODE_RAYON_CHUNKED;
    else if (m == "Hip") k = QR_MODE_HIP;
    if (k < 0) return fail(QR_ERR_MODE, "to_matrix_mode: unrecognized mode " + m);
    if ((k == QR_MODE_ROWWISE_UNSAFE_CHUNKED || k == QR_MODE_RAYON_CHUNKED) && st == 0)
        return fail(QR_ERR_MODE, "to_matrix_mode: chunk size must be a positive integer in " + m);
    if (kind) *kind = k;
    if (step) *step = st;
    if (phase_convention) {
        bool kron = (k == QR_MODE_DEFAULT || k == QR_MODE_BINARY || k == QR_MODE_REDUCE ||
                     k == QR_MODE_RAYON);
        *phase_convention = kron ? QR_PHASE_KRON : QR_PHASE_ROWWISE;
    }
    return QR_OK;
}

int qr_csr_build(const qr_op *op, uint64_t *d_indptr, uint64_t *d_indices, double *d_data,
                 void *stream) {
    if (!op || !d_indptr || !d_indices || !d_data) return fail(QR_ERR_ARG, "null argument");
    if (op->nq > 40) return fail(QR_ERR_SIZE, "CSR of more than 40 qubits is not supported");
    DeviceTables *t;
    int rc = device_tables(op, &t, false, /*with_words=*/true);
    if (rc) return rc;
    return launch_csr_build(op, t, 0, uint64_t(1) << op->nq, d_indptr, d_indices, d_data,
                            (hipStream_t)stream);
}

int qr_csr_build_rows(const qr_op *op, uint64_t row_begin, uint64_t row_end, uint64_t *d_indices,
                      double *d_data, void *stream) {
    if (!op || !d_indices || !d_data) return fail(QR_ERR_ARG, "null argument");
    if (op->nq > 40) return fail(QR_ERR_SIZE, "CSR of more than 40 qubits is not supported");
    if (row_end < row_begin || row_end > (uint64_t(1) << op->nq))
        return fail(QR_ERR_ARG, "row range out of bounds");
    if (row_end == row_begin) return QR_OK;
    DeviceTables *t;
    int rc = device_tables(op, &t, false, /*with_words=*/true);
    if (rc) return rc;
    return launch_csr_build(op, t, row_begin, row_end, nullptr, d_indices, d_data,
                            (hipStream_t)stream);
}

int qr_csr_matvec(uint64_t nrows, uint64_t ncols, uint64_t nnz, const uint64_t *d_indptr,
                  const uint64_t *d_indices, const double *d_data, const double *d_x, double *d_y,
                  void *stream) {
    if (nrows == 0) return QR_OK;
    if (!d_indptr || !d_y) return fail(QR_ERR_ARG, "null argument");
    if (nnz != 0 && (!d_indices || !d_data || !d_x || ncols == 0))
        return fail(QR_ERR_ARG, "null argument");
    return launch_csr_matvec(nrows, ncols, nnz, d_indptr, d_indices, d_data, d_x, d_y,
                             (hipStream_t)stream);
}

int qr_csr_diagonal(uint64_t nrows, uint64_t ncols, uint64_t nnz, const uint64_t *d_indptr,
                    const uint64_t *d_indices, const double *d_data, double *d_out, void *stream) {
    if (nrows == 0 || ncols == 0) return QR_OK;
    if (!d_indptr || !d_out || (nnz && (!d_indices || !d_data)))
        return fail(QR_ERR_ARG, "null argument");
    return launch_csr_diagonal(nrows, ncols, nnz, d_indptr, d_indices, d_data, d_out,
                               (hipStream_t)stream);
}

int qr_axpby(uint64_t n, const double *a, const double *d_x, const double *b, const double *d_y,
             double *d_z, void *stream) {
    if (!a || !b || (n && (!d_x || !d_y || !d_z))) return fail(QR_ERR_ARG, "null argument");
    return launch_axpby(n, 0, a, d_x, b, d_y, d_z, (hipStream_t)stream);
}

int qr_axpy(uint64_t n, const double *a, const double *d_x, const double *d_y, double *d_z,
            void *stream) {
    if (!a || (n && (!d_x || !d_y || !d_z))) return fail(QR_ERR_ARG, "null argument");
    return launch_axpby(n, 1, a, d_x, nullptr, d_y, d_z, (hipStream_t)stream);
}

int qr_ax(uint64_t n, const double *a, const double *d_x, double *d_z, void *stream) {
    if (!a || (n && (!d_x || !d_z))) return fail(QR_ERR_ARG, "null argument");
    return launch_axpby(n, 2, a, d_x, nullptr, nullptr, d_z, (hipStream_t)stream);
}

int qr_precond(uint64_t nrows, uint64_t ncols, uint64_t nnz, const uint64_t *d_indptr,
               const uint64_t *d_indices, const double *d_data, const double *d_dx,
               const double *e, double tol, double *d_out, void *stream) {
    const uint64_t n = nrows < ncols ? nrows : ncols;
    if (!e || (n && (!d_indptr || !d_dx || !d_out || (nnz && (!d_indices || !d_data)))))
        return fail(QR_ERR_ARG, "null argument");
    return launch_precond(n, nullptr, nnz, d_indptr, d_indices, d_data, d_dx, e, tol, d_out,
                          (hipStream_t)stream);
}

int qr_precond2(uint64_t n, const double *d_diag, const double *d_dx, const double *e, double tol,
                double *d_out, void *stream) {
    if (!e || (n && (!d_diag || !d_dx || !d_out))) return fail(QR_ERR_ARG, "null argument");
    return launch_precond(n, d_diag, 0, nullptr, nullptr, nullptr, d_dx, e, tol, d_out,
                          (hipStream_t)stream);
}

int qr_csr_add_count(uint64_t nrows, const double *a, uint64_t nnz1, const uint64_t *d_indptr1,
                     const uint64_t *d_indices1, const double *d_data1, const double *b,
                     uint64_t nnz2, const uint64_t *d_indptr2, const uint64_t *d_indices2,
                     const double *d_data2, uint64_t *d_indptr_out, uint64_t *nnz_out,
                     void *stream) {
    if (!a || !b || !nnz_out || !d_indptr_out) return fail(QR_ERR_ARG, "null argument");
    *nnz_out = 0;
    if (nrows == 0) {
        QR_HIP_CHECK(hipMemsetAsync(d_indptr_out, 0, sizeof(uint64_t), (hipStream_t)stream));
        return QR_OK;
    }
    if (!d_indptr1 || !d_indptr2 || (nnz1 && (!d_indices1 || !d_data1)) ||
        (nnz2 && (!d_indices2 || !d_data2)))
        return fail(QR_ERR_ARG, "null argument");
    return launch_spadd_count(nrows, a, nnz1, d_indptr1, d_indices1, d_data1, b, nnz2, d_indptr2,
                              d_indices2, d_data2, d_indptr_out, nnz_out, (hipStream_t)stream);
}

int qr_csr_add_fill(uint64_t nrows, const double *a, uint64_t nnz1, const uint64_t *d_indptr1,
                    const uint64_t *d_indices1, const double *d_data1, const double *b,
                    uint64_t nnz2, const uint64_t *d_indptr2, const uint64_t *d_indices2,
                    const double *d_data2, const uint64_t *d_indptr_out, uint64_t *d_indices_out,
                    double *d_data_out, void *stream) {
    if (!a || !b || !d_indptr_out) return fail(QR_ERR_ARG, "null argument");
    if (nrows == 0) return QR_OK;
    if (!d_indptr1 || !d_indptr2 || (nnz1 && (!d_indices1 || !d_data1)) ||
        (nnz2 && (!d_indices2 || !d_data2)))
        return fail(QR_ERR_ARG, "null argument");
    return launch_spadd_fill(nrows, a, nnz1, d_indptr1, d_indices1, d_data1, b, nnz2, d_indptr2,
                             d_indices2, d_data2, d_indptr_out, d_indices_out, d_data_out,
                             (hipStream_t)stream);
}

int qr_csr_count_zeros(uint64_t nnz, const double *d_data, double tol, uint64_t *count,
                       void *stream) {
    if (!count || (nnz && !d_data)) return fail(QR_ERR_ARG, "null argument");
    return launch_count_zeros(nnz, d_data, tol, count, (hipStream_t)stream);
}

int qr_csr_eliminate_zeros(uint64_t nrows, uint64_t nnz, const uint64_t *d_indptr,
                           const uint64_t *d_indices, const double *d_data, double tol,
                           uint64_t *d_indptr_out, uint64_t *d_indices_out, double *d_data_out,
                           uint64_t *nnz_out, void *stream) {
    if (!nnz_out || !d_indptr || !d_indptr_out ||
        (nnz && (!d_indices || !d_data || !d_indices_out || !d_data_out)))
        return fail(QR_ERR_ARG, "null argument");
    *nnz_out = 0;
    return launch_eliminate_zeros(nrows, nnz, d_indptr, d_indices, d_data, tol, d_indptr_out,
                                  d_indices_out, d_data_out, nnz_out, (hipStream_t)stream);
}

int qr_csr_write_raw(const char *path, uint64_t rows, uint64_t cols, uint64_t nnz,
                     const uint64_t *d_indptr, const uint64_t *d_indices, const double *d_data,
                     void *stream) {
    if (!path || !d_indptr || (nnz && (!d_indices || !d_data))) return fail(QR_ERR_ARG, "null argument");
    return io_write_raw(path, rows, cols, nnz, d_indptr, d_indices, d_data, (hipStream_t)stream);
}

int qr_csr_read_raw_info(const char *path, uint64_t *rows, uint64_t *cols, uint64_t *nnz) {
    if (!path || !rows || !cols || !nnz) return fail(QR_ERR_ARG, "null argument");
    return io_read_raw_info(path, rows, cols, nnz);
}

int qr_csr_read_raw(const char *path, uint64_t rows, uint64_t nnz, uint64_t *d_indptr,
                    uint64_t *d_indices, double *d_data, void *stream) {
    if (!path || !d_indptr || (nnz && (!d_indices || !d_data))) return fail(QR_ERR_ARG, "null argument");
    return io_read_raw(path, rows, nnz, d_indptr, d_indices, d_data, (hipStream_t)stream);
}

int qr_csr_write_mm(const char *path, uint64_t rows, uint64_t cols, uint64_t nnz,
                    const uint64_t *d_indptr, const uint64_t *d_indices, const double *d_data,
                    int32_t symmetry, void *stream) {
    if (!path || !d_indptr || (nnz && (!d_indices || !d_data))) return fail(QR_ERR_ARG, "null argument");
    return io_write_mm(path, rows, cols, nnz, d_indptr, d_indices, d_data, symmetry,
                       (hipStream_t)stream);
}

int qr_mm_read_open(const char *path, qr_mm_reader **out, uint64_t *rows, uint64_t *cols,
                    uint64_t *nnz, void *stream) {
    if (!path || !out || !rows || !cols || !nnz) return fail(QR_ERR_ARG, "null argument");
    *out = nullptr;
    const int rc = io_read_mm(path, out, (hipStream_t)stream);
    if (rc != QR_OK) return rc;
    *rows = (*out)->rows;
    *cols = (*out)->cols;
    *nnz = (*out)->nnz;
    return QR_OK;
}

int qr_mm_read_take(const qr_mm_reader *r, uint64_t *d_indptr, uint64_t *d_indices, double *d_data,
                    void *stream) {
    if (!r || !d_indptr || (r->nnz && (!d_indices || !d_data))) return fail(QR_ERR_ARG, "null argument");
    hipStream_t s = (hipStream_t)stream;
    QR_HIP_CHECK(hipMemcpyAsync(d_indptr, r->indptr, (r->rows + 1) * 8, hipMemcpyDeviceToDevice, s));
    if (r->nnz) {
        QR_HIP_CHECK(hipMemcpyAsync(d_indices, r->indices, r->nnz * 8, hipMemcpyDeviceToDevice, s));
        QR_HIP_CHECK(hipMemcpyAsync(d_data, r->data, r->nnz * 16, hipMemcpyDeviceToDevice, s));
    }
    QR_HIP_CHECK(hipStreamSynchronize(s));
    return QR_OK;
}

int qr_mm_read_close(qr_mm_reader *r) {
    delete r;
    return QR_OK;
}

static int apply_args(const qr_op *op, int32_t precision, uint32_t nvec, const void *d_x,
                      void *d_y, double *d_expect) {
    if (!op || !d_x || (!d_y && !d_expect)) return fail(QR_ERR_ARG, "null argument");
    if (precision != QR_PREC_FP64 && precision != QR_PREC_MIXED)
        return fail(QR_ERR_ARG, "unknown precision");
    if (nvec == 0) return QR_OK;
    if (op->nq > 36) return fail(QR_ERR_SIZE, "states of more than 36 qubits are not supported");
    if (d_y) {
        // y is written while other blocks still gather x: no overlap allowed
        const uint64_t bytes = uint64_t(nvec) << (op->nq + (precision == QR_PREC_MIXED ? 3 : 4));
        const uintptr_t x0 = uintptr_t(d_x), y0 = uintptr_t(d_y);
        if (x0 < y0 + bytes && y0 < x0 + bytes)
            return fail(QR_ERR_ARG, "apply: y overlaps x (the apply is not in place)");
    }
    return QR_OK;
}

int qr_pauli_apply(const qr_op *op, int32_t precision, uint32_t nvec, const void *d_x, void *d_y,
                   double *d_expect, void *stream) {
    int rc = apply_args(op, precision, nvec, d_x, d_y, d_expect);
    if (rc || nvec == 0) return rc;
    DeviceTables *t;
    if ((rc = device_tables(op, &t))) return rc;
    return launch_pauli_apply(op, t, precision, nvec, d_x, d_y, d_expect, (hipStream_t)stream);
}

int qr_pauli_apply_noalloc(const qr_op *op, int32_t precision, uint32_t nvec, const void *d_x,
                           void *d_y, double *d_expect, void *stream) {
    int rc = apply_args(op, precision, nvec, d_x, d_y, d_expect);
    if (rc || nvec == 0) return rc;
    DeviceTables *t;
    if ((rc = device_tables(op, &t, /*noalloc=*/true))) return rc;
    return launch_pauli_apply(op, t, precision, nvec, d_x, d_y, d_expect, (hipStream_t)stream,
                              /*noalloc=*/true);
}

}  // extern "C"
