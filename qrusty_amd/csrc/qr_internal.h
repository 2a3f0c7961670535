// qr_internal.h -- shared declarations of libqrhip (host tables, launchers).
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/qrhip.h"

struct qr_op;

// a parsed MatrixMarket file: the CSR in device memory (qr_mm_read_open)
struct qr_mm_reader {
    uint64_t rows = 0, cols = 0, nnz = 0;
    uint64_t *indptr = nullptr, *indices = nullptr;  // device
    double *data = nullptr;                          // device, re/im pairs
    ~qr_mm_reader() {
        if (indptr) (void)hipFree(indptr);
        if (indices) (void)hipFree(indices);
        if (data) (void)hipFree(data);
    }
};

namespace qr {

// Sets the thread's last error and returns `code`.
int fail(int code, const std::string &msg);
int hip_fail(hipError_t e, const char *what);

#define QR_HIP_CHECK(call)                                      \
    do {                                                        \
        hipError_t qr_e_ = (call);                              \
        if (qr_e_ != hipSuccess) return ::qr::hip_fail(qr_e_, #call); \
    } while (0)

constexpr int kMaxDevices = 16;
// heavy groups the CSR build folds per row in a pass of their own: molecular
// Hamiltonians (the reference's H8..H12) have 17-111 groups of 22-301 terms
// next to groups of at most 6 (the sign-word builder's tiles hold all of them;
// of the shared tile builder, as many as the LDS holds, heavy_fit in qr_tile.h)
constexpr uint32_t kMaxHeavy = 128;
// Tail table of an operator with heavy groups: terms 2, 3, ... of every group
// transposed, slot u * G + g = term 2 + u of group g, for u < ntail <=
// kMaxTail and at most kMaxTailSlots slots (24 B each: at most 96 MiB per
// device; the builder reads the terms past the table from the grouped table)
constexpr uint32_t kMaxTail = 16;
constexpr uint64_t kMaxTailSlots = uint64_t(1) << 22;
constexpr uint32_t kSubMaxG = 2048;  // groups of one CSR-build sub-operator
constexpr uint32_t kWordMaxG = 1024;  // the same of the sign-word builder
constexpr uint32_t kWordHold = 6;     // terms of a group that it holds (real form)

// Row-ordering entry: while building row r, a group whose sorted-x position is j
// moves by `sigma` positions when bit `bit` of r is set (see build_rank_lists).
struct RankEntry {
    int32_t bit;
    int32_t sigma;
};

// Matrix-free apply: D_g(r) by table.  Inside a tile, D_g is a sum of
// "patterns" A_p (-1)^popcount(l & zl_p) (see build_patterns).  The patterns
// of a group are cut into parts whose zl span at most kPartRank dimensions:
// with a basis b_j of the part's zl, the part's sum depends on the row only
// through the index whose bit j is parity(l & b_j), so the block tabulates it
// once per tile (at most 16 values) and a row reads its value.  The index is
// linear in the bits of l, so it is the XOR of the indices of the thread bits
// 0-2 (nibble tid & 7 of w0), 3-5 (nibble of w1), of the wave (byte of w2)
// and of the row index k (byte of rc).  w2 and rc are scaled to bytes of the
// part's table, which starts at `tab` (in 4-byte units) of the block's LDS,
// aligned to its size.
constexpr int kPartRank = 4;
struct ApplyPart {
    uint32_t w0, w1, w2, tab;
    uint64_t rc;
};
// One (sub)group: its x mask and its first part, or, with more than one part
// (nparts > 1), the index of its parts in the part array in w0.  32 bytes,
// read with one scalar load.
struct ApplyGroup {
    uint64_t m;
    uint32_t w0, w1, w2;
    uint32_t tab_n;  // tab | nparts << 16 | flags
    uint64_t rc;
    __host__ __device__ uint32_t tab() const { return tab_n & 0xffffu; }
    __host__ __device__ uint32_t nparts() const { return (tab_n >> 16) & 0xfffu; }
};
constexpr uint32_t kGroupRowvar = 1u << 28;  // D varies with the row index: rc is not 0
constexpr uint32_t kGroupCplx = 1u << 29;    // a coefficient with an imaginary part
// The patterns of table i of the slot: entry 16 i + c is the term range of
// its pattern of code c (whose zl is the sum of the basis vectors in c), empty
// if it has none.  tab[i] is the table's place (4-byte units) | 2^rank << 16.
// Table entries are FP64, complex unless every coefficient of the operator
// (pass) is real.
struct ApplyRange {
    uint32_t t0, t1;
};

// Groups whose tables [t0, t1) are formed in LDS together.  Inside a chunk the
// groups are ordered by class -- bit 0 (the paired-row layout): row bit 0 of
// the mask set, so that the rows of a pair exchange partners; bit 1: the mask
// reaches outside the tile ("far") -- and class c holds the groups
// [cg[c], cg[c+1]).  Masks ascend: the near groups come first, while the
// neighbouring blocks load the tiles that the far ones read from L2 (24-qubit
// ring, complex64, 8 states: 1.47 ms, 1.77 the other way round).  For the
// partner-staged kernel the groups are ordered by partner tile instead, in
// runs [r0, r1), the tile itself last (28-qubit k-local 236 -> 226 ms, 20-qubit
// molecule 927 -> 891 us against the tile itself first).
constexpr int kApplyClasses = 4;
struct ApplyChunk {
    uint32_t cg[kApplyClasses + 1];
    uint32_t t0, t1;
    uint32_t r0, r1;
};

// Partner-staged apply: the groups of a chunk whose masks share the bits
// above the tile (`hi`, a row offset) gather from the same partner tile,
// which is loaded into LDS once for all of them: the groups up to g1.
struct ApplyRun {
    uint64_t hi;
    uint32_t g1, pad;
};

// Window pass of an FP64 apply: tiles of 2^L rows whose index bits are the
// state's bits [0, f) and [s, s + L - f).  The groups whose masks lie in those
// bits gather inside the tile there, where tiles of consecutive rows would
// read a partner tile each; y is added to.  s = 0: no window.
struct ApplyWindow {
    uint32_t f = 0, s = 0;
};
constexpr int kMaxWindows = 3;

constexpr int kApplySlots = 6;

// A term of a heavy group (masks of 32 bits): c' and z.
struct WordTerm {
    double re, im;
    uint32_t z, pad;
};

// A sub-operator of the sign-word builder: the g groups from s0, a subtree of
// the mask trie; the heavy ones' terms are word_terms[word_ptr[at + k] ..
// word_ptr[at + k + 1]), k < hcnt.  In row r its groups begin at position
// s0 + the sum of off[b] over the bits b of r.
struct WordLeaf {
    uint32_t s0, g, hcnt, at;
    int32_t off[32];
};

// A group: its x mask, its first term, its number of terms, and which of its
// sub-operator's heavy groups it is (-1: none).
struct WordGroup {
    uint32_t x, tf, n;
    int32_t heavy;
};

// Device copies of an operator's tables (one set per device that used it).
struct DeviceTables {
    bool ready = false;
    // what holds the arrays: one allocation, or (tables built on the device,
    // qr_group.hip) one for those uploaded and gx to gkind each their own
    void *mem = nullptr;
    bool apart = false;
    uint64_t *gx = nullptr;      // [G]   distinct x masks, ascending
    uint32_t *gterm = nullptr;   // [G+1] term range of each group
    uint64_t *tz = nullptr;      // [T]   z masks, grouped (term order inside a group)
    double2 *tc = nullptr;       // [T]   c', grouped
    uint32_t *rl_ptr = nullptr;  // [G+1]
    RankEntry *rl = nullptr;     // [E]
    uint8_t *gkind = nullptr;    // [G]   0 complex, 1 real, 2 imaginary coefficients
    uint32_t *heavy = nullptr;   // [nheavy] heavy groups (qr_op::heavy)
    uint32_t nheavy = 0;
    uint64_t *ttz = nullptr;     // [ntail * G] tail table (qr_op::ttz, ttc)
    double2 *ttc = nullptr;
    uint32_t ntail = 0;
    uint32_t *leaf_heavy = nullptr;  // qr_op::leaf_heavy
    // the sign-word builder's, from the first CSR build on (word_tables): in
    // `mem`, or in word_mem where another call made that one
    bool words = false;
    void *word_mem = nullptr;
    WordLeaf *word_leaves = nullptr;  // qr_op::word_leaves, word_groups, word_ptr, word_terms
    WordGroup *word_groups = nullptr;
    int32_t *word_rank = nullptr;  // [nq][G]: what bit b of r adds to the place of group g in its sub-operator
    uint32_t *word_ptr = nullptr;
    WordTerm *word_terms = nullptr;
    // matrix-free apply tables, one set per tile kind and form (slot =
    // 2 * kind + staged; kind 0: FP64, 1: complex64, 2: small complex64 tiles)
    // and pass (slot + kApplySlots * (k + 1): window pass k)
    struct Patterns {
        int L = -1;
        void *mem = nullptr;  // holds the arrays
        uint32_t nchunk = 0, nrun = 0, max_tab = 0;
        ApplyGroup *grp = nullptr;    // by chunk
        ApplyChunk *chunk = nullptr;  // [nchunk]
        ApplyRun *run = nullptr;      // [nrun] (staged form only)
        ApplyPart *part = nullptr;  // parts of the groups that have more than one
        uint32_t *tab = nullptr;    // every part's table, by chunk
        ApplyRange *pat = nullptr;  // [16 * tables] term range of each pattern
        uint64_t *ptz = nullptr;    // [T]   z masks in pattern order
        double2 *ptc = nullptr;     // [T]   c' in pattern order
        bool cplx = false;          // complex tables
        uint32_t nwin = 0;          // window passes after this one
        ApplyWindow win;            // (of a window pass)
    } pat[kApplySlots * (1 + kMaxWindows)];
};

// Host build of the apply tables for tile size L, tb thread-index bits, of
// the groups g with pass[g] == id (pass empty: all).  A
// chunk takes up to tcap bytes of tables; a group that needs more has a chunk
// of its own, and one of more than psplit patterns is split into several
// ApplyGroups with the same mask.  The table area starts at byte
// tab0 of the block's LDS.  `staged` orders each chunk by partner tile
// (ApplyRun) instead of by class.
struct PatternShape {
    int L, tb;
    uint32_t psplit, tcap, tab0;
    bool staged, pairs;
    ApplyWindow win;  // {}: tiles of consecutive rows
};
struct HostPatterns {
    std::vector<ApplyGroup> grp;
    std::vector<ApplyChunk> chunk;
    std::vector<ApplyPart> part;
    std::vector<uint32_t> tab;
    std::vector<ApplyRange> pat;
    std::vector<uint64_t> ptz;
    std::vector<double> ptc;  // 2 per term
    std::vector<ApplyRun> run;  // staged form only
    uint32_t max_tab = 0;
    bool cplx = false;
};
// Paired-row layout of the mixed gather form: thread t owns the row pairs
// (2t, 2t+1) + 2^(tb+1) j, so row-bit 0 counts with the row index (bit 0 of
// k) and row-bits 1..tb are the thread bits.  The patterns then hold z in
// that order: bits 1..tb moved down to 0..tb-1, bit 0 up to bit tb.
inline uint64_t pair_row_bits(uint64_t zl, int tb) {
    const uint64_t tmask = (uint64_t(1) << tb) - 1;
    return ((zl >> 1) & tmask) | ((zl & 1) << tb) | (zl & ~((tmask << 1) | 1));
}
void build_patterns(const qr_op *op, const PatternShape &shape, const std::vector<uint8_t> &pass, uint8_t id,
                    HostPatterns &out);
// The window passes of an operator: pass[g] = 0 for the groups of the pass
// over tiles of consecutive rows, k + 1 for those of wins[k] (see qr_api.cpp).
// Returns whether they hold most of the masks that reach past L2.
bool choose_windows(const qr_op *op, int L, std::vector<ApplyWindow> &wins,
                    std::vector<uint8_t> &pass);
// Whether slot `slot` holds the apply tables for tile size L.
bool tables_ready(const qr_op *op, const DeviceTables *t, int slot, int L);
// The tables of slot `slot` and of its window passes (win_shape.L = 0: none
// wanted).  With `noalloc` they must already be on the device (QR_ERR_ARG if
// not): nothing is allocated or uploaded.
int device_patterns(const qr_op *op, DeviceTables *t, int slot, const PatternShape &shape,
                    const PatternShape &win_shape, bool noalloc = false);

}  // namespace qr

struct qr_op {
    uint32_t nq = 0;
    uint64_t T = 0, G = 0;
    // make_params table, input order
    std::vector<uint64_t> x, z;
    std::vector<double> cp;  // 2*T
    // grouped tables (groups ascending by x; terms of a group in input order)
    std::vector<uint64_t> gx;
    std::vector<uint32_t> gterm;
    std::vector<uint64_t> tz;
    std::vector<double> tc;
    std::vector<uint8_t> gkind;
    std::vector<uint32_t> rl_ptr;
    std::vector<qr::RankEntry> rl;
    // groups with many more terms than the others (at most kMaxHeavy,
    // ascending): the CSR build folds them once per tile row, not per lane
    std::vector<uint32_t> heavy;
    // G > kSubMaxG: the mask trie cut into subtrees of at most kSubMaxG
    // groups [s0, s1) at depth `depth`; the CSR build runs one sub-operator
    // per subtree (qr_tile.h TileOp::gbase)
    struct SubLeaf {
        uint32_t s0, s1, depth;
        uint32_t hoff, hcnt;  // its heavy groups: leaf_heavy[hoff, hoff + hcnt)
    };
    std::vector<SubLeaf> leaves;
    std::vector<uint32_t> leaf_heavy;  // heavy groups of each leaf, leaf-local
    // the sign-word builder (k_csr_build_words; at most 32 qubits): its form,
    // real if every coefficient c' is and few groups have terms past
    // kWordHold; the whole operator or its sub-operators of at most kWordMaxG
    // groups, in the order of their place (word_joint: one launch builds them
    // all, launch_build_words) or those of at most 256, 512 and 1024 groups one
    // after another; every group, and the terms of the heavy ones
    bool word_real = false, word_joint = false;
    std::vector<qr::WordLeaf> word_leaves;
    std::vector<qr::WordGroup> word_groups;
    std::vector<uint32_t> word_ptr;
    std::vector<qr::WordTerm> word_terms;
    // operators with heavy groups: the terms past each group's second,
    // transposed (slot u * G + g holds term gterm[g] + 2 + u, zero where the
    // group is shorter), so that the lanes of a batch -- one group each --
    // read one contiguous run per term position instead of one line apiece
    uint32_t ntail = 0;
    std::vector<uint64_t> ttz;
    std::vector<double> ttc;  // 2 * ntail * G
    // the matrix-free apply's form by tile kind (apply_form in qr_apply.hip)
    // plus one, 0: not chosen yet
    mutable std::atomic<int> form[qr::kApplySlots / 2] = {};
    // device state
    mutable std::mutex mu;
    mutable qr::DeviceTables dev[qr::kMaxDevices];
};

namespace qr {

// An operator whose term tables are built on the current device
// (qr_group.hip): the same tables as qr_op_create's host path, and its device
// tables for this device already in place.  Synchronises the stream.
int group_terms_device(const char *const *labels, const double *coeffs, uint64_t T, int32_t conv,
                       hipStream_t s, qr_op **out);

// Sub-operators, heavy groups and tail table of an op whose grouped tables
// are set.
void finish_op(qr_op *op);
// Uploads the op's heavy groups and tail table (where it has them) into t;
// with_base, with_words: the grouped tables, the sign-word builder's as well.
int upload_tables(const qr_op *op, DeviceTables &t, bool with_base, bool with_words);
// Frees one device's tables of an op.
void free_tables(DeviceTables &t);

// Uploads the op's tables to the current device if needed; returns the tables.
// with_words: for a CSR build, whose own tables then come in the same copy.
int device_tables(const qr_op *op, DeviceTables **out, bool noalloc = false, bool with_words = false);
// The sign-word builder's tables (4 n bytes per group and more, which only it
// reads).  *have = false: they are not on the device and `s` is being captured,
// which allows no upload; the shared tile builder needs none of them.
int word_tables(const qr_op *op, DeviceTables *t, hipStream_t s, bool *have);

// Kernel launchers (qr_csr.hip, qr_apply.hip).
int launch_csr_indptr(const qr_op *op, uint64_t row_begin, uint64_t nrows, uint64_t *d_indptr, hipStream_t s);
int launch_csr_build(const qr_op *op, DeviceTables *t, uint64_t row_begin,
                     uint64_t row_end, uint64_t *d_indptr, uint64_t *d_indices,
                     double *d_data, hipStream_t s);
int launch_csr_matvec(uint64_t nrows, uint64_t ncols, uint64_t nnz, const uint64_t *d_indptr,
                      const uint64_t *d_indices, const double *d_data, const double *d_x,
                      double *d_y, hipStream_t s);
int launch_csr_diagonal(uint64_t nrows, uint64_t ncols, uint64_t nnz, const uint64_t *indptr,
                        const uint64_t *indices, const double *data, double *out, hipStream_t s);
int launch_axpby(uint64_t n, int mode, const double *a, const double *x, const double *b,
                 const double *y, double *z, hipStream_t s);
int launch_precond(uint64_t n, const double *diag, uint64_t nnz, const uint64_t *indptr,
                   const uint64_t *indices, const double *data, const double *dx, const double *e,
                   double tol, double *out, hipStream_t s);
int launch_spadd_count(uint64_t nrows, const double *a, uint64_t nnz1, const uint64_t *ip1,
                       const uint64_t *ix1, const double *d1, const double *b, uint64_t nnz2,
                       const uint64_t *ip2, const uint64_t *ix2, const double *d2, uint64_t *ipo,
                       uint64_t *nnz_out, hipStream_t s);
int launch_spadd_fill(uint64_t nrows, const double *a, uint64_t nnz1, const uint64_t *ip1,
                      const uint64_t *ix1, const double *d1, const double *b, uint64_t nnz2,
                      const uint64_t *ip2, const uint64_t *ix2, const double *d2,
                      const uint64_t *ipo, uint64_t *ixo, double *dout, hipStream_t s);
int launch_count_zeros(uint64_t nnz, const double *d, double tol, uint64_t *count, hipStream_t s);
int launch_eliminate_zeros(uint64_t nrows, uint64_t nnz, const uint64_t *ip, const uint64_t *ix,
                           const double *d, double tol, uint64_t *ipo, uint64_t *ixo, double *dout,
                           uint64_t *nnz_out, hipStream_t s);
int io_write_raw(const char *path, uint64_t rows, uint64_t cols, uint64_t nnz, const uint64_t *ip,
                 const uint64_t *ix, const double *d, hipStream_t s);
int io_read_raw_info(const char *path, uint64_t *rows, uint64_t *cols, uint64_t *nnz);
int io_read_raw(const char *path, uint64_t rows, uint64_t nnz, uint64_t *ip, uint64_t *ix, double *d,
                hipStream_t s);
int io_write_mm(const char *path, uint64_t rows, uint64_t cols, uint64_t nnz, const uint64_t *ip,
                const uint64_t *ix, const double *d, int sym, hipStream_t s);
int io_read_mm(const char *path, qr_mm_reader **out, hipStream_t s);
// the tables of an FP64 apply of the operator, so that a launch_pauli_apply
// without allocation finds them
int apply_tables(const qr_op *op, DeviceTables *t);
// The same apply of one state without <x|y>, its groups in apply_parts(op)
// shares (1: not in shares), given memory for as many states in d_sums.
uint32_t apply_parts(const qr_op *op);
int launch_apply_parts(const qr_op *op, DeviceTables *t, uint32_t parts, const void *d_x, void *d_y, void *d_sums,
                       hipStream_t s);
// noalloc: no device allocation -- the tables must be on the device already
// and the <x|y> block partials go to the file-scope scratch array (qr_apply.hip)
int launch_pauli_apply(const qr_op *op, DeviceTables *t, int32_t precision, uint32_t nvec,
                       const void *d_x, void *d_y, double *d_expect, hipStream_t s,
                       bool noalloc = false);

}  // namespace qr
