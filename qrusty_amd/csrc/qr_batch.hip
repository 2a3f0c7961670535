// qr_batch.hip -- many operators of uneven size: CSR builds plus one product
// each, captured in one hipGraph.
//
// The reference builds and applies operators one at a time
// (qrusty/src/lib.rs:573-585 then accel.rs:338-370).  Here the operators go to
// kBranches branches of one graph, each to the branch with the least work so
// far, so that launches that leave part of the chip idle, and the ends of
// large ones, run beside others.  An operator's CSR is written by the
// single-operator build (qr_csr.hip); small operators share the launches of
// k_batch.  CSR entries are bit-identical either way.  Two forms (a tuning
// choice):
//   fused  y = A x by the matrix-free apply of the same operator
//          (qr_apply.hip), which reads no CSR back and so needs none: 0.5 ps
//          per entry of a random 20-qubit operator, where reading the entry's
//          24 bytes takes 4; states of few tiles with the operator's groups
//          in shares (launch_apply_parts);
//   split  (needs every CSR) after the builds, one matvec pass (k_batch_mv)
//          over the written CSRs.
// Measured, 16 operators of 8 to 18 qubits and 10 to 5000 random terms (443e6
// entries, 10.6 GB written): one persistent build-and-apply kernel per
// register class 4850 us, this form 2370.  What bounds it: the CSR stores
// (1.65 ms at the builds' 6.4 TB/s), then the applies.
//
// Tuning knobs (qr_tuning): the order in which operators go to the branches
// (input order or largest first), the form, and, for k_batch and the matvec
// pass, tiles per item and resident blocks per CU.  qr_batch_tune times every
// candidate on the caller's buffers and keeps the fastest.
#include "qr_internal.h"
#include "qr_tile.h"

#include <algorithm>
#include <numeric>

namespace qr {

struct BatchOpDesc {
    TileOp op;
    uint64_t item_begin;  // first work item of this operator
    uint64_t tiles;       // row tiles of this operator
};

// Small operators (kBatchSmall): one persistent kernel for those of one group
// chunk per thread and one for those of two (at most 2048 groups), whose
// blocks take (operator, tiles) items from an atomic counter and build them
// with the shared tile builder (qr_tile.h); fused, with the same rows of
// y = A x from the entries still in registers.  No item depends on another,
// so every block leaves the loop as soon as the counter passes the end.
template <int kChunks, bool kMatvec>
__global__ __launch_bounds__(kStageThreads, !kMatvec && kChunks <= 1 ? 8 : 1) void k_batch(
    const BatchOpDesc *__restrict__ ops, uint32_t nops, uint64_t total_items, uint32_t tiles_per_item,
    unsigned long long *__restrict__ counter) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ unsigned long long item_s;
    for (;;) {
        if (threadIdx.x == 0) item_s = atomicAdd(counter, 1ull);
        __syncthreads();
        const uint64_t item = item_s;
        __syncthreads();
        if (item >= total_items) break;
        // operator owning the item: last k with item_begin <= item
        uint32_t lo = 0, hi = nops;
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) / 2;
            if (ops[mid].item_begin <= item) lo = mid;
            else hi = mid;
        }
        const BatchOpDesc &d = ops[lo];
        const uint64_t t0 = (item - d.item_begin) * tiles_per_item;
        const uint64_t t1 = t0 + tiles_per_item < d.tiles ? t0 + tiles_per_item : d.tiles;
        for (uint64_t t = t0; t < t1; ++t) {
            build_tile_staged<true, kChunks, kMatvec, kTilePlain>(d.op, t, smem_raw);
            __syncthreads();  // the stage is reused by the next tile
        }
    }
}

// Most groups of an operator whose y the fused form gives without CSR buffers (a
// limit of the interface: the apply has none).
constexpr uint64_t kBatchMostG = 6144;

// Entries up to which an operator is small: it runs in k_batch, which takes
// all of them in a launch or two, at 11 ps per entry fused, where a build and
// an apply of its own take two launches and 5.  Measured (us, 2^20 / 2^21 /
// 2^22 / 2^24): 64 operators of 8 to 14 qubits 442 / 460 / 495 / 560, 16 of
// 12 to 17 qubits 560 / 560 / 658 / 800, and the first run, which makes the
// apply's tables, 4 of 8 to 16 qubits 1240 / 710 / 470.
constexpr uint64_t kBatchSmall = uint64_t(1) << 21;

// Split form, second pass: y_k = A_k x_k from the CSR just written, over
// (operator, block of kMvRows rows) items taken from one counter.  Operators
// of at least kMvStagedMinRow groups run the row-staged walker of qr_mv.h
// (contiguous row streams, gathers of 8 neighbouring rows per instruction);
// shorter rows 8 lanes per row, a 256-thread block covering 32 consecutive
// rows per step, so that the gathers x[r ^ x_g] of neighbouring rows share
// cache lines.  Every row of a batch operator holds exactly G entries.  The
// arrays come from descriptors in memory, so they are read through pointers
// cast to the global address space (flat instructions otherwise).
struct BatchMvDesc {
    const uint64_t *indices;
    const double2 *data;
    const double2 *x;
    double2 *y;
    uint64_t rows, G, item_begin;
};
// 128 rows per item: the 256-operator uneven batch measured 100 ms per step
// at 1024 rows, 94-95 at 512, 93.6 at 256, 92.5-94 at 128, 93 at 64 and 32
// (smaller items leave less of a tail).
constexpr uint32_t kMvRows = 128;

// Rows [r0, r1) of one operator's y = A x, 8 lanes per row (rows of fewer
// than kMvStagedMinRow entries; plain loads, which beat nontemporal ones for
// short rows as in k_csr_matvec).
__device__ __forceinline__ void batch_mv_rows(const BatchMvDesc &d, uint64_t r0, uint64_t r1,
                                              uint32_t lane) {
    auto ld = [](const auto p) { return *p; };
    const auto indices = as_global(d.indices);
    const auto data = as_global(reinterpret_cast<const dvec2 *>(d.data));
    const auto x = as_global(reinterpret_cast<const dvec2 *>(d.x));
    const auto y = as_global(reinterpret_cast<dvec2 *>(d.y));
    for (uint64_t rb = r0; rb < r1; rb += 32) {
        const uint64_t row = rb + (threadIdx.x >> 3);
        double2 acc = make_double2(0.0, 0.0);
        if (row < r1) {
            const uint64_t k1 = (row + 1) * d.G;
            uint64_t k = row * d.G + lane;
            // full chunks of 64 entries for all 8 lanes of the row together
            for (; k - lane + 64 <= k1; k += 64) {
                uint64_t c[8];
                double2 a[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    c[u] = ld(indices + k + 8 * u);
                    const dvec2 av = ld(data + k + 8 * u);
                    a[u] = make_double2(av.x, av.y);
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const dvec2 xb = x[c[u]];
                    acc.x = fma(a[u].x, xb.x, acc.x);
                    acc.x = fma(-a[u].y, xb.y, acc.x);
                    acc.y = fma(a[u].x, xb.y, acc.y);
                    acc.y = fma(a[u].y, xb.x, acc.y);
                }
            }
            if (k < k1) {
                // the fewer than 8 entries left (all of a short row):
                // predicated, every load issued before the first is used
                uint64_t c[8];
                double2 a[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    c[u] = 0;
                    a[u] = make_double2(0.0, 0.0);
                    if (k + 8 * u < k1) {
                        c[u] = ld(indices + k + 8 * u);
                        const dvec2 av = ld(data + k + 8 * u);
                        a[u] = make_double2(av.x, av.y);
                    }
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    if (k + 8 * u < k1) {
                        const dvec2 xb = x[c[u]];
                        acc.x = fma(a[u].x, xb.x, acc.x);
                        acc.x = fma(-a[u].y, xb.y, acc.x);
                        acc.y = fma(a[u].x, xb.y, acc.y);
                        acc.y = fma(a[u].y, xb.x, acc.y);
                    }
                }
            }
        }
#pragma unroll
        for (int off = 4; off > 0; off /= 2) {
            acc.x += __shfl_xor(acc.x, off, 8);
            acc.y += __shfl_xor(acc.y, off, 8);
        }
        if (row < r1 && lane == 0) y[row] = dvec2{acc.x, acc.y};
    }
}

// dynamic LDS: the row-staged walker's regions for the block's 4 waves
constexpr size_t kBatchMvLds = 4 * MvStagedShape<kMvStagedChunk>::kWaveBytes;

// (3 waves per SIMD: the LDS of three blocks fills a CU)
__global__ __launch_bounds__(256, 3) void k_batch_mv(const BatchMvDesc *__restrict__ ops, uint32_t nops,
                                                  uint64_t total_items,
                                                  unsigned long long *__restrict__ counter) {
    using S = MvStagedShape<kMvStagedChunk>;
    extern __shared__ __align__(16) unsigned char mv_lds[];
    __shared__ unsigned long long item_s;
    const uint32_t lane = threadIdx.x & 7u;
    const uint32_t wave = threadIdx.x / 64;
    uint64_t *s_idx = reinterpret_cast<uint64_t *>(mv_lds + size_t(wave) * S::kWaveBytes);
    dvec2 *s_dat = reinterpret_cast<dvec2 *>(s_idx + S::kRows * S::kIdxStride);
    for (;;) {
        if (threadIdx.x == 0) item_s = atomicAdd(counter, 1ull);
        __syncthreads();
        const uint64_t item = item_s;
        __syncthreads();
        if (item >= total_items) break;
        uint32_t lo = 0, hi = nops;
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) / 2;
            if (ops[mid].item_begin <= item) lo = mid;
            else hi = mid;
        }
        const BatchMvDesc &d = ops[lo];
        const uint64_t r0 = (item - d.item_begin) * kMvRows;
        const uint64_t r1 = r0 + kMvRows < d.rows ? r0 + kMvRows : d.rows;
        if (d.G >= kMvStagedMinRow) {
            const uint64_t G = d.G;
            auto bounds = [G](uint64_t r, uint64_t *k0, uint64_t *len) {
                *k0 = r * G;
                *len = G;
            };
            for (uint64_t rb = r0; rb < r1; rb += 4 * S::kRows)
                mv_staged_rows<kMvStagedChunk>(rb + wave * S::kRows, r1, d.rows, bounds, d.indices,
                                               d.data, d.x, d.y, s_idx, s_dat, 0, 0);
        } else {
            batch_mv_rows(d, r0, r1, lane);
        }
    }
}

// graph-safe reset of the work counter (a kernel, not a memset node)
__global__ void k_zero_counter(unsigned long long *counter) { *counter = 0ull; }

}  // namespace qr

using namespace qr;

// (us, 4 / 8 / 16 branches: 16 operators of 8 to 18 qubits 2450 / 2370 / 2670,
// of 12 to 17 qubits 620 / 565 / 565; one branch 3170 and 930)
constexpr int kBranches = 8;

struct qr_batch {
    std::vector<const qr_op *> ops;
    int dev = -1;
    hipStream_t cap = nullptr;  // private capture stream (default priority)
    hipStream_t side[kBranches] = {};  // branches 1 on (0: the recording stream)
    hipEvent_t fork = nullptr, join[kBranches] = {};
    BatchOpDesc *d_desc = nullptr;
    size_t d_desc_cap = 0;
    BatchMvDesc *d_mv = nullptr;
    size_t d_mv_cap = 0;
    double *d_sums = nullptr;  // of the applies in shares (apply_parts), one after another
    size_t d_sums_cap = 0;
    unsigned long long *d_counter = nullptr;
    int ncu = 0;
    // graph of the last (buffers, tuning)
    bool have_graph = false;
    std::vector<uintptr_t> graph_key;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    bool have_tuned = false;
    qr_tuning tuned{};
};

namespace {

struct Plan {
    // small operators, by group chunks per thread (1 or 2), and their branch
    int small_branch = 0;
    std::vector<BatchOpDesc> small[2];
    uint64_t items[2] = {};
    size_t shmem[2] = {};
    std::vector<uint32_t> branch[kBranches];  // the others, in order
    std::vector<bool> csr;                    // whether operator k's CSR is built
    std::vector<size_t> sums_at;              // operator k's place in d_sums
    size_t sums = 0;                          // doubles there
    std::vector<BatchMvDesc> mv;              // split form: one per operator
    uint64_t mv_items = 0;
};

bool has_csr(uint64_t *const *d_indices, double *const *d_data, size_t k) {
    return d_indices && d_indices[k] && d_data && d_data[k];
}

int make_plan(qr_batch *b, uint64_t *const *d_indptr, uint64_t *const *d_indices,
              double *const *d_data, const double *const *d_x, double *const *d_y,
              const qr_tuning &tu, Plan &plan) {
    const uint32_t nops = uint32_t(b->ops.size());
    // the split form needs every operator's CSR
    for (uint32_t k = 0; tu.split && k < nops; ++k)
        if (!has_csr(d_indices, d_data, k))
            return fail(QR_ERR_ARG, "the split batch form needs CSR output buffers for every operator");
    std::vector<uint32_t> order(nops);
    std::iota(order.begin(), order.end(), 0u);
    if (tu.order == 1)  // largest operator first
        std::stable_sort(order.begin(), order.end(), [b](uint32_t a, uint32_t c) {
            return (b->ops[a]->G << b->ops[a]->nq) > (b->ops[c]->G << b->ops[c]->nq);
        });
    uint64_t load[kBranches] = {};
    plan.csr.resize(nops);
    plan.sums_at.resize(nops);
    for (uint32_t k : order) {
        const qr_op *op = b->ops[k];
        if (op->nq > 32) return fail(QR_ERR_SIZE, "batch operators are limited to 32 qubits");
        if (!d_x || !d_x[k] || !d_y || !d_y[k]) return fail(QR_ERR_ARG, "null state pointer in batch");
        const bool csr = plan.csr[k] = has_csr(d_indices, d_data, k);
        if (!tu.split && op->G > kBatchMostG && !(csr && d_indptr && d_indptr[k]))
            return fail(QR_ERR_ARG, "batch operators with more than 6144 distinct x masks "
                                    "need CSR output buffers");
        const uint64_t N = uint64_t(1) << op->nq;
        if (tu.split) {
            plan.mv.push_back(BatchMvDesc{d_indices[k], reinterpret_cast<double2 *>(d_data[k]),
                                          reinterpret_cast<const double2 *>(d_x[k]),
                                          reinterpret_cast<double2 *>(d_y[k]), N, op->G, plan.mv_items});
            plan.mv_items += (N + kMvRows - 1) / kMvRows;
        }
        if (N * op->G <= kBatchSmall && op->G <= kSubMaxG) {
            DeviceTables *t;
            if (int rc = device_tables(op, &t)) return rc;
            const uint32_t G = uint32_t(op->G), jw = stage_jw_log2(G), nch = (G + (1u << jw) - 1) >> jw;
            const uint32_t c = nch <= 1 ? 0 : 1;
            uint32_t dbuf = 0;
            plan.shmem[c] = std::max(plan.shmem[c], stage_bytes(G, jw, &dbuf));
            BatchOpDesc d{};
            d.op = TileOp{t->gx, t->gterm, t->tz, t->tc, t->rl_ptr, t->rl, csr ? d_indices[k] : nullptr,
                          csr ? reinterpret_cast<double2 *>(d_data[k]) : nullptr, d_indptr ? d_indptr[k] : nullptr,
                          reinterpret_cast<const double2 *>(d_x[k]), reinterpret_cast<double2 *>(d_y[k]), 0, N, G,
                          jw, nch, dbuf, nullptr, 0, 0, 0, G};
            d.tiles = ((N - 1) >> (10 - jw + 4)) + 1;
            d.item_begin = plan.items[c];
            plan.items[c] += (d.tiles + tu.tiles_per_item - 1) / tu.tiles_per_item;
            plan.small[c].push_back(d);
            continue;
        }
        // the branch with the least work: entries, and about what a launch of
        // next to none costs in them
        const int to = int(std::min_element(load, load + kBranches) - load);
        load[to] += N * op->G + (uint64_t(1) << 20);
        plan.branch[to].push_back(k);
        const uint32_t parts = tu.split ? 1 : apply_parts(op);
        plan.sums_at[k] = plan.sums;
        if (parts > 1) plan.sums += 2 * N * parts;
    }
    plan.small_branch = int(std::min_element(load, load + kBranches) - load);
    return QR_OK;
}

int record(qr_batch *b, const Plan &plan, const qr_tuning &tu, uint64_t *const *d_indptr,
           uint64_t *const *d_indices, double *const *d_data, const double *const *d_x,
           double *const *d_y, hipStream_t s) {
    int rc;
    QR_HIP_CHECK(hipEventRecord(b->fork, s));
    for (int i = 0; i < kBranches; ++i) {
        if (plan.branch[i].empty() && i != plan.small_branch) continue;
        const hipStream_t bs = i ? b->side[i] : s;
        if (i) QR_HIP_CHECK(hipStreamWaitEvent(bs, b->fork, 0));
        for (uint32_t k : plan.branch[i]) {
            const qr_op *op = b->ops[k];
            DeviceTables *t;
            if ((rc = device_tables(op, &t))) return rc;
            const uint64_t N = uint64_t(1) << op->nq;
            uint64_t *ip = d_indptr ? d_indptr[k] : nullptr;
            if (has_csr(d_indices, d_data, k))
                rc = launch_csr_build(op, t, 0, N, ip, d_indices[k], d_data[k], bs);
            else if (ip) rc = launch_csr_indptr(op, 0, N, ip, bs);
            const uint32_t parts = tu.split ? 1 : apply_parts(op);
            if (!rc && parts > 1)
                rc = launch_apply_parts(op, t, parts, d_x[k], d_y[k], b->d_sums + plan.sums_at[k], bs);
            else if (!rc && !tu.split)
                rc = launch_pauli_apply(op, t, QR_PREC_FP64, 1, d_x[k], d_y[k], nullptr, bs, true);
            if (rc) return rc;
        }
        for (int c = 0; i == plan.small_branch && c < 2; ++c) {
            if (plan.small[c].empty()) continue;
            const uint64_t grid = std::min<uint64_t>(uint64_t(b->ncu) * tu.blocks_per_cu, plan.items[c]);
            auto kern = c == 0 ? (tu.split ? k_batch<1, false> : k_batch<1, true>)
                               : (tu.split ? k_batch<2, false> : k_batch<2, true>);
            hipLaunchKernelGGL(k_zero_counter, dim3(1), dim3(1), 0, bs, b->d_counter + 1 + c);
            hipLaunchKernelGGL(kern, dim3(unsigned(grid)), dim3(kStageThreads), plan.shmem[c], bs,
                               b->d_desc + (c ? plan.small[0].size() : 0), uint32_t(plan.small[c].size()),
                               plan.items[c], tu.tiles_per_item, b->d_counter + 1 + c);
            QR_HIP_CHECK(hipGetLastError());
        }
        if (i) {
            QR_HIP_CHECK(hipEventRecord(b->join[i], bs));
            QR_HIP_CHECK(hipStreamWaitEvent(s, b->join[i], 0));
        }
    }
    if (tu.split && plan.mv_items) {
        // 8 resident 256-thread blocks per CU and slot
        const uint64_t grid = std::min<uint64_t>(uint64_t(b->ncu) * 8 * tu.blocks_per_cu, plan.mv_items);
        hipLaunchKernelGGL(k_zero_counter, dim3(1), dim3(1), 0, s, b->d_counter);
        hipLaunchKernelGGL(k_batch_mv, dim3(unsigned(grid)), dim3(256), kBatchMvLds, s, b->d_mv,
                           uint32_t(plan.mv.size()), plan.mv_items, b->d_counter);
        QR_HIP_CHECK(hipGetLastError());
    }
    return QR_OK;
}

void drop_graph(qr_batch *b) {
    if (b->exec) (void)hipGraphExecDestroy(b->exec);
    if (b->graph) (void)hipGraphDestroy(b->graph);
    b->exec = nullptr;
    b->graph = nullptr;
    b->have_graph = false;
}

// Everything that a recording must not do: streams, the operators' tables,
// the matvec pass's descriptors.
int prepare(qr_batch *b, const Plan &plan, const qr_tuning &tu) {
    int dev = 0, rc;
    QR_HIP_CHECK(hipGetDevice(&dev));
    if (b->dev != dev) {
        if (b->dev >= 0) return fail(QR_ERR_ARG, "a batch is bound to the device it first ran on");
        b->dev = dev;
        QR_HIP_CHECK(hipStreamCreateWithFlags(&b->cap, hipStreamNonBlocking));
        QR_HIP_CHECK(hipEventCreateWithFlags(&b->fork, hipEventDisableTiming));
        QR_HIP_CHECK(hipMalloc(&b->d_counter, 3 * sizeof(unsigned long long)));
        for (const void *kf : {reinterpret_cast<const void *>(k_batch<1, true>), reinterpret_cast<const void *>(k_batch<2, true>),
                               reinterpret_cast<const void *>(k_batch<1, false>), reinterpret_cast<const void *>(k_batch<2, false>)})
            QR_HIP_CHECK(hipFuncSetAttribute(kf, hipFuncAttributeMaxDynamicSharedMemorySize,
                                             int(stage_bytes(kSubMaxG, 10, nullptr))));
        QR_HIP_CHECK(hipDeviceGetAttribute(&b->ncu, hipDeviceAttributeMultiprocessorCount, dev));
    }
    for (int i = 0; i < kBranches; ++i) {
        const auto &branch = plan.branch[i];
        if (i && !b->join[i] && (!branch.empty() || i == plan.small_branch)) {
            QR_HIP_CHECK(hipStreamCreateWithFlags(&b->side[i], hipStreamNonBlocking));
            QR_HIP_CHECK(hipEventCreateWithFlags(&b->join[i], hipEventDisableTiming));
        }
        for (uint32_t k : branch) {
            DeviceTables *t;
            bool have;
            if ((rc = device_tables(b->ops[k], &t, false, plan.csr[k]))) return rc;
            if (plan.csr[k] && (rc = word_tables(b->ops[k], t, b->cap, &have))) return rc;
            if (!tu.split && (rc = apply_tables(b->ops[k], t))) return rc;
        }
    }
    const size_t nsmall = plan.small[0].size() + plan.small[1].size();
    // a previous graph or tuning pass may still run and read the descriptors; no
    // graph outlives them
    QR_HIP_CHECK(hipDeviceSynchronize());
    drop_graph(b);
    auto room = [](auto **d, size_t *cap, size_t n) {
        if (*cap >= n) return int(QR_OK);
        if (*d) (void)hipFree(*d);
        *d = nullptr;
        *cap = 0;
        QR_HIP_CHECK(hipMalloc(d, n * sizeof(**d)));
        *cap = n;
        return int(QR_OK);
    };
    if ((rc = room(&b->d_desc, &b->d_desc_cap, nsmall)) || (rc = room(&b->d_mv, &b->d_mv_cap, plan.mv.size())) ||
        (rc = room(&b->d_sums, &b->d_sums_cap, plan.sums)))
        return rc;
    for (size_t c = 0, at = 0; c < 2; at += plan.small[c++].size())
        if (!plan.small[c].empty())
            QR_HIP_CHECK(hipMemcpy(b->d_desc + at, plan.small[c].data(), plan.small[c].size() * sizeof(BatchOpDesc),
                                   hipMemcpyHostToDevice));
    if (!plan.mv.empty())
        QR_HIP_CHECK(hipMemcpy(b->d_mv, plan.mv.data(), plan.mv.size() * sizeof(BatchMvDesc),
                               hipMemcpyHostToDevice));
    return QR_OK;
}

std::vector<uintptr_t> key_of(const qr_batch *b, uint64_t *const *d_indptr,
                              uint64_t *const *d_indices, double *const *d_data,
                              const double *const *d_x, double *const *d_y, const qr_tuning &tu) {
    std::vector<uintptr_t> k;
    const size_t n = b->ops.size();
    k.reserve(5 * n + 3);
    for (size_t i = 0; i < n; ++i) {
        k.push_back(d_indptr ? uintptr_t(d_indptr[i]) : 0);
        k.push_back(d_indices ? uintptr_t(d_indices[i]) : 0);
        k.push_back(d_data ? uintptr_t(d_data[i]) : 0);
        k.push_back(uintptr_t(d_x[i]));
        k.push_back(uintptr_t(d_y[i]));
    }
    k.push_back(tu.tiles_per_item);
    k.push_back(tu.blocks_per_cu);
    k.push_back(tu.order);
    k.push_back(tu.split);
    return k;
}

const qr_tuning kDefaultTuning{1, 1, 1, 0};

}  // namespace

extern "C" {

int qr_batch_create(const qr_op *const *ops, uint32_t nops, qr_batch **out) {
    if (!out) return fail(QR_ERR_ARG, "null output pointer");
    *out = nullptr;
    if (!ops || nops == 0) return fail(QR_ERR_ARG, "empty batch");
    for (uint32_t k = 0; k < nops; ++k)
        if (!ops[k]) return fail(QR_ERR_ARG, "null operator in batch");
    qr_batch *b = new (std::nothrow) qr_batch;
    if (!b) return fail(QR_ERR_NOMEM, "out of host memory");
    b->ops.assign(ops, ops + nops);
    *out = b;
    return QR_OK;
}

int qr_batch_destroy(qr_batch *b) {
    if (!b) return QR_OK;
    drop_graph(b);
    if (b->d_desc) (void)hipFree(b->d_desc);
    if (b->d_mv) (void)hipFree(b->d_mv);
    if (b->d_sums) (void)hipFree(b->d_sums);
    if (b->d_counter) (void)hipFree(b->d_counter);
    for (int i = 1; i < kBranches; ++i) {
        if (b->side[i]) (void)hipStreamDestroy(b->side[i]);
        if (b->join[i]) (void)hipEventDestroy(b->join[i]);
    }
    if (b->fork) (void)hipEventDestroy(b->fork);
    if (b->cap) (void)hipStreamDestroy(b->cap);
    delete b;
    return QR_OK;
}

int qr_batch_run(qr_batch *b, uint64_t *const *d_indptr, uint64_t *const *d_indices,
                 double *const *d_data, const double *const *d_x, double *const *d_y,
                 const qr_tuning *tuning, void *stream) {
    if (!b || !d_x || !d_y) return fail(QR_ERR_ARG, "null argument");
    const qr_tuning tu = tuning ? *tuning : (b->have_tuned ? b->tuned : kDefaultTuning);
    if (tu.tiles_per_item == 0 || tu.tiles_per_item > 4096 || tu.blocks_per_cu == 0 ||
        tu.blocks_per_cu > 8 || tu.order > 1 || tu.split > 1)
        return fail(QR_ERR_ARG, "tuning out of range");
    hipStream_t s = (hipStream_t)stream;
    std::vector<uintptr_t> key = key_of(b, d_indptr, d_indices, d_data, d_x, d_y, tu);
    if (!(b->have_graph && key == b->graph_key)) {
        Plan plan;
        int rc = make_plan(b, d_indptr, d_indices, d_data, d_x, d_y, tu, plan);
        if (rc) return rc;
        rc = prepare(b, plan, tu);
        if (rc) return rc;
        QR_HIP_CHECK(hipStreamBeginCapture(b->cap, hipStreamCaptureModeThreadLocal));
        rc = record(b, plan, tu, d_indptr, d_indices, d_data, d_x, d_y, b->cap);
        hipGraph_t g = nullptr;
        hipError_t e = hipStreamEndCapture(b->cap, &g);
        if (rc) {
            if (g) (void)hipGraphDestroy(g);
            return rc;
        }
        if (e != hipSuccess) return hip_fail(e, "hipStreamEndCapture");
        b->graph = g;
        QR_HIP_CHECK(hipGraphInstantiate(&b->exec, b->graph, nullptr, nullptr, 0));
        b->have_graph = true;
        b->graph_key = key;
    }
    QR_HIP_CHECK(hipGraphLaunch(b->exec, s));
    return QR_OK;
}

int qr_batch_tune(qr_batch *b, uint64_t *const *d_indptr, uint64_t *const *d_indices,
                  double *const *d_data, const double *const *d_x, double *const *d_y,
                  qr_tuning *best, void *stream) {
    if (!b || !d_x || !d_y) return fail(QR_ERR_ARG, "null argument");
    hipStream_t s = (hipStream_t)stream;
    const uint32_t tpis[] = {1, 2, 4, 8};
    const uint32_t bpcs[] = {1, 2};
    const uint32_t orders[] = {0, 1};
    // the split form is a candidate only when every operator keeps its CSR
    bool can_split = d_indices && d_data;
    for (size_t k = 0; can_split && k < b->ops.size(); ++k)
        can_split = d_indices[k] && d_data[k];
    hipEvent_t e0, e1;
    QR_HIP_CHECK(hipEventCreate(&e0));
    QR_HIP_CHECK(hipEventCreate(&e1));
    float best_ms = -1.0f;
    qr_tuning bt = kDefaultTuning;
    int rc = QR_OK;
    for (uint32_t split = 0; split < (can_split ? 2u : 1u); ++split)
    for (uint32_t order : orders)
        for (uint32_t bpc : bpcs)
            for (uint32_t tpi : tpis) {
                const qr_tuning tu{tpi, bpc, order, split};
                Plan plan;
                if ((rc = make_plan(b, d_indptr, d_indices, d_data, d_x, d_y, tu, plan))) goto done;
                // without small operators the tiles per item reach no kernel, and
                // the blocks per CU the matvec pass alone
                if (plan.small[0].empty() && plan.small[1].empty() &&
                    (tpi != tpis[0] || (!split && bpc != bpcs[0])))
                    continue;
                if ((rc = prepare(b, plan, tu))) goto done;
                // one untimed pass (first touch), then one timed pass
                for (int rep = 0; rep < 2; ++rep) {
                    if (rep == 1 && hipEventRecord(e0, s) != hipSuccess) { rc = fail(QR_ERR_HIP, "event"); goto done; }
                    if ((rc = record(b, plan, tu, d_indptr, d_indices, d_data, d_x, d_y, s))) goto done;
                }
                if (hipEventRecord(e1, s) != hipSuccess || hipEventSynchronize(e1) != hipSuccess) {
                    rc = fail(QR_ERR_HIP, "event");
                    goto done;
                }
                float ms = 0.0f;
                (void)hipEventElapsedTime(&ms, e0, e1);
                if (best_ms < 0.0f || ms < best_ms) { best_ms = ms; bt = tu; }
            }
done:
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (rc) return rc;
    b->tuned = bt;
    b->have_tuned = true;
    if (best) *best = bt;
    return QR_OK;
}

}  // extern "C"
