// bruteforce_api.cpp -- coral_bruteforce_knn*: exact k nearest neighbours of a batch of
// queries among the index's resident vectors (kernels in bruteforce.hip, bruteforce_mfma.hip).
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstring>
#include <utility>
#include <vector>

#include "beam_search.h"
#include "bruteforce.h"
#include "graph_build.h"
#include "index_internal.h"

using coral::fail;

namespace {
constexpr int64_t kSegment = (int64_t)1 << 22;   // base points per pass
constexpr int64_t kBufferFloats = (int64_t)1 << 29;  // 2 GiB distance buffer

// the passes over the base: distances of a block of queries to a segment of the base into D, the k best of every row
// of D, and at the end the k best of the per-segment winners.  screen: approximate distances from the matrix cores
// (qn, bn: squared norms) instead of the reference-order ones.
int knn_passes(coral_index* idx, const float* d_queries, int32_t Q, int32_t k, int32_t have_delete, bool screen,
               float* d_qn, int metric_out, int32_t* d_ids, float* d_dists, hipStream_t stream) {
    const int64_t n = idx->n;
    int64_t seg = std::min(n, kSegment);
    int64_t nseg = (n + seg - 1) / seg;
    while (nseg * k > 8192) {  // the final merge sorts nseg*k keys in LDS
        seg *= 2;
        nseg = (n + seg - 1) / seg;
    }
    const int64_t ld = (seg + 3) & ~(int64_t)3;
    int64_t qc = std::max<int64_t>(128, (kBufferFloats / ld) & ~(int64_t)127);
    qc = std::min<int64_t>(qc, ((int64_t)Q + 127) & ~(int64_t)127);
    float* D = nullptr;
    unsigned long long* part = nullptr;
    int* redo = nullptr;
    void* d_split = nullptr;
    auto release = [&]() {
        (void)hipFree(d_split);
        (void)hipFree(D);
        (void)hipFree(part);
        (void)hipFree(redo);
    };
#define HIP_TRY_R(expr)                                                                  \
    do {                                                                                 \
        hipError_t e_ = (expr);                                                          \
        if (e_ != hipSuccess) {                                                          \
            release();                                                                   \
            return fail(e_ == hipErrorOutOfMemory ? CORAL_ERR_MEMORY : CORAL_ERR_DEVICE, \
                        "%s failed: %s", #expr, hipGetErrorString(e_));                  \
        }                                                                                \
    } while (0)
    HIP_TRY_R(hipMalloc(&D, (size_t)qc * ld * sizeof(float)));
    HIP_TRY_R(hipMalloc(&part, (size_t)Q * nseg * k * sizeof(unsigned long long)));
    HIP_TRY_R(hipMalloc(&redo, (size_t)qc * sizeof(int)));
    if (screen) HIP_TRY_R(hipMalloc(&d_split, coral::split_queries_bytes((int)qc, idx->dim, 3)));
    for (int64_t q0 = 0; q0 < Q; q0 += qc) {
        const int nq = (int)std::min<int64_t>(qc, Q - q0);
        if (screen)
            HIP_TRY_R(coral::launch_prepare_queries(d_queries + (size_t)q0 * idx->dim, nq, idx->dim, 3, d_qn + q0, nullptr, d_split,
                                                    nullptr, nullptr, stream));
        for (int64_t s = 0; s < nseg; ++s) {
            const int64_t b0 = s * seg, nb = std::min(seg, n - b0);
            const float* qp = d_queries + (size_t)q0 * idx->dim;
            const float* bp = idx->d_vec + (size_t)b0 * idx->dim;
            const uint32_t* del = have_delete ? idx->d_deleted : nullptr;
            if (screen)
                HIP_TRY_R(coral::launch_approx_tile(d_split, bp, nq, nb, idx->dim, idx->metric, 3, d_qn + q0, idx->d_bnorm + b0, del,
                                                    b0, D, ld, stream));
            else
                HIP_TRY_R(coral::launch_distance_tile(qp, bp, nq, nb, idx->dim, idx->metric, del, b0, D, ld, stream));
            HIP_TRY_R(coral::launch_row_select(D, ld, nq, nb, k, b0, part + ((size_t)q0 * nseg + s) * k, nseg * k, redo,
                                               stream));
        }
    }
    HIP_TRY_R(coral::launch_merge_segments(part, Q, (int)nseg, k, metric_out, d_ids, d_dists, stream));
    HIP_TRY_R(hipStreamSynchronize(stream));
#undef HIP_TRY_R
    release();
    return CORAL_OK;
}

}  // namespace

namespace coral {
// |b|^2 of the base, once per index
int ensure_base_norms(coral_index* idx, hipStream_t stream) {
    if (idx->d_bnorm) return CORAL_OK;
    if (!idx->d_bnorm_max) HIP_TRY(hipMalloc(&idx->d_bnorm_max, 2 * sizeof(uint32_t)));  // the largest norm; the largest loss
    float* norms = nullptr;
    HIP_TRY(hipMalloc(&norms, (size_t)idx->n * sizeof(float)));
    hipError_t e = launch_fill_u32(idx->d_bnorm_max, 2, 0u, stream);
    if (e == hipSuccess) e = launch_row_norms(idx->d_vec, idx->n, idx->dim, norms, idx->d_bnorm_max, nullptr, stream);
    if (e != hipSuccess) {
        (void)hipFree(norms);
        HIP_TRY(e);
    }
    idx->d_bnorm = norms;  // kept only once its kernel is on the stream
    return CORAL_OK;
}

// what the base's rows lose at most when they are rounded to halves (d_bnorm_max[1]), once per index; after
// ensure_base_norms
int ensure_base_loss(coral_index* idx, hipStream_t stream) {
    if (idx->bloss_ready) return CORAL_OK;
    HIP_TRY(launch_row_norms(idx->d_vec, idx->n, idx->dim, nullptr, nullptr, idx->d_bnorm_max + 1, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    idx->bloss_ready = true;
    return CORAL_OK;
}

}  // namespace coral

namespace {
constexpr int kScreenSlack = 32;  // candidates kept beyond k
constexpr int64_t kListCap = 16384;  // keys a query's candidate list holds at most in the fused screening
constexpr size_t kKnnKeepBytes = (size_t)384 << 20;

// Scratch of one call, carved from one block.  A block of up to kKnnKeepBytes stays with the index until it is
// destroyed: a dozen allocations and releases were 150 of the 274 us of a call with 100 queries.  Every call waits for
// its stream before it returns, so a call on another stream finds the block idle.  What needs more, and what finds the
// block taken -- by the call it is part of, which sends some of its queries through another screening -- has a block of
// its own.
class KnnScratch {
public:
    explicit KnnScratch(coral_index* idx) : idx_(idx) {}
    KnnScratch(const KnnScratch&) = delete;
    KnnScratch& operator=(const KnnScratch&) = delete;
    ~KnnScratch() {
        if (kept_)
            idx_->knn_block_taken.store(false, std::memory_order_release);
        else
            (void)hipFree(base_);
    }
    template <typename T>
    void reserve(T** p, size_t count) {
        parts_.push_back({reinterpret_cast<void**>(p), total_});
        total_ += (count * sizeof(T) + 255) & ~(size_t)255;
    }
    hipError_t allocate() {
        if (total_ <= kKnnKeepBytes && !idx_->knn_block_taken.exchange(true, std::memory_order_acquire)) {
            kept_ = true;
            if (idx_->knn_block_bytes < total_) {
                (void)hipFree(idx_->knn_block);
                idx_->knn_block = nullptr, idx_->knn_block_bytes = 0;
                if (hipError_t e = hipMalloc(&idx_->knn_block, total_)) return e;
                idx_->knn_block_bytes = total_;
            }
            base_ = idx_->knn_block;
        } else if (hipError_t e = hipMalloc(&base_, total_)) {
            return e;
        }
        for (auto& p : parts_) *p.first = static_cast<char*>(base_) + p.second;
        return hipSuccess;
    }
    size_t total() const { return total_; }
    // pinned room for the flags of Q queries and one more, or null: for the holder of the kept block
    int* flags(int32_t Q) const { return kept_ && Q < coral::kKnnFlags ? idx_->h_knn_flags : nullptr; }

private:
    coral_index* idx_;
    std::vector<std::pair<void**, size_t>> parts_;
    size_t total_ = 0;
    void* base_ = nullptr;
    bool kept_ = false;
};

// The screening with the selection inside the matrix-core kernel: no distance matrix goes to memory.  Per block of
// queries: (1) the distances to a sample of the base (every stride-th tile of 128 points) as a small matrix, whose
// kc-th smallest entry per row is a bound tau[q] that at least kc entries of the whole row do not exceed; (2) one
// pass over the whole base that appends the entries up to tau[q] to the query's list (about kc * n / sample of
// them) -- or two, where the base is many times the sample: first every step-th tile, whose kc smallest entries give
// a tighter bound for the rest, then the tiles between; (3) the kc smallest keys of every list.  The kept candidates
// are those of knn_passes(screen = true): the same approximate values, the kc smallest under (value, id).
struct FusedScreen {
    bool suits = false;  // the shape does: kc within what list_select_kernel takes, a base large enough to sample
    int64_t tiles = 0, stride = 0, ns = 0, qc = 0, qs = 0, cap = 0;
    int step = 1, kc = 0, products = 3;
    float *D = nullptr, *tau = nullptr;
    unsigned long long* lists = nullptr;
    unsigned int* cnt = nullptr;
    int *redo = nullptr, *overflow = nullptr;
    char* split = nullptr;

    void plan(const coral_index* idx, int32_t Q, int32_t kc_, int products_) {
        kc = kc_, products = products_;
        const int64_t n = idx->n, full_tiles = n / 128;
        tiles = (2 * (int64_t)kc * full_tiles + kListCap - 1) / kListCap;
        tiles = std::max<int64_t>(8, (tiles + 7) & ~(int64_t)7);
        if (kc > 1024 || tiles * 8 > full_tiles || n > 0x7fffffff) return;
        suits = true;
        // A larger sample than the lists need: an entry that passes costs an atomic and a scattered write.  A
        // sixteenth of the base, up to 16 384 points.
        tiles = std::max(tiles, std::min<int64_t>(128, (full_tiles / 16) & ~(int64_t)7));
        stride = full_tiles / tiles, ns = tiles * 128;
        // Two passes with bounds from ns and then from n / step points let through kc (n / step / ns + step) entries
        // per query instead of kc n / ns; step balances the two.  Worth a pass more only where the appending weighs
        // more than the launches.
        if (Q >= 1024 && stride >= 16)
            while ((step + 1) * (step + 1) <= stride) ++step;
        // three times the entries a list should see, of two passes the larger: kc to start with and kc * step more
        const int64_t expect = kc * (step > 1 ? (stride + step - 1) / step + step : stride) + kc;
        cap = 2048;
        while (cap < 3 * expect && cap < kListCap) cap <<= 1;
        // queries per block: a pass over the base for 4096 is hundreds of tiles per compute unit; the sample's matrix is
        // made and read for 2048 at a time
        const int64_t rows = ((int64_t)Q + 127) & ~(int64_t)127;
        qc = std::min<int64_t>(4096, rows);
        qs = std::min<int64_t>(2048, std::min(qc, std::max<int64_t>(256, (kBufferFloats / ns) & ~(int64_t)255)));
    }
    void reserve(const coral_index* idx, KnnScratch& mem) {
        if (!suits) return;
        // What is kept between calls holds 4096 lists of up to 8192 entries beside the sample's matrix for 1024 queries, but not
        // for 2048: 10 000 queries of a million points, k = 100, 349 MB and 413, which each call would allocate and release (11.0 and
        // 11.4 ms).  Elsewhere half the queries at a time cost up to 8 % of a call.  (Lists of 16 384, for k in the hundreds, are not
        // kept.)
        const size_t lists_bytes = (size_t)qc * cap * sizeof(unsigned long long) + (size_t)qc * coral::kCntStride * sizeof(unsigned int) +
                                   coral::split_queries_bytes((int)qc, idx->dim, 3) + 4096 * 8;  // (and the small parts, each rounded up)
        const auto fits = [&](int64_t rows) { return mem.total() + lists_bytes + (size_t)rows * ns * sizeof(float) <= kKnnKeepBytes; };
        if (!fits(qs) && qs > 1024 && fits(1024)) qs = 1024;
        mem.reserve(&D, (size_t)qs * ns), mem.reserve(&tau, (size_t)qc);
        mem.reserve(&lists, (size_t)qc * cap), mem.reserve(&cnt, (size_t)qc * coral::kCntStride);
        mem.reserve(&redo, (size_t)qs), mem.reserve(&overflow, 2);
        mem.reserve(&split, coral::split_queries_bytes((int)qc, idx->dim, 3));  // (the larger form: one product may give way to three)
    }
    // *used = false, with one product, when the sample says that too many entries lie where it cannot tell them apart
    // (d_qres: what it loses per query).  *overflow != 0 in the end where a list did (sample unlike the base, rows of equal
    // values, too few live points in the sample): its query has no candidates, and the caller goes through the matrix.
    // d_qn, d_qres: written here.
    int run(coral_index* idx, const float* d_queries, int32_t Q, int32_t have_delete, float* d_qn, float* d_qres,
            int32_t* d_cid, float* d_cd, hipStream_t stream, bool* used) {
        *used = false;
        const int64_t n = idx->n;
        const uint32_t* del = have_delete ? idx->d_deleted : nullptr;
        if (products == 1) {
            // The kc kept are meant to hold the k best whatever one product lost: kScreenSlack entries may lie too close.
            // How many do is asked of the sample and 64 queries first: at its kc-th entry; the k-th of the whole base
            // lies further out, where entries thin out up to twice as fast (as the 1.6th power: 1e-2 against 1e-4 of a
            // Gaussian).  (Costs 60 us whatever the answer.)
            const int probe = std::min(Q, 64);
            int extra = 0;
            HIP_TRY(coral::launch_prepare_queries(d_queries, probe, idx->dim, 1, d_qn, d_qres, split, nullptr, overflow, stream));
            HIP_TRY(coral::launch_approx_tile(split, idx->d_vec, probe, n, idx->dim, idx->metric, 1, d_qn, idx->d_bnorm, del, 0, D,
                                              ns, stream, tiles, (int)stride));
            HIP_TRY(coral::launch_row_select(D, ns, probe, ns, kc, 0, nullptr, 0, redo, stream, tau));
            HIP_TRY(coral::launch_count_close(D, ns, probe, ns, kc, idx->metric, d_qn, idx->d_bnorm_max, d_qres,
                                              idx->d_bnorm_max + 1, tau, overflow + 1, stream));
            HIP_TRY(hipMemcpyAsync(&extra, overflow + 1, sizeof extra, hipMemcpyDeviceToHost, stream));
            HIP_TRY(hipStreamSynchronize(stream));
            const double grown = 1.0 + (double)extra / ((double)probe * kc);
            if ((kc - kScreenSlack) * (std::pow(grown, 1.6) - 1.0) > 0.6 * kScreenSlack) return CORAL_OK;
        }
        for (int64_t q0 = 0; q0 < Q; q0 += qc) {
            const int nq = (int)std::min<int64_t>(qc, Q - q0);
            const float* qp = d_queries + (size_t)q0 * idx->dim;
            float* qn = d_qn + q0;
            HIP_TRY(coral::launch_prepare_queries(qp, nq, idx->dim, products, qn, d_qres ? d_qres + q0 : nullptr, split, cnt,
                                                  q0 == 0 ? overflow : nullptr, stream));
            for (int64_t s0 = 0; s0 < nq; s0 += qs) {
                const int ms = (int)std::min<int64_t>(qs, nq - s0);
                HIP_TRY(coral::launch_approx_tile(split + coral::split_queries_offset(s0, idx->dim, products), idx->d_vec, ms, n,
                                                  idx->dim, idx->metric, products, qn + s0, idx->d_bnorm, del, 0, D, ns, stream,
                                                  tiles, (int)stride));
                HIP_TRY(coral::launch_row_select(D, ns, ms, ns, kc, 0, nullptr, 0, redo, stream, tau + s0));
            }
            HIP_TRY(coral::launch_approx_filter(split, idx->d_vec, nq, n, idx->dim, idx->metric, products, qn, idx->d_bnorm, del, tau,
                                                lists, cap, cnt, step, stream));
            if (step > 1) {
                HIP_TRY(coral::launch_list_shrink(lists, cap, cnt, nq, kc, tau, overflow, stream));
                HIP_TRY(coral::launch_approx_filter(split, idx->d_vec, nq, n, idx->dim, idx->metric, products, qn, idx->d_bnorm, del,
                                                    tau, lists, cap, cnt, -step, stream));
            }
            HIP_TRY(coral::launch_list_select(lists, cap, cnt, nq, kc, d_cid + (size_t)q0 * kc, d_cd + (size_t)q0 * kc,
                                              overflow, stream));
        }
        *used = true;
        return CORAL_OK;
    }
};

}  // namespace

extern "C" {

int coral_bruteforce_set_exact_only(coral_index* idx, int32_t on) {
    if (!idx) return fail(CORAL_ERR_ARG, "null index");
    if (on < 0 || on > 2) return fail(CORAL_ERR_ARG, "on must be 0, 1 or 2 (got %d)", on);
    idx->knn_mode = on;
    return CORAL_OK;
}

int64_t coral_bruteforce_last_redone(coral_index* idx) { return idx ? idx->knn_last_redone : -1; }

int64_t coral_bruteforce_last_handed_on(coral_index* idx) { return idx ? idx->knn_last_handed_on : -1; }

int32_t coral_bruteforce_last_fused(coral_index* idx) { return idx ? (int32_t)idx->knn_last_fused : -1; }

static int check_knn(const coral_index* idx, int32_t Q, int32_t k, int32_t have_delete) {
    if (Q <= 0) return fail(CORAL_ERR_ARG, "Q must be positive");
    if (k <= 0 || k > 2048) return fail(CORAL_ERR_ARG, "k must be in 1..2048 (got %d)", k);
    if (have_delete && !idx->d_deleted)
        return fail(CORAL_ERR_STATE, "have_delete set but no tombstone mask was given");
    return CORAL_OK;
}

namespace {

// One product per pair pays where the products are what a call takes its time for, from about 0.7 ms of them on (one
// product against three, k = 10 / 200: 300 000 x 200, 1000 queries (6e10) 598 / 916 us against 642 / 866, 3000 queries 1247 /
// 2019 against 1625 / 2210; 1M x 200, 10 000 queries 8.9 / 13.4 ms against 15.0 / 19.0; 100 000 x 64, 3000 queries (1.9e10) the
// same).
bool one_product_pays(const coral_index* idx, int32_t Q) { return Q >= 256 && (double)Q * (double)idx->n * idx->dim >= 1e11; }

// Screening on the matrix cores, exact distances for the kc candidates of each query, and for the queries whose
// candidates cannot vouch for the result (bruteforce_mfma.hip): after the screening on one product the one on three,
// after that the exact passes.
struct Screening {
    int products = 3, kc = 0;
    float *d_qn = nullptr, *d_qres = nullptr, *d_cd = nullptr;
    int32_t* d_cid = nullptr;
    int* d_redo = nullptr;
    FusedScreen fused_screen;
    bool waited = false;  // the call's last work was what run() has waited for and `done` stands behind

    void reserve(const coral_index* idx, int32_t Q, int32_t k, int products_, KnnScratch& mem) {
        products = products_, kc = k + kScreenSlack;
        mem.reserve(&d_qn, (size_t)Q), mem.reserve(&d_qres, (size_t)Q), mem.reserve(&d_cid, (size_t)Q * kc);
        mem.reserve(&d_cd, (size_t)Q * kc), mem.reserve(&d_redo, (size_t)Q + 1);
        if (idx->knn_mode == 0) fused_screen.plan(idx, Q, kc, products);
        fused_screen.reserve(idx, mem);
    }

    // flags: pinned room for Q + 1 of them, or null; done (or null): recorded behind the re-rank
    int run(coral_index* idx, const float* d_queries, int32_t Q, int32_t k, int32_t have_delete, int32_t* d_ids, float* d_dists,
            hipStream_t stream, int* flags, hipEvent_t done) {
        if (int rc = coral::ensure_base_norms(idx, stream)) return rc;
        if (products == 1)
            if (int rc = coral::ensure_base_loss(idx, stream)) return rc;
        std::vector<int> copied;
        if (!flags) copied.resize((size_t)Q + 1);
        const int* redo = flags ? flags : copied.data();
        // One wait per attempt, behind the re-rank of its candidates: whether the lists were whole comes back with the
        // flags.  (Waits of their own for that and for the clock, two copies and three launches more were 50 of the 173 us of
        // a call with 100 queries.)
        for (bool matrix = !fused_screen.suits;; matrix = products == 3, products = fused_screen.products = 3) {
            const float* qres = products == 1 ? d_qres : nullptr;
            if (matrix) {
                products = 3, qres = nullptr;
                if (int rc = knn_passes(idx, d_queries, Q, kc, have_delete, true, d_qn, /*signed distances*/ 0, d_cid, d_cd, stream))
                    return rc;
            } else {
                bool used = false;
                if (int rc = fused_screen.run(idx, d_queries, Q, have_delete, d_qn, products == 1 ? d_qres : nullptr, d_cid, d_cd,
                                              stream, &used))
                    return rc;
                if (!used) continue;
            }
            idx->knn_last_fused = !matrix;
            HIP_TRY(coral::launch_rerank(d_queries, idx->d_vec, Q, idx->dim, idx->metric, d_cid, d_cd, kc, k, d_qn, idx->d_bnorm_max,
                                         qres, idx->d_bnorm_max + 1, d_ids, d_dists, flags ? flags : d_redo,
                                         matrix ? nullptr : fused_screen.overflow, stream));
            if (done) HIP_TRY(hipEventRecord(done, stream));
            if (!flags)
                HIP_TRY(hipMemcpyAsync(copied.data(), d_redo, copied.size() * sizeof(int), hipMemcpyDeviceToHost, stream));
            HIP_TRY(hipStreamSynchronize(stream));
            if (redo[Q] == 0) break;  // (the matrix path loses none)
        }
        std::vector<int32_t> rows;
        for (int32_t q = 0; q < Q; ++q)
            if (redo[(size_t)q]) rows.push_back(q);
        if (products == 1) idx->knn_last_handed_on = (int64_t)rows.size();
        if (products == 3) idx->knn_last_redone = (int64_t)rows.size();
        if (rows.empty()) {
            waited = done != nullptr;
            return CORAL_OK;
        }
        const int m = (int)rows.size();
        float *d_rq = nullptr, *d_rd = nullptr;
        int32_t *d_rows = nullptr, *d_rid = nullptr;
        KnnScratch mem(idx);
        mem.reserve(&d_rows, (size_t)m), mem.reserve(&d_rq, (size_t)m * idx->dim);
        mem.reserve(&d_rid, (size_t)m * k), mem.reserve(&d_rd, (size_t)m * k);
        HIP_TRY(mem.allocate());
        int rc = CORAL_OK;
        hipError_t e = hipMemcpyAsync(d_rows, rows.data(), (size_t)m * sizeof(int32_t), hipMemcpyHostToDevice, stream);
        if (e == hipSuccess) e = coral::launch_gather_rows(d_queries, idx->dim, d_rows, m, d_rq, stream);
        if (e == hipSuccess) {
            rc = products == 1 ? run_on_three(idx, d_rq, m, k, have_delete, d_rid, d_rd, stream)
                               : knn_passes(idx, d_rq, m, k, have_delete, false, nullptr, idx->metric, d_rid, d_rd, stream);
            if (rc == CORAL_OK) e = coral::launch_scatter_results(d_rows, m, k, d_rid, d_rd, d_ids, d_dists, stream);
        }
        const hipError_t ended = hipStreamSynchronize(stream);  // before the scratch and `rows` go
        if (rc == CORAL_OK) HIP_TRY(e);
        if (rc == CORAL_OK) HIP_TRY(ended);
        return rc;
    }

    static int run_on_three(coral_index* idx, const float* d_queries, int32_t Q, int32_t k, int32_t have_delete, int32_t* d_ids,
                            float* d_dists, hipStream_t stream) {
        Screening next;
        KnnScratch mem(idx);
        next.reserve(idx, Q, k, 3, mem);
        HIP_TRY(mem.allocate());
        const int rc = next.run(idx, d_queries, Q, k, have_delete, d_ids, d_dists, stream, mem.flags(Q), nullptr);
        if (rc != CORAL_OK) (void)hipStreamSynchronize(stream);  // nothing is in flight when the scratch goes back
        return rc;
    }
};

}  // namespace

// The search of one call.  Host buffers (h_queries, h_ids, h_dists) are staged in the call's scratch; otherwise the
// queries and results are d_queries, d_ids, d_dists.
static int knn_call(coral_index* idx, const float* d_queries, const float* h_queries, int32_t Q, int32_t k,
                    int32_t have_delete, int32_t* d_ids, int32_t* h_ids, float* d_dists, float* h_dists, hipStream_t stream,
                    double* time_s) {
    int rc = CORAL_OK;
    const int kc = k + kScreenSlack;
    const bool screen = !(idx->knn_mode == 1 || kc > 2048 || idx->n <= kc);
    const size_t qb = (size_t)Q * idx->dim * sizeof(float), ib = (size_t)Q * k * sizeof(int32_t);
    float* d_q = nullptr;
    Screening screening;
    KnnScratch mem(idx);
    if (h_queries) {
        mem.reserve(&d_q, (size_t)Q * idx->dim), mem.reserve(&d_ids, (size_t)Q * k);
        if (h_dists) mem.reserve(&d_dists, (size_t)Q * k);
    }
    if (screen) screening.reserve(idx, Q, k, idx->knn_mode == 0 && one_product_pays(idx, Q) ? 1 : 3, mem);
    auto ok = [&](hipError_t e, const char* what) {
        if (e == hipSuccess) return true;
        rc = fail(e == hipErrorOutOfMemory ? CORAL_ERR_MEMORY : CORAL_ERR_DEVICE, "%s failed: %s", what, hipGetErrorString(e));
        return false;
    };
    if ((h_queries || screen) && !ok(mem.allocate(), "hipMalloc")) return rc;
    if (h_queries) {
        if (!ok(hipMemcpy(d_q, h_queries, qb, hipMemcpyHostToDevice), "upload")) return rc;
        d_queries = d_q;
    }
    hipEvent_t ev0, ev1;
    HIP_TRY(hipEventCreate(&ev0));
    HIP_TRY(hipEventCreate(&ev1));
    HIP_TRY(hipEventRecord(ev0, stream));
    idx->knn_last_redone = 0, idx->knn_last_handed_on = -1;
    idx->knn_last_fused = false;
    if (!screen)
        rc = knn_passes(idx, d_queries, Q, k, have_delete, false, nullptr, idx->metric, d_ids, d_dists, stream);
    else
        rc = screening.run(idx, d_queries, Q, k, have_delete, d_ids, d_dists, stream, mem.flags(Q), ev1);
    if (rc == CORAL_OK) {
        float ms = 0.f;
        if ((screening.waited || (ok(hipEventRecord(ev1, stream), "event") && ok(hipEventSynchronize(ev1), "synchronize"))) &&
            ok(hipEventElapsedTime(&ms, ev0, ev1), "event") && time_s)
            *time_s = ms / 1000.0;
    }
    (void)hipEventDestroy(ev0);
    (void)hipEventDestroy(ev1);
    if (rc == CORAL_OK && h_queries &&
        (hipMemcpy(h_ids, d_ids, ib, hipMemcpyDeviceToHost) != hipSuccess ||
         (h_dists && hipMemcpy(h_dists, d_dists, ib, hipMemcpyDeviceToHost) != hipSuccess)))
        rc = fail(CORAL_ERR_DEVICE, "download failed");
    if (rc != CORAL_OK) (void)hipStreamSynchronize(stream);  // nothing of this call is in flight when the scratch goes back
    return rc;
}

int coral_bruteforce_knn_gpu(coral_index* idx, const float* d_queries, int32_t Q, int32_t k,
                             int32_t have_delete, int32_t* d_ids, float* d_dists, void* stream_,
                             double* time_s) {
    if (!idx || !d_queries || !d_ids) return fail(CORAL_ERR_ARG, "null argument");
    if (int rc = check_knn(idx, Q, k, have_delete)) return rc;
    HIP_TRY(hipSetDevice(idx->device));
    return knn_call(idx, d_queries, nullptr, Q, k, have_delete, d_ids, nullptr, d_dists, nullptr,
                    stream_ ? (hipStream_t)stream_ : idx->stream, time_s);
}

int coral_bruteforce_knn(coral_index* idx, const float* h_queries, int32_t Q, int32_t k, int32_t have_delete,
                         int32_t* h_ids, float* h_dists, double* time_s) {
    if (!idx || !h_queries || !h_ids) return fail(CORAL_ERR_ARG, "null argument");
    if (int rc = check_knn(idx, Q, k, have_delete)) return rc;
    HIP_TRY(hipSetDevice(idx->device));
    return knn_call(idx, nullptr, h_queries, Q, k, have_delete, nullptr, h_ids, nullptr, h_dists, idx->stream, time_s);
}

}  // extern "C"
