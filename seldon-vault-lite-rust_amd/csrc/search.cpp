// Host runtime of the exact vector search (the svl_vector_* part of
// include/svl_hip.h): vector::rank of src/index/vector.rs:17-97 plus the
// pagination slice of Index::search (src/index/mod.rs:347-359), for a batch
// of queries against chunk embeddings resident in HBM.
//
// The index keeps the chunk matrix in ascending chunk-id order (a stable sort
// of the caller's order), so the stable ranking sort breaks score ties by
// chunk id, then by the caller's order, as the reference's stable sort_by
// does. Each chunk's norm is sqrt of its squared sum accumulated in double in
// d order, computed once here instead of per query (it does not depend on
// the query); chunks whose sum is zero or non-finite are remembered and
// reported when a query's filter admits them (vector.rs:77-82).
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cmath>
#include <memory>
#include <mutex>
#include <numeric>
#include <thread>
#include <vector>

#include "../../include/svl_hip.h"
#include "host_common.hpp"
#include "svl_internal.hpp"

namespace {

using namespace svl;

constexpr int64_t MAX_EMBEDDING_DIMENSION = 8192;  // storage/model.rs:35

// Pinned host memory of an index that the kernels of one call read and write
// in place of copies: per query a flag word, a candidate count and the page
// length, and the page where it is small.
constexpr size_t HOST_PAGE_BYTES = (size_t)1 << 20;  // larger pages are copied instead
// Allocated with the index (64 queries of 63 hits; larger ones grow it): in an
// index's first call it took 30 to 100 us, which a small index does not win back
// there.
constexpr size_t HOST_PAGE_START = (size_t)64 << 10;
struct HostPage {
    unsigned char *p = nullptr;
    size_t bytes = 0;
    int *flags = nullptr;
    unsigned int *found = nullptr;
    int64_t *take = nullptr, *index = nullptr;  // index, score: null for large pages
    double *score = nullptr;

    hipError_t reserve(size_t need) {
        if (need <= bytes) return hipSuccess;
        release();
        const hipError_t e = hipHostMalloc((void **)&p, need, hipHostMallocDefault);
        if (e != hipSuccess) p = nullptr;
        else bytes = need;
        return e;
    }
    hipError_t ensure(int64_t nq, int64_t limit) {
        const bool page = limit <= (int64_t)(HOST_PAGE_BYTES / 16) / nq;
        const hipError_t e = reserve((size_t)nq * 16 + (page ? (size_t)(nq * limit) * 16 : 0));
        if (e != hipSuccess) return e;
        take = reinterpret_cast<int64_t *>(p);
        flags = reinterpret_cast<int *>(take + nq);
        found = reinterpret_cast<unsigned int *>(flags + nq);
        index = page ? reinterpret_cast<int64_t *>(found + nq) : nullptr;
        score = page ? reinterpret_cast<double *>(index + nq * limit) : nullptr;
        return hipSuccess;
    }
    void release() {
        if (p) (void)hipHostFree(p);
        p = nullptr;
        bytes = 0;
    }
};

}  // namespace

struct svl_vector_index {
    int device = -1;
    hipStream_t stream = nullptr;
    int64_t n = 0, D = 0;
    std::vector<uint64_t> ids;     // caller order
    std::vector<uint8_t> bad;      // caller order: zero / non-finite norm
    std::vector<int64_t> bad_list;  // caller indices with bad norms
    DevBuf<float> V;                // [n, D] chunk-id order
    DevBuf<double> cnorm;           // [n] chunk-id order
    DevBuf<int64_t> perm;           // chunk-id order -> caller index
    // per-call workspace
    DevBuf<float> Q;
    DevBuf<double> qnorm, Qd;
    HostPage page;  // flags, counts and page entries that kernels write for the host
    DevBuf<uint8_t> mask;
    DevBuf<uint64_t> keys, keys_alt;
    DevBuf<uint32_t> idx, idx_alt, qkey;
    DevBuf<unsigned char> tmp;
    DevBuf<uint64_t> thresh, cand_key, cand_key_alt;
    DevBuf<uint32_t> cand_idx, cand_idx_alt;
    DevBuf<unsigned int> cnt, seg_begin, seg_end, blk_count;
    DevBuf<int64_t> take, out_index;
    DevBuf<double> out_score;
    std::mutex mu;

    ~svl_vector_index() {
        if (device >= 0) (void)hipSetDevice(device);
        V.release(); cnorm.release(); perm.release(); Q.release(); qnorm.release();
        page.release(); Qd.release(); mask.release(); keys.release(); keys_alt.release(); idx.release();
        idx_alt.release(); qkey.release(); tmp.release(); take.release(); out_index.release();
        thresh.release(); cand_key.release(); cand_key_alt.release();
        cand_idx.release(); cand_idx_alt.release(); cnt.release(); seg_begin.release();
        seg_end.release(); blk_count.release();
        out_score.release();
        if (stream) (void)hipStreamDestroy(stream);
    }
};

namespace {

// vector.rs:24-53, one query on the host. Returns its norm.
svl_status check_query(const float *q, int64_t len, int64_t index_dim, bool has_dim, int32_t which,
                       double &norm) {
    if (len <= 0)
        return fail(SVL_USAGE, "query %d: query embedding must have at least one dimension", which);
    if (len > MAX_EMBEDDING_DIMENSION)
        return fail(SVL_LIMIT, "query %d: query embedding has %lld dimensions, above the %lld-dimension cap",
                    which, (long long)len, (long long)MAX_EMBEDDING_DIMENSION);
    double sum = 0.0;
    for (int64_t d = 0; d < len; ++d) {
        if (!std::isfinite(q[d]))
            return fail(SVL_USAGE, "query %d: query embedding contains a non-finite value", which);
        sum += (double)q[d] * (double)q[d];
    }
    if (!std::isfinite(sum) || sum <= 0.0)
        return fail(SVL_USAGE,
                    "query %d: query embedding norm is zero or non-finite; cosine similarity is undefined",
                    which);
    norm = std::sqrt(sum);
    if (has_dim && len != index_dim)
        return fail(SVL_USAGE, "query %d: query embedding dimension %lld does not match the index dimension %lld",
                    which, (long long)len, (long long)index_dim);
    return SVL_OK;
}

// The page from device memory, after the kernels that write it.
svl_status copy_page(svl_vector_index *ix, int32_t nq, int64_t limit, int64_t *out_index,
                     double *out_score, hipStream_t s) {
    HIP_TRY(hipMemcpyAsync(out_index, ix->out_index.p, (size_t)(nq * limit) * 8,
                           hipMemcpyDeviceToHost, s));
    HIP_TRY(hipMemcpyAsync(out_score, ix->out_score.p, (size_t)(nq * limit) * 8,
                           hipMemcpyDeviceToHost, s));
    HIP_TRY(hipStreamSynchronize(s));
    return SVL_OK;
}

// vector.rs:24-53 for queries in HBM: what launch_prepare_queries found, read
// after a synchronisation. `flags` null: checked on the host before.
svl_status check_flags(const int *flags, int32_t nq, int64_t query_dim, int64_t index_dim,
                       bool has_dim) {
    for (int32_t q = 0; flags && q < nq; ++q) {
        if (flags[q] & 1)
            return fail(SVL_USAGE, "query %d: query embedding contains a non-finite value", q);
        if (flags[q] & 2)
            return fail(SVL_USAGE,
                        "query %d: query embedding norm is zero or non-finite; cosine similarity is undefined", q);
        if (has_dim && query_dim != index_dim)
            return fail(SVL_USAGE, "query %d: query embedding dimension %lld does not match the index dimension %lld",
                        q, (long long)query_dim, (long long)index_dim);
    }
    return SVL_OK;
}

// Pages much smaller than the index (offset + limit <= n / 16): exact top-K
// by threshold. The sample (of 4096 evenly spaced keys per query) at a rank
// with margin above the expected (offset + limit) / n quantile is a threshold,
// and every admitted key at or below it is a candidate. When each query has at
// least min(offset + limit, admitted) candidates (and no more than the buffer
// holds), its page lies among them, and sorting only the candidates by (key,
// position) gives the ranking's exact entries; otherwise `selected` stays
// false and the full sort runs.
//
// Where twice the expected candidates fit one block's sort (pages within the
// first 300 hits of 1M chunks, 1000 of 200k), candidates are collected in any order, sorted
// and their page written, all enqueued at once: the host waits once and finds
// flags, counts and entries in its own memory. One query against 200003 x 768
// chunks takes 178 us this way (294 us with two waits in between, four copies
// and candidates counted, scanned and written in order), 64 queries 508
// (667). Longer lists are gathered in position order for a stable sort.
struct Selection {
    bool small = false, runs = false;
    int rank = 0;
    int64_t cap = 0;
};

Selection plan_selection(int64_t n, int64_t K, int32_t nq) {
    Selection p;
    constexpr int S = SAMPLE_COUNT;
    if (n < 16 * S || K > n / 16) return p;
    const int64_t stride = n / S;
    const double f = (double)K * S / (double)n;
    p.rank = (int)std::min<double>(S - 1, std::ceil(1.5 * f + 4.0 * std::sqrt(f) + 8.0));
    const int64_t twice = 2 * (int64_t)(p.rank + 1) * stride;
    p.small = twice <= CAND_LDS;
    p.cap = p.small ? CAND_LDS : std::min<int64_t>(n, twice + 4096);
    p.runs = (int64_t)nq * p.cap <= (int64_t)UINT32_MAX;
    return p;
}

bool lists_hold_pages(const unsigned int *found, const std::vector<int64_t> &pass, int64_t K,
                      int64_t cap, int64_t &most) {
    most = 0;
    for (size_t q = 0; q < pass.size(); ++q) {
        if ((int64_t)found[q] < std::min(K, pass[q]) || (int64_t)found[q] > cap) return false;
        most = std::max<int64_t>(most, found[q]);
    }
    return true;
}

svl_status ensure_candidates(svl_vector_index *ix, int32_t nq, int64_t cap) {
    HIP_TRY(ix->thresh.ensure((size_t)nq));
    HIP_TRY(ix->cnt.ensure((size_t)nq * CNT_STRIDE));
    HIP_TRY(ix->cand_key.ensure((size_t)(nq * cap)));
    HIP_TRY(ix->cand_idx.ensure((size_t)(nq * cap)));
    return SVL_OK;
}

// Short lists: enqueued whole. The entries are in the host page, or in
// out_index / out_score of the device for a large one.
svl_status enqueue_short_lists(svl_vector_index *ix, const Selection &p, int32_t nq, int64_t offset,
                               int64_t limit, hipStream_t s) {
    HIP_TRY(launch_sample_threshold(ix->keys.p, nq, ix->n, p.rank, ix->thresh.p, ix->cnt.p, s));
    HIP_TRY(launch_collect_candidates(ix->keys.p, nq, ix->n, ix->thresh.p, p.cap, ix->cnt.p,
                                      ix->cand_key.p, ix->cand_idx.p, s));
    const bool direct = ix->page.index != nullptr;
    HIP_TRY(launch_rank_candidates(ix->cand_key.p, ix->cand_idx.p, ix->cnt.p, nq, ix->n, p.cap,
                                   ix->perm.p, offset, limit, ix->page.take, ix->page.found,
                                   direct ? ix->page.index : ix->out_index.p,
                                   direct ? ix->page.score : ix->out_score.p, s));
    return SVL_OK;
}

svl_status select_long_lists(svl_vector_index *ix, const Selection &p, int32_t nq, int64_t offset,
                             int64_t limit, const std::vector<int64_t> &pass, int64_t *out_index,
                             double *out_score, hipStream_t s, bool &selected) {
    const int64_t n = ix->n, cap = p.cap;
    HIP_TRY(ix->cand_key_alt.ensure((size_t)(nq * cap)));
    HIP_TRY(ix->cand_idx_alt.ensure((size_t)(nq * cap)));
    HIP_TRY(ix->blk_count.ensure((size_t)nq * (size_t)candidate_blocks(n)));
    HIP_TRY(launch_sample_threshold(ix->keys.p, nq, n, p.rank, ix->thresh.p, ix->cnt.p, s));
    HIP_TRY(launch_compact_keys(ix->keys.p, nq, n, ix->thresh.p, cap, ix->blk_count.p, ix->cnt.p,
                                ix->page.found, ix->cand_key.p, ix->cand_idx.p, s));
    HIP_TRY(hipStreamSynchronize(s));
    int64_t most;
    if (!lists_hold_pages(ix->page.found, pass, offset + limit, cap, most)) return SVL_OK;
    if (most <= CAND_LDS) {
        HIP_TRY(launch_rank_candidates(ix->cand_key.p, ix->cand_idx.p, ix->cnt.p, nq, n, cap,
                                       ix->perm.p, offset, limit, ix->page.take, ix->page.found,
                                       ix->out_index.p, ix->out_score.p, s));
    } else {
        HIP_TRY(ix->seg_begin.ensure((size_t)nq));
        HIP_TRY(ix->seg_end.ensure((size_t)nq));
        size_t b = 0;
        HIP_TRY(sort_candidates(ix->cand_key.p, ix->cand_idx.p, ix->cand_key_alt.p,
                                ix->cand_idx_alt.p, ix->cnt.p, ix->seg_begin.p, ix->seg_end.p, nq,
                                cap, nullptr, &b, s));
        HIP_TRY(ix->tmp.ensure(std::max<size_t>(b, 1)));
        HIP_TRY(sort_candidates(ix->cand_key.p, ix->cand_idx.p, ix->cand_key_alt.p,
                                ix->cand_idx_alt.p, ix->cnt.p, ix->seg_begin.p, ix->seg_end.p, nq,
                                cap, ix->tmp.p, &b, s));
        HIP_TRY(launch_gather_candidates(ix->cand_key_alt.p, ix->cand_idx_alt.p, nq, n, cap,
                                         ix->perm.p, offset, limit, ix->page.take,
                                         ix->out_index.p, ix->out_score.p, s));
    }
    ST_TRY(copy_page(ix, nq, limit, out_index, out_score, s));
    selected = true;
    return SVL_OK;
}

// The ranking of `nq` queries [nq, D] in HBM. With `norms` null their norms
// are taken and checked on the device here (the first wait reports them),
// otherwise `norms` holds those of queries that were checked on the host.
svl_status rank_queries(svl_vector_index *ix, const float *queries, const double *norms,
                        int32_t nq, int64_t query_dim, const uint8_t *mask, int64_t mask_stride,
                        int64_t offset, int64_t limit, int64_t *out_index, double *out_score,
                        int64_t *out_count, hipStream_t s) {
    const int64_t n = ix->n, count = (int64_t)nq * n;
    HIP_TRY(ix->qnorm.ensure((size_t)nq));
    HIP_TRY(ix->page.ensure(nq, limit));
    int *flags = norms ? nullptr : ix->page.flags;
    // admitted chunks per query, and the first admitted bad chunk (vector.rs:77-82)
    std::vector<int64_t> pass((size_t)nq, n);
    int64_t bad = -1;
    int32_t bad_query = nq;
    for (int32_t q = 0; q < nq && bad < 0; ++q) {
        if (mask) {
            const uint8_t *m = mask + (int64_t)q * mask_stride;
            int64_t cnt = 0;
            for (int64_t c = 0; c < n; ++c) cnt += m[c] != 0;
            pass[(size_t)q] = cnt;
        }
        for (int64_t b : ix->bad_list)
            if (!mask || mask[(int64_t)q * mask_stride + b]) {
                bad = b;
                bad_query = q;
                break;
            }
        ix->page.take[q] = std::max<int64_t>(0, std::min(limit, pass[(size_t)q] - offset));
    }
    if (bad >= 0 || n == 0 || limit == 0 || query_dim != ix->D || count > (int64_t)UINT32_MAX) {
        // nothing to rank: the queries' own errors come first
        if (flags) {
            HIP_TRY(launch_prepare_queries(queries, nq, (int)query_dim, nullptr, ix->qnorm.p,
                                           flags, s));
            HIP_TRY(hipStreamSynchronize(s));
            ST_TRY(check_flags(flags, nq, query_dim, ix->D, n > 0));
        }
        for (int32_t q = 0; q < bad_query; ++q) out_count[q] = ix->page.take[q];
        if (bad >= 0)
            return fail(SVL_INTERNAL, "query %d: chunk %llu has a zero or non-finite embedding norm",
                        bad_query, (unsigned long long)ix->ids[(size_t)bad]);
        if (n == 0 || limit == 0) return SVL_OK;
        return fail(SVL_LIMIT, "queries x chunks exceeds 2^32 pairs");
    }
    HIP_TRY(ix->keys.ensure((size_t)count));
    HIP_TRY(ix->out_index.ensure((size_t)(nq * limit)));
    HIP_TRY(ix->out_score.ensure((size_t)(nq * limit)));
    const int qb = cosine_query_block(nq);
    HIP_TRY(ix->Qd.ensure((size_t)(ix->D * ((nq + qb - 1) / qb * qb))));
    const uint8_t *d_mask = nullptr;
    int64_t d_stride = 0;
    if (mask) {
        const int64_t rows = mask_stride == 0 ? 1 : nq;
        HIP_TRY(ix->mask.ensure((size_t)(rows * n)));
        for (int64_t r = 0; r < rows; ++r)
            HIP_TRY(hipMemcpyAsync(ix->mask.p + r * n, mask + r * mask_stride, (size_t)n,
                                   hipMemcpyHostToDevice, s));
        d_mask = ix->mask.p;
        d_stride = mask_stride == 0 ? 0 : n;
    }
    if (norms)
        HIP_TRY(hipMemcpyAsync(ix->qnorm.p, norms, (size_t)nq * 8, hipMemcpyHostToDevice, s));
    const Selection plan = plan_selection(n, offset + limit, nq);
    if (plan.runs) ST_TRY(ensure_candidates(ix, nq, plan.cap));
    HIP_TRY(launch_prepare_queries(queries, nq, (int)ix->D, ix->Qd.p, ix->qnorm.p, flags, s));
    HIP_TRY(launch_cosine_keys(ix->V.p, ix->cnorm.p, ix->Qd.p, ix->qnorm.p, nq, n, (int)ix->D,
                               d_mask, d_stride, ix->perm.p, ix->keys.p, s));
    const bool small = plan.runs && plan.small;
    if (small) ST_TRY(enqueue_short_lists(ix, plan, nq, offset, limit, s));
    if (small || flags) HIP_TRY(hipStreamSynchronize(s));
    ST_TRY(check_flags(flags, nq, query_dim, ix->D, true));
    std::copy(ix->page.take, ix->page.take + nq, out_count);
    int64_t most;
    if (small && lists_hold_pages(ix->page.found, pass, offset + limit, plan.cap, most)) {
        if (!ix->page.index) return copy_page(ix, nq, limit, out_index, out_score, s);
        for (int32_t q = 0; q < nq; ++q) {
            const int64_t at = (int64_t)q * limit, m = ix->page.take[q];
            std::copy(ix->page.index + at, ix->page.index + at + m, out_index + at);
            std::copy(ix->page.score + at, ix->page.score + at + m, out_score + at);
        }
        return SVL_OK;
    }
    bool selected = false;
    if (plan.runs && !plan.small)
        ST_TRY(select_long_lists(ix, plan, nq, offset, limit, pass, out_index, out_score, s,
                                 selected));
    if (selected) return SVL_OK;
    HIP_TRY(ix->keys_alt.ensure((size_t)count));
    HIP_TRY(ix->idx.ensure((size_t)count));
    HIP_TRY(ix->idx_alt.ensure((size_t)count));
    HIP_TRY(ix->qkey.ensure((size_t)count));
    size_t tmp_bytes = 0;
    const uint32_t *sorted = nullptr;
    HIP_TRY(rank_sort(ix->keys.p, ix->keys_alt.p, ix->idx.p, ix->idx_alt.p, ix->qkey.p, nq, n,
                      nullptr, &tmp_bytes, &sorted, s));
    HIP_TRY(ix->tmp.ensure(std::max<size_t>(tmp_bytes, 1)));
    HIP_TRY(rank_sort(ix->keys.p, ix->keys_alt.p, ix->idx.p, ix->idx_alt.p, ix->qkey.p, nq, n,
                      ix->tmp.p, &tmp_bytes, &sorted, s));
    HIP_TRY(launch_gather_hits(ix->keys.p, sorted, nq, n, ix->perm.p, offset, limit, ix->page.take,
                               ix->out_index.p, ix->out_score.p, s));
    return copy_page(ix, nq, limit, out_index, out_score, s);
}

svl_status check_page(int32_t nq, int64_t offset, int64_t limit, int64_t *out_index,
                      double *out_score, int64_t *out_count) {
    if (nq < 0 || offset < 0 || limit < 0) return fail(SVL_USAGE, "negative query count, offset or limit");
    if (nq > 0 && (!out_count || (limit > 0 && (!out_index || !out_score))))
        return fail(SVL_USAGE, "outputs are required");
    return SVL_OK;
}

}  // namespace

extern "C" {

svl_status svl_vector_index_create(svl_ctx *ctx, const float *embeddings,
                                   const uint64_t *chunk_ids, int64_t n, int64_t dimension,
                                   svl_vector_index **out) {
    if (!ctx || !out || n < 0 || (n > 0 && (!embeddings || !chunk_ids)))
        return fail(SVL_USAGE, "context, embeddings, chunk ids and output are required");
    *out = nullptr;
    if (n > 0 && (dimension <= 0 || dimension > MAX_EMBEDDING_DIMENSION))
        return fail(SVL_LIMIT, "embedding dimension %lld is outside 1..=%lld", (long long)dimension,
                    (long long)MAX_EMBEDDING_DIMENSION);
    if (n * std::max<int64_t>(dimension, 1) > MAX_TENSOR_ELEMENTS * 4)
        return fail(SVL_LIMIT, "index of %lld x %lld embeddings is too large", (long long)n,
                    (long long)dimension);
    std::unique_ptr<svl_vector_index> ix(new svl_vector_index());
    ix->device = ctx->device;
    ix->n = n;
    ix->D = n > 0 ? dimension : 0;
    HIP_TRY(hipSetDevice(ix->device));
    HIP_TRY(hipStreamCreateWithFlags(&ix->stream, hipStreamNonBlocking));
    HIP_TRY(ix->page.reserve(HOST_PAGE_START));
    ix->ids.assign(chunk_ids, chunk_ids + n);
    std::vector<int64_t> perm((size_t)n);
    std::iota(perm.begin(), perm.end(), 0);
    std::stable_sort(perm.begin(), perm.end(),
                     [&](int64_t a, int64_t b) { return chunk_ids[a] < chunk_ids[b]; });
    // squared sums in d order (vector.rs:71-78), chunk by chunk on host threads
    std::vector<double> norm((size_t)n);
    ix->bad.assign((size_t)n, 0);
    const int64_t D = ix->D;
    const int threads = (int)std::min<int64_t>(std::max(1u, std::thread::hardware_concurrency()),
                                               std::min<int64_t>(16, std::max<int64_t>(n / 1024, 1)));
    auto work = [&](int k) {
        for (int64_t c = k; c < n; c += threads) {
            const float *v = embeddings + c * D;
            double sum = 0.0;
            for (int64_t d = 0; d < D; ++d) sum += (double)v[d] * (double)v[d];
            if (!std::isfinite(sum) || sum <= 0.0) {
                ix->bad[(size_t)c] = 1;
                norm[(size_t)c] = 1.0;
            } else {
                norm[(size_t)c] = std::sqrt(sum);
            }
        }
    };
    std::vector<std::thread> pool;
    for (int k = 1; k < threads; ++k) pool.emplace_back(work, k);
    work(0);
    for (auto &t : pool) t.join();
    for (int64_t c = 0; c < n; ++c)
        if (ix->bad[(size_t)c]) ix->bad_list.push_back(c);
    if (n > 0) {
        std::vector<double> cn((size_t)n);
        for (int64_t p = 0; p < n; ++p) cn[(size_t)p] = norm[(size_t)perm[(size_t)p]];
        HIP_TRY(ix->V.ensure((size_t)(n * D)));
        HIP_TRY(ix->cnorm.ensure((size_t)n));
        HIP_TRY(ix->perm.ensure((size_t)n));
        // rows in chunk-id order, staged through a bounded host buffer
        const int64_t rows_per = std::max<int64_t>(1, ((int64_t)64 << 20) / (D * 4));
        std::vector<float> stage((size_t)(std::min(rows_per, n) * D));
        for (int64_t p0 = 0; p0 < n; p0 += rows_per) {
            const int64_t rows = std::min(rows_per, n - p0);
            for (int64_t r = 0; r < rows; ++r)
                std::copy(embeddings + perm[(size_t)(p0 + r)] * D,
                          embeddings + (perm[(size_t)(p0 + r)] + 1) * D, stage.data() + r * D);
            HIP_TRY(hipMemcpy(ix->V.p + p0 * D, stage.data(), (size_t)(rows * D) * 4,
                              hipMemcpyHostToDevice));
        }
        HIP_TRY(hipMemcpy(ix->cnorm.p, cn.data(), (size_t)n * 8, hipMemcpyHostToDevice));
        HIP_TRY(hipMemcpy(ix->perm.p, perm.data(), (size_t)n * 8, hipMemcpyHostToDevice));
    }
    *out = ix.release();
    return SVL_OK;
}

svl_status svl_vector_index_destroy(svl_vector_index *index) {
    delete index;
    return SVL_OK;
}

int64_t svl_vector_index_size(const svl_vector_index *index) { return index ? index->n : -1; }

int64_t svl_vector_index_dimension(const svl_vector_index *index) {
    return index ? index->D : -1;
}

svl_status svl_vector_rank(svl_vector_index *ix, const float *queries, int32_t nq,
                           int64_t query_dim, const uint8_t *mask, int64_t mask_stride,
                           int64_t offset, int64_t limit, int64_t *out_index, double *out_score,
                           int64_t *out_count) {
    if (!ix || (nq > 0 && !queries)) return fail(SVL_USAGE, "index and queries are required");
    ST_TRY(check_page(nq, offset, limit, out_index, out_score, out_count));
    if (mask_stride != 0 && mask_stride < ix->n) return fail(SVL_USAGE, "mask stride is shorter than the index");
    std::lock_guard<std::mutex> lock(ix->mu);
    std::vector<double> qn((size_t)nq);
    for (int32_t q = 0; q < nq; ++q)
        ST_TRY(check_query(queries + (int64_t)q * std::max<int64_t>(query_dim, 0), query_dim, ix->D,
                           ix->n > 0, q, qn[(size_t)q]));
    if (nq == 0) return SVL_OK;
    HIP_TRY(hipSetDevice(ix->device));
    hipStream_t s = ix->stream;
    if (ix->n > 0) {
        HIP_TRY(ix->Q.ensure((size_t)(nq * ix->D)));
        HIP_TRY(hipMemcpyAsync(ix->Q.p, queries, (size_t)(nq * ix->D) * 4, hipMemcpyHostToDevice, s));
    }
    return rank_queries(ix, ix->Q.p, qn.data(), nq, ix->D, mask, mask_stride, offset, limit,
                        out_index, out_score, out_count, s);
}

svl_status svl_vector_rank_device(svl_vector_index *ix, const float *d_queries, int32_t nq,
                                  int64_t query_dim, const uint8_t *mask, int64_t mask_stride,
                                  int64_t offset, int64_t limit, int64_t *out_index,
                                  double *out_score, int64_t *out_count, void *stream) {
    if (!ix || (nq > 0 && !d_queries)) return fail(SVL_USAGE, "index and queries are required");
    ST_TRY(check_page(nq, offset, limit, out_index, out_score, out_count));
    if (mask_stride != 0 && mask_stride < ix->n) return fail(SVL_USAGE, "mask stride is shorter than the index");
    if (nq > 0 && query_dim <= 0)
        return fail(SVL_USAGE, "query embedding must have at least one dimension");
    if (query_dim > MAX_EMBEDDING_DIMENSION)
        return fail(SVL_LIMIT, "query embedding has %lld dimensions, above the %lld-dimension cap",
                    (long long)query_dim, (long long)MAX_EMBEDDING_DIMENSION);
    std::lock_guard<std::mutex> lock(ix->mu);
    if (nq == 0) return SVL_OK;
    HIP_TRY(hipSetDevice(ix->device));
    hipStream_t s = stream ? (hipStream_t)stream : ix->stream;
    return rank_queries(ix, d_queries, nullptr, nq, query_dim, mask, mask_stride, offset, limit,
                        out_index, out_score, out_count, s);
}

}  // extern "C"
