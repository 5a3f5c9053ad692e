"""GPU parity of the exact vector search (vector::rank,
src/index/vector.rs:17-97, sliced like Index::search, index/mod.rs:347-359)
through the C ABI. The bar is bit-identical: the same chunk indices in the
same order and the same f64 score bits as the oracle, which restates the
reference's sequential double accumulation.

Cases: the reference's unit tests; a ragged dimension (not a multiple of the
32-wide slice) and a chunk count that is not a multiple of the 256-chunk
tile; exact score ties broken by chunk id; per-query and shared filters;
every query-block width (1, 4, 8, 16, 32, 64 and tails), dimensions that are
and are not a multiple of 4 (vector and scalar staging); pagination slices and
the full ranking; queries already in HBM; a 200k x 768 index, on which blocks
of 16-64 queries (FP64 matrix cores) equal single queries (vector FMAs) bit for
bit; the error taxonomy."""
import math

import numpy as np
import pytest

import svl_amd as S
import svl_search as V
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def corpus(n, d, seed, ties=True):
    rng = np.random.default_rng(seed)
    emb = rng.standard_normal((n, d)).astype(np.float32)
    if ties and n > 40:
        emb[20:30] = emb[3]            # exact score ties
        emb[31] = -emb[3]
    ids = rng.permutation(np.arange(1, n + 1) * 3 + 11).astype(np.uint64)
    return emb, ids


def check_query(ix, emb, ids, q, got, mask=None, offset=0, limit=None, label=""):
    want_i, want_s = O.vector_rank(q, emb, ids, mask=mask)
    lim = want_i.size if limit is None else limit
    want_i, want_s = want_i[offset:offset + lim], want_s[offset:offset + lim]
    gi, gs = got
    assert np.array_equal(gi, want_i), f"{label}: order differs at {np.flatnonzero(gi != want_i)[:5]}"
    assert np.array_equal(gs.view(np.uint64), want_s.view(np.uint64)), f"{label}: score bits"


def test_reference_unit_cases():
    ix = V.VectorIndex(np.array([[1, 0], [0, 1], [1, 1]], np.float32), [1, 2, 3])
    (idx, score), = ix.rank([1.0, 0.0])
    assert list(idx) == [0, 2, 1]
    assert abs(score[0] - 1) < 1e-9 and abs(score[1] - math.sqrt(0.5)) < 1e-6 and abs(score[2]) < 1e-9
    ix2 = V.VectorIndex(np.array([[1, 0], [1, 0]], np.float32), [1, 2])
    (idx, _), = ix2.rank([1.0, 0.0], masks=np.array([[0, 1]], np.uint8))
    assert list(idx) == [1]
    empty = V.VectorIndex(np.zeros((0, 2), np.float32), [])
    (idx, _), = empty.rank([1.0, 0.0])
    assert idx.size == 0 and empty.dimension() is None
    hits = ix.search(np.array([1.0, 0.0], np.float32), limit=2, offset=1)
    assert [(h.index, h.chunk_id, h.vector_rank) for h in hits] == [(2, 3, 2), (1, 2, 3)]


@pytest.mark.parametrize("nq,d", [(1, 100), (3, 100), (8, 100), (16, 100), (33, 100), (64, 100),
                                  (65, 100), (40, 99), (12, 99)])
def test_batches_match_oracle_bit_for_bit(nq, d):
    n = 1000 + 37                              # ragged tile; d ragged against the 32-wide slice
    emb, ids = corpus(n, d, seed=nq)
    ix = V.VectorIndex(emb, ids)
    rng = np.random.default_rng(100 + nq)
    qs = rng.standard_normal((nq, d)).astype(np.float32)
    qs[0] = emb[3] * 0.5                        # ties at the top
    masks = (rng.random((nq, n)) > 0.3).astype(np.uint8)
    masks[0, :] = 1
    full = ix.rank(qs)
    page = ix.rank(qs, masks=masks, offset=5, limit=40)
    for q in range(nq):
        check_query(ix, emb, ids, qs[q], full[q], label=f"query {q} full")
        check_query(ix, emb, ids, qs[q], page[q], mask=masks[q], offset=5, limit=40,
                    label=f"query {q} page")
    one = (rng.random(n) > 0.5).astype(np.uint8)
    shared = ix.rank(qs, masks=one, limit=10)
    for q in range(nq):
        check_query(ix, emb, ids, qs[q], shared[q], mask=one, limit=10,
                    label=f"query {q} shared mask")


def test_device_queries_and_large_index():
    import torch
    n, d = 200_000, 768
    emb, ids = corpus(n, d, seed=9)
    ix = V.VectorIndex(emb, ids)
    rng = np.random.default_rng(10)
    qs = rng.standard_normal((5, d)).astype(np.float32)
    host = ix.rank(qs, limit=100)
    dq = torch.from_numpy(qs).to("cuda:0")
    torch.cuda.synchronize()
    dev = ix.rank_device(dq.data_ptr(), 5, d, limit=100)
    for q in range(5):
        assert np.array_equal(host[q][0], dev[q][0])
        assert np.array_equal(host[q][1].view(np.uint64), dev[q][1].view(np.uint64))
    for q in (0, 4):
        check_query(ix, emb, ids, qs[q], host[q], limit=100, label=f"200k query {q}")
    deep = ix.rank(qs[:1], offset=150_000, limit=1000)
    check_query(ix, emb, ids, qs[0], deep[0], offset=150_000, limit=1000, label="deep page")


def test_matrix_core_blocks_equal_single_queries_at_scale():
    """Blocks of 16, 32 and 64 queries take the FP64 matrix-core score kernel
    and single queries the vector-FMA kernel. Both sum in dimension order, so
    on a 200k x 768 index every ranking and every score bit must agree; three
    queries are also checked against the oracle."""
    n, d = 200_000, 768
    emb, ids = corpus(n, d, seed=31)
    ix = V.VectorIndex(emb, ids)
    rng = np.random.default_rng(32)
    qs = rng.standard_normal((64, d)).astype(np.float32)
    single = [ix.rank(qs[q:q + 1], limit=50)[0] for q in range(64)]
    for nq in (16, 32, 64):
        block = ix.rank(qs[:nq], limit=50)
        for q in range(nq):
            assert np.array_equal(block[q][0], single[q][0]), f"{nq}-query block, query {q}"
            assert np.array_equal(block[q][1].view(np.uint64), single[q][1].view(np.uint64)), \
                f"{nq}-query block, query {q} score bits"
    for q in (0, 17, 63):
        check_query(ix, emb, ids, qs[q], single[q], limit=50, label=f"200k query {q}")


def test_concurrent_calls_equal_serial_calls():
    """Calls on one index from several threads (the reference's server runs
    searches concurrently) are serialised by the index and give the serial
    results bit for bit, across the vector-FMA and matrix-core paths."""
    from concurrent.futures import ThreadPoolExecutor
    n, d = 20_000, 128
    emb, ids = corpus(n, d, seed=41)
    ix = V.VectorIndex(emb, ids)
    rng = np.random.default_rng(42)
    batches = [rng.standard_normal((nq, d)).astype(np.float32) for nq in (1, 16, 3, 64, 33, 8)]
    serial = [ix.rank(b, limit=20) for b in batches]
    with ThreadPoolExecutor(max_workers=6) as ex:
        threaded = list(ex.map(lambda b: ix.rank(b, limit=20), batches * 3))
    for i, got in enumerate(threaded):
        want = serial[i % len(batches)]
        for (gi, gs), (wi, ws) in zip(got, want):
            assert np.array_equal(gi, wi) and np.array_equal(gs.view(np.uint64), ws.view(np.uint64))


def test_error_taxonomy():
    import torch
    emb = np.array([[1, 0], [0, 0], [0, 1]], np.float32)    # chunk 2 has a zero norm
    ix = V.VectorIndex(emb, [5, 6, 7])
    for q, kind in (([1.0, 0.0, 0.0], "Usage"), ([0.0, 0.0], "Usage"), ([np.nan, 1.0], "Usage"),
                    ([np.inf, 0.0], "Usage")):
        with pytest.raises(S.SvlError) as e:
            ix.rank(np.array(q, np.float32))
        assert e.value.kind == kind
        d = torch.tensor(np.array(q, np.float32).reshape(1, -1), device="cuda:0")
        torch.cuda.synchronize()
        with pytest.raises(S.SvlError) as e:
            ix.rank_device(d.data_ptr(), 1, d.shape[1])
        assert e.value.kind == kind
    with pytest.raises(S.SvlError) as e:       # the admitted zero-norm chunk
        ix.rank(np.array([1.0, 0.0], np.float32))
    assert e.value.kind == "Internal"
    (idx, _), = ix.rank(np.array([1.0, 0.0], np.float32), masks=np.array([[1, 0, 1]], np.uint8))
    assert list(idx) == [0, 2]
    with pytest.raises(S.SvlError) as e:
        ix.rank(np.ones((1, 8193), np.float32))
    assert e.value.kind == "LimitExceeded"
    with pytest.raises(S.SvlError) as e:       # SearchRequest::validate
        ix.search(np.array([1.0, 0.0], np.float32), limit=0)
    assert e.value.kind == "Usage"


def test_top_k_selection_path():
    """Pages far smaller than the index take the threshold selection; ties
    at the top (400 identical chunks), sparse filters and a query with fewer
    admitted chunks than the page must still give the exact ranking."""
    n, d = 80_000, 64
    emb, ids = corpus(n, d, seed=21, ties=False)
    emb[1000:1400] = emb[7]
    ix = V.VectorIndex(emb, ids)
    rng = np.random.default_rng(22)
    qs = rng.standard_normal((6, d)).astype(np.float32)
    qs[1] = emb[7]
    masks = np.ones((6, n), np.uint8)
    masks[2] = rng.random(n) > 0.97
    masks[3] = 0
    masks[3, rng.choice(n, 5, replace=False)] = 1          # 5 admitted < page
    for offset, limit in ((0, 10), (3, 50), (100, 1000)):
        got = ix.rank(qs, masks=masks, offset=offset, limit=limit)
        for q in range(6):
            check_query(ix, emb, ids, qs[q], got[q], mask=masks[q], offset=offset, limit=limit,
                        label=f"query {q} page ({offset}, {limit})")
            # one query alone: the same page, bit for bit
            one = ix.rank(qs[q:q + 1], masks=masks[q:q + 1], offset=offset, limit=limit)[0]
            assert np.array_equal(one[0], got[q][0]), f"query {q} alone ({offset}, {limit})"
            assert np.array_equal(one[1].view(np.uint64), got[q][1].view(np.uint64))
        # and three and four queries
        for k in (3, 4):
            few = ix.rank(qs[:k], masks=masks[:k], offset=offset, limit=limit)
            for q in range(k):
                assert np.array_equal(few[q][0], got[q][0]), f"{k} queries, query {q}"
                assert np.array_equal(few[q][1].view(np.uint64), got[q][1].view(np.uint64))


@pytest.mark.parametrize("n,offset,limit", [(70_001, 0, 10), (70_001, 390, 10), (70_001, 5, 1000),
                                            (70_001, 0, 2150), (140_000, 8000, 700)])
@pytest.mark.parametrize("nq,d", [(1, 36), (5, 37), (70, 36)])
def test_candidate_lists_of_every_length(n, offset, limit, nq, d):
    """Pages whose candidate lists take one, two, four and eight entries per
    lane of the block that sorts them, and more than it holds; queries in HBM
    at an address that is a multiple of 4 bytes only, padded to a block of 4,
    8 and 128; pages above and below the size that is written into host memory."""
    import torch
    emb, ids = corpus(n, d, seed=n + limit)
    ix = V.VectorIndex(emb, ids)
    rng = np.random.default_rng(nq + limit)
    qs = rng.standard_normal((nq, d)).astype(np.float32)
    buf = torch.zeros(nq * d + 1, device="cuda:0")
    buf[1:] = torch.from_numpy(qs.reshape(-1)).to("cuda:0")
    torch.cuda.synchronize()
    got = ix.rank_device(buf.data_ptr() + 4, nq, d, offset=offset, limit=limit)
    host = ix.rank(qs, offset=offset, limit=limit)
    for q in range(nq):
        assert np.array_equal(got[q][0], host[q][0])
        assert np.array_equal(got[q][1].view(np.uint64), host[q][1].view(np.uint64))
    for q in {0, nq // 2, nq - 1}:
        check_query(ix, emb, ids, qs[q], got[q], offset=offset, limit=limit, label=f"query {q}")
    # a query that must be refused does not disturb the next call
    buf[1 + (nq - 1) * d] = float("nan")
    torch.cuda.synchronize()
    with pytest.raises(S.SvlError) as e:
        ix.rank_device(buf.data_ptr() + 4, nq, d, offset=offset, limit=limit)
    assert e.value.kind == "Usage" and f"query {nq - 1}" in str(e.value)
    again = ix.rank(qs, offset=offset, limit=limit)
    assert all(np.array_equal(a[0], h[0]) for a, h in zip(again, host))
