"""GPU parity of k_batch_rq (batched scoring with 64, 128 or 256 queries per workgroup in
registers, 16-row tiles through LDS, a sampled score floor).

- against the fp32 oracle's top-K (the bar of tests/parity.py: scores within 2e-3 of the
  scale, id sets equal up to near-ties) at every supported width, both list sizes, with
  and without a modality filter, one or per-query times, ragged row counts;
- bit for bit against k_batch_scan, which computes the same MFMA products in the same order:
  mars_query_batch_static in blocks of 32 queries always takes it (scan_batch below);
- floors, lists, tiles with many and few passing rows, and the form that keeps every row's score;
- the neighbour-search form (plain dot products, the node itself excluded) against the
  exact CPU k-NN;
- the merge of the ranges' keys.
"""
from __future__ import annotations

import numpy as np
import pytest

import mars_amd
from mars_amd import RetrievalConfig, corpus

from parity import LAM, T_Q, Dev, batch_check, random_graph

pytestmark = pytest.mark.gpu


def static_batch(dg, qs, tq, cfg, uniform, block=None):
    """mars_query_batch_static in blocks of `block` queries; up to 64 of them take k_batch_scan."""
    out = []
    for j in range(0, len(qs), block or len(qs)):
        x, t = np.ascontiguousarray(qs[j:j + (block or len(qs))]), np.ascontiguousarray(tq[j:j + (block or len(qs))])
        bufs = [mars_amd.DeviceBuffer.from_array(x), mars_amd.DeviceBuffer.from_array(t),
                mars_amd.DeviceBuffer(len(x) * cfg.top_k * 4), mars_amd.DeviceBuffer(len(x) * cfg.top_k * 4)]
        mars_amd.query_batch_static(dg, bufs[0].ptr, len(x), bufs[1].ptr, cfg, bufs[2].ptr, bufs[3].ptr, uniform_tq=uniform)
        mars_amd.synchronize()
        out.append((bufs[2].to_array(np.int32, len(x) * cfg.top_k).reshape(len(x), -1),
                    bufs[3].to_array(np.float32, len(x) * cfg.top_k).reshape(len(x), -1)))
        for b in bufs:
            b.free()
    return np.concatenate([o[0] for o in out]), np.concatenate([o[1] for o in out])


def scan_batch(dg, qs, tq, cfg, uniform):
    """The same queries by k_batch_scan (no floor; uniform: one decay weight per row)."""
    return static_batch(dg, qs, tq, cfg, uniform, 32)


@pytest.mark.parametrize("d,q,k,filt,uniform", [(256, 129, 5, -1, True), (384, 200, 16, 1, False),
                                                 (512, 256, 8, 2, True), (768, 300, 10, -1, False),
                                                 (768, 520, 16, 0, True), (256, 1000, 3, -1, True),
                                                 (768, 65, 10, -1, True), (384, 96, 16, 2, False),
                                                 (512, 100, 8, -1, False), (768, 128, 16, 1, True)])
def test_rq_against_oracle(d, q, k, filt, uniform, rng):
    n = 3001                                   # ragged: not a multiple of the 16-row tile
    emb, mods, ts, row, col, _ = random_graph(rng, n, d)
    dev = Dev(emb, mods, ts, row, col, fp16=True)
    try:
        qn = rng.choice(n, q, replace=False)
        tq = np.float32(T_Q) if uniform else rng.uniform(300, 600, q).astype(np.float32)
        batch_check(dev, qn, RetrievalConfig(top_k=k, time_decay_lambda=LAM, modality_filter=filt), tq, emb)
    finally:
        dev.close()


@pytest.mark.parametrize("q,k,filt,uniform", [(256, 10, -1, True), (256, 5, 1, False), (128, 16, 2, True),
                                               (96, 10, -1, False)])
def test_rq_equals_scan_bit_for_bit(q, k, filt, uniform, rng):
    n, d = 20000, 768
    emb, mods, ts, row, col, _ = random_graph(rng, n, d)
    dev = Dev(emb, mods, ts, row, col, fp16=True)
    qs = np.ascontiguousarray(emb[rng.choice(n, q, replace=False)])
    tq = np.full(q, T_Q, np.float32) if uniform else rng.uniform(300, 600, q).astype(np.float32)
    cfg = RetrievalConfig(top_k=k, time_decay_lambda=LAM, modality_filter=filt)
    buf = mars_amd.DeviceBuffer.from_array(qs)
    try:
        ids, sc = mars_amd.query_batch(dev.dg, dev.ctx, buf.ptr, q, tq, cfg)                  # k_batch_rq
        want_ids, want_sc = scan_batch(dev.dg, qs, tq, cfg, uniform)
    finally:
        buf.free()
        dev.close()
    np.testing.assert_array_equal(ids, want_ids)
    np.testing.assert_array_equal(sc.view(np.uint32), want_sc.view(np.uint32))


def test_rq_sampled_floor(rng):
    """200K rows, 600 queries (three 256-query groups over 80 row ranges of 2,512 rows):
    each range's first tiles are scored first and set the queries' floors."""
    n, d = 200_000, 256
    emb = rng.standard_normal((n, d)).astype(np.float32)
    emb /= np.linalg.norm(emb, axis=1, keepdims=True)
    mods = rng.integers(0, 3, size=n).astype(np.int32)
    ts = rng.uniform(0, 600, size=n).astype(np.float32)
    dev = Dev(emb, mods, ts, None, None, fp16=True)
    try:
        qn = rng.choice(n, 600, replace=False)
        ids, _ = batch_check(dev, qn[:600], RetrievalConfig(top_k=10, time_decay_lambda=LAM), T_Q, emb)
        assert np.all(ids[:, 0] >= 0)
        batch_check(dev, qn[:300], RetrievalConfig(top_k=16, time_decay_lambda=LAM, modality_filter=1), T_Q, emb)
    finally:
        dev.close()


@pytest.mark.parametrize("q,k,filt,uniform", [(600, 10, -1, True), (300, 16, 1, False), (600, 5, 2, False)])
def test_rq_sampled_floor_equals_scan_bit_for_bit(q, k, filt, uniform, rng):
    """The sampled floor drops no row that belongs in a list: on 200K rows (each 256-query
    group's ranges sampled for the floor), the batch's ids and score bits equal those of
    the same queries scored by k_batch_scan, which takes no floor, with a modality filter and
    with per-query times too."""
    n, d = 200_000, 256
    emb = rng.standard_normal((n, d)).astype(np.float32)
    emb /= np.linalg.norm(emb, axis=1, keepdims=True)
    mods = rng.integers(0, 3, size=n).astype(np.int32)
    ts = rng.uniform(0, 600, size=n).astype(np.float32)
    dev = Dev(emb, mods, ts, None, None, fp16=True)
    qs = np.ascontiguousarray(emb[rng.choice(n, q, replace=False)])
    tq = np.full(q, T_Q, np.float32) if uniform else rng.uniform(300, 600, q).astype(np.float32)
    cfg = RetrievalConfig(top_k=k, time_decay_lambda=LAM, modality_filter=filt)
    buf = mars_amd.DeviceBuffer.from_array(qs)
    try:
        ids, sc = mars_amd.query_batch(dev.dg, dev.ctx, buf.ptr, q, tq, cfg)                  # sampled floor
        want_ids, want_sc = scan_batch(dev.dg, qs, tq, cfg, uniform)
    finally:
        buf.free()
        dev.close()
    np.testing.assert_array_equal(ids, want_ids)
    np.testing.assert_array_equal(sc.view(np.uint32), want_sc.view(np.uint32))


def test_rq_sampled_floor_sparse_filter_and_neighbours(rng):
    """280K rows, 300 queries (two 256-query groups over 128 row ranges of 2,192 rows,
    sampled): a modality filter that keeps 1 row in 2,000 (the sampled rows hold fewer than
    K of them, so the floors are -FLT_MAX scores), and the neighbour-search form (plain dot
    products, self excluded) over the same sampled ranges."""
    n, d = 280_000, 256
    emb = rng.standard_normal((n, d)).astype(np.float32)
    emb /= np.linalg.norm(emb, axis=1, keepdims=True)
    mods = (rng.random(n) < 0.0005).astype(np.int32)
    ts = rng.uniform(0, 600, size=n).astype(np.float32)
    dev = Dev(emb, mods, ts, None, None, fp16=True)
    try:
        qn = rng.choice(n, 300, replace=False)
        batch_check(dev, qn, RetrievalConfig(top_k=10, time_decay_lambda=LAM, modality_filter=1), T_Q, emb)
        got = mars_amd.graph_knn_range(dev.dg, 8, 5000, 300)
    finally:
        dev.close()
    q = emb[5000:5300]
    s = q @ emb.T
    s[np.arange(300), 5000 + np.arange(300)] = -np.inf
    want = np.argsort(-s, axis=1, kind="stable")[:, :8]
    for i in range(300):
        if not np.array_equal(np.sort(got[i]), np.sort(want[i])):
            kth = s[i, want[i, 7]]
            for j in set(got[i].tolist()) ^ set(want[i].tolist()):
                assert abs(s[i, j] - kth) <= 1e-3, (i, j)
    assert np.all(got != 5000 + np.arange(300)[:, None])


def test_rq_neighbour_search(rng):
    """graph_knn_range over 300 nodes runs one batch of 300 plain queries (self excluded)."""
    n, d = 2500, 512
    emb, mods, ts, _, _, _ = random_graph(rng, n, d)
    dev = Dev(emb, mods, ts, None, None, fp16=True)
    try:
        got = mars_amd.graph_knn_range(dev.dg, 8, 100, 300)
    finally:
        dev.close()
    want, sims = corpus.knn_cpu(emb, 8)
    s = emb[100:400] @ emb.T
    for i in range(300):
        s[i, 100 + i] = -np.inf
        if not np.array_equal(got[i], want[100 + i]):
            for j in set(got[i].tolist()) ^ set(want[100 + i].tolist()):
                assert abs(s[i, j] - sims[100 + i, 7]) <= 1e-3, (i, j)
    assert np.all(got != np.arange(100, 400)[:, None])


# below 12 tiles for each of 256 workgroups every row's score is kept (10 rows to 45,056); from there
# on a floor and lists; 30 and 64 queries: the form of 64 per workgroup
@pytest.mark.parametrize("n", [10, 41, 4097, 12_289, 11 * 4096, 11 * 4096 + 1, 50_000])
@pytest.mark.parametrize("q,k,lam,uniform", [(70, 8, LAM, False), (130, 16, LAM, True), (256, 9, 0.0, False),
                                             (100, 16, -1e-3, False), (30, 7, LAM, True), (64, 16, LAM, True)])
def test_rq_floors_and_lists_equal_scan_bit_for_bit(n, q, k, lam, uniform, rng):
    """Rows that improve along every range (the sampled first tiles give weak floors, so tiles
    go through the dense and the sparse way in turn), 40 copies of one row (ties across ranges),
    rows of zeros and one NaN row: ids and score bits equal k_batch_scan's."""
    d = 256
    emb = rng.standard_normal((n, d)).astype(np.float32)
    emb /= np.linalg.norm(emb, axis=1, keepdims=True)
    base = emb[:8].mean(axis=0)
    emb += (np.linspace(0.0, 3.0, n, dtype=np.float32) % 0.4)[:, None] * base
    emb[rng.choice(n, min(n // 3, 40), replace=False)] = emb[n // 2]
    emb[n - 5:n - 2] = 0.0
    emb[n // 3, 7] = np.nan
    mods = rng.integers(0, 3, size=n).astype(np.int32)
    ts = rng.uniform(0, 600, size=n).astype(np.float32)
    dev = Dev(emb, mods, ts, None, None, fp16=True)
    pick = rng.choice(n, q, replace=n < q)
    pick[pick == n // 3] = 0
    qs = np.ascontiguousarray(emb[pick])
    tq = np.full(q, T_Q, np.float32) if uniform else rng.uniform(300, 600, q).astype(np.float32)
    cfg = RetrievalConfig(top_k=k, time_decay_lambda=lam, modality_filter=-1 if n % 2 else 1)
    buf = mars_amd.DeviceBuffer.from_array(qs)
    try:
        ids, sc = mars_amd.query_batch(dev.dg, dev.ctx, buf.ptr, q, tq, cfg)                  # k_batch_rq
        want_ids, want_sc = scan_batch(dev.dg, qs, tq, cfg, uniform)
    finally:
        buf.free()
        dev.close()
    np.testing.assert_array_equal(ids, want_ids)
    np.testing.assert_array_equal(sc.view(np.uint32), want_sc.view(np.uint32))


# one merge wave's 512 keys (32 ranges of 16, 64 of 8), more lists, ragged ones
@pytest.mark.parametrize("n", [5, 500, 512, 520, 1040, 4096, 9000])
@pytest.mark.parametrize("q,k", [(1, 1), (33, 8), (64, 16), (3, 9)])
def test_merge_of_few_and_many_keys(n, q, k, rng):
    """k_batch_merge on lists with equal keys' scores (60 copies of one row), whose cut lets more
    than 64 keys through, and on fewer keys than asked for: the oracle's top-K by (score, id)."""
    d = 256
    emb, mods, ts, _, _, _ = random_graph(rng, n, d)
    emb[: min(n, 60)] = emb[0]
    ts[:] = 0.0
    dev = Dev(emb, mods, ts, None, None, fp16=True)
    buf = mars_amd.DeviceBuffer.from_array(np.ascontiguousarray(np.repeat(emb[:1], q, axis=0)))
    try:
        ids, sc = mars_amd.query_batch(dev.dg, dev.ctx, buf.ptr, q, np.zeros(q, np.float32),
                                       RetrievalConfig(top_k=k, time_decay_lambda=0.0))
    finally:
        buf.free()
        dev.close()
    want = np.full(k, -1)
    want[: min(n, k)] = np.arange(min(n, k))                 # the copies, least ids first
    np.testing.assert_array_equal(ids, np.tile(want, (q, 1)))
    live = want >= 0
    assert np.all(sc[:, live] == sc[0, 0]) and abs(sc[0, 0] - 1.0) < 2e-3


@pytest.mark.parametrize("d", [256, 768])
@pytest.mark.parametrize("q,k,filt", [(1, 9, -1), (15, 16, 1), (17, 13, -1), (63, 10, 2)])
def test_small_uniform_batch_equals_scan_bit_for_bit(d, q, k, filt, rng):
    """Up to 64 queries of one time take k_batch_rq for more than 8 results; with one more query of another
    time the batch takes k_batch_scan (50,000 rows: more than are kept whole). Same ids and score bits."""
    n = 50_000
    emb, mods, ts, _, _, _ = random_graph(rng, n, d)
    emb[100:130] = emb[100]
    dev = Dev(emb, mods, ts, None, None, fp16=True)
    qs = np.ascontiguousarray(emb[np.r_[100, rng.choice(n, q, replace=False)]])
    tq = np.full(q + 1, T_Q, np.float32)
    tq[q] -= 50.0
    cfg = RetrievalConfig(top_k=k, time_decay_lambda=LAM, modality_filter=filt)
    buf = mars_amd.DeviceBuffer.from_array(qs)
    try:
        ids, sc = mars_amd.query_batch(dev.dg, dev.ctx, buf.ptr, q, tq[:q], cfg)
        ids2, sc2 = mars_amd.query_batch(dev.dg, dev.ctx, buf.ptr, q + 1, tq, cfg)
    finally:
        buf.free()
        dev.close()
    np.testing.assert_array_equal(ids, ids2[:q])
    np.testing.assert_array_equal(sc.view(np.uint32), sc2[:q].view(np.uint32))


@pytest.mark.parametrize("q,k,uniform", [(40, 8, True), (70, 10, False), (130, 16, False), (300, 5, True), (600, 16, False)])
def test_nan_query_with_sampled_floors(q, k, uniform, rng):
    """A query whose every score is NaN (which ranks below -inf) in a batch with floors (50,000 rows:
    at least 12 tiles per workgroup): its sampled rows set no floor, and it gets the least ids, as from
    a scan without floors; the other queries' answers stay. So does a node of a NaN row in a range of
    neighbour searches."""
    n, d = 50_000, 256
    emb, mods, ts, _, _, _ = random_graph(rng, n, d)
    bad = 20_000 + q // 2
    emb[bad, 9] = np.nan
    dev = Dev(emb, mods, ts, None, None, fp16=True)
    qs = np.ascontiguousarray(emb[rng.choice(20_000, q, replace=False)])
    tq = np.full(q, T_Q, np.float32) if uniform else rng.uniform(300, 600, q).astype(np.float32)
    cfg = RetrievalConfig(top_k=k, time_decay_lambda=LAM)
    try:
        out = []
        for at in (None, 2, q - 1):
            x = qs.copy()
            if at is not None:
                x[at, 3] = np.nan
            buf = mars_amd.DeviceBuffer.from_array(x)
            out.append(mars_amd.query_batch(dev.dg, dev.ctx, buf.ptr, q, tq, cfg))
            buf.free()
        knn = mars_amd.graph_knn_range(dev.dg, 8, 20_000, q)
    finally:
        dev.close()
    for at, (ids, sc) in zip((2, q - 1), out[1:]):
        np.testing.assert_array_equal(ids[at], np.arange(k))
        assert np.all(np.isnan(sc[at]))
        rest = np.arange(q) != at
        np.testing.assert_array_equal(ids[rest], out[0][0][rest])
        np.testing.assert_array_equal(sc[rest].view(np.uint32), out[0][1][rest].view(np.uint32))
    np.testing.assert_array_equal(knn[bad - 20_000], np.arange(8))


# ranges of 7 and 11 tiles, of more keys than are kept whole
@pytest.mark.parametrize("q,n,k,uniform", [(256, 24_700, 5, True), (256, 45_000, 16, False), (230, 28_001, 10, False)])
def test_static_short_ranges_equal_scan_bit_for_bit(q, n, k, uniform, rng):
    """Batches of the static entry point whose short ranges keep lists with a floor, against
    k_batch_scan: same ids and score bits."""
    d = 256
    emb, mods, ts, _, _, _ = random_graph(rng, n, d)
    emb[100:140] = emb[100]
    dev = Dev(emb, mods, ts, None, None, fp16=True)
    qs = emb[np.r_[100, rng.choice(n, q - 1, replace=False)]]
    tq = np.full(q, T_Q, np.float32) if uniform else rng.uniform(300, 600, q).astype(np.float32)
    cfg = RetrievalConfig(top_k=k, time_decay_lambda=LAM, modality_filter=-1 if uniform else 1)
    try:
        ids, sc = static_batch(dev.dg, qs, tq, cfg, uniform)
        ids2, sc2 = static_batch(dev.dg, qs, tq, cfg, uniform, 32)
    finally:
        dev.close()
    np.testing.assert_array_equal(ids, ids2)
    np.testing.assert_array_equal(sc.view(np.uint32), sc2.view(np.uint32))


# of more scores than are kept: ranges of 3 tiles (lists without a floor) and of 6 (with one)
@pytest.mark.parametrize("q,n,k,uniform", [(34_000, 380, 5, False), (34_000, 380, 16, True), (20_000, 700, 7, True),
                                           (20_000, 700, 12, False)])
def test_very_large_batches_of_few_rows(q, n, k, uniform, rng):
    """A batch too large for every row's score keeps lists in short ranges: ids and score bits of a part
    of its queries equal k_batch_scan's."""
    emb, mods, ts, _, _, _ = random_graph(rng, n, 256)
    emb[50:70] = emb[50]
    emb[n - 3, 1] = np.nan
    dev = Dev(emb, mods, ts, None, None, fp16=True)
    qs = emb[rng.integers(0, n - 3, q)]
    tq = np.full(q, T_Q, np.float32) if uniform else rng.uniform(300, 600, q).astype(np.float32)
    cfg = RetrievalConfig(top_k=k, time_decay_lambda=LAM, modality_filter=-1 if uniform else 2)
    buf = mars_amd.DeviceBuffer.from_array(np.ascontiguousarray(qs))
    try:
        ids, sc = mars_amd.query_batch(dev.dg, dev.ctx, buf.ptr, q, tq, cfg)
        part = np.unique(np.r_[0:256, rng.choice(q, 1000), q - 100:q])
        want_ids, want_sc = scan_batch(dev.dg, qs[part], tq[part], cfg, uniform)
    finally:
        buf.free()
        dev.close()
    np.testing.assert_array_equal(ids[part], want_ids)
    np.testing.assert_array_equal(sc[part].view(np.uint32), want_sc.view(np.uint32))
