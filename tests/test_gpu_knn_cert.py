"""Certified k-NN builds (mars_graph_knn / _range / _blocked and mars_graph_knn_report).

Bars:
  * every list of an all-pairs build is exact: the k-NN of 2,000 sampled nodes of the
    100K benchmark corpus (and 1,000 of a 150K one, whose row ranges take the sampled
    floors) equal the fp64 oracle's up to near-ties (1e-5), and the report says that every
    node the certificate missed was scanned again exactly;
  * rows whose neighbours tie (80 copies of one row) miss the certificate, are scanned
    again, and their lists hold copies of the row (score 1, the node itself excluded);
  * a build within blocks counts the nodes the certificate missed and scans none again;
  * the range builder in pieces reports the same lists as the one-call build.
"""
from __future__ import annotations

import numpy as np
import pytest

import mars_amd
import oracle
from mars_amd import corpus

pytestmark = pytest.mark.gpu
D = 768


def device_graph(emb, mods, ts):
    g = mars_amd.MemoryGraph(len(mods), emb.shape[1], None, None, emb, mods, ts)
    dg = mars_amd.upload_to_device(g)
    mars_amd.upload_fp16_embeddings(dg)
    return dg


def check_lists(emb, nodes, got, k=8):
    want, sims = oracle.knn(emb, np.asarray(nodes, np.int32), k)
    e = emb.astype(np.float64)
    for i, node in enumerate(nodes):
        assert len(set(got[i].tolist())) == k and node not in got[i], (node, got[i])
        for j in set(got[i].tolist()) ^ set(want[i].tolist()):
            s = float(e[node] @ e[j])
            assert abs(s - sims[i, k - 1]) <= 1e-5, (node, j, s, sims[i, k - 1])


def test_all_pairs_100k_exact():
    c = corpus.make_corpus(100_000, D, seed=2026, threads=16)
    dg = device_graph(c.embeddings, c.modalities, c.timestamps)
    try:
        got = mars_amd.graph_knn(dg, 8)
        u, r = dg.knn_report
        print(f"100K all-pairs 8-NN: {u} lists uncertified, {r} scanned again")
        assert r == u and u <= 1000
        nodes = np.random.default_rng(5).choice(100_000, 2000, replace=False)
        check_lists(c.embeddings, nodes, got[nodes])
        # in pieces of 30,000 query nodes: the same lists
        got2 = mars_amd.graph_knn(dg, 8, progress=lambda *_: None, piece=30_000)
        np.testing.assert_array_equal(got2, got)
        assert dg.knn_report == (u, r)
    finally:
        mars_amd.free_device(dg)


def test_all_pairs_150k_with_floors_exact():
    """150,000 nodes: row ranges of 2,560 rows, long enough for the sampled pass, so
    k_batch_mm's thresholds start from its floors; 1,000 sampled nodes against the fp64
    oracle, up to near-ties, and every list the certificate missed scanned again."""
    c = corpus.make_corpus(150_000, D, seed=2027, threads=16)
    dg = device_graph(c.embeddings, c.modalities, c.timestamps)
    try:
        got = mars_amd.graph_knn(dg, 8)
        u, r = dg.knn_report
        assert r == u and u <= 1500
        nodes = np.random.default_rng(6).choice(150_000, 1000, replace=False)
        check_lists(c.embeddings, nodes, got[nodes])
    finally:
        mars_amd.free_device(dg)


def test_knn_range_2_2m_multi_tile_floors_exact():
    """2,200,000 nodes: row ranges of 34,560 rows, whose sampled pass covers 528 rows
    (three tiles, the last one partial), so k_batch_mm's floors come from block maxima kept
    over several tiles. The 2,048 query nodes start at range 28's first row, so 528 of them
    have their own row among the sampled rows. 100 of them against the fp64 oracle, up to
    near-ties."""
    n = 2_200_000
    c = corpus.make_corpus(n, D, seed=2028, threads=16)
    dg = device_graph(c.embeddings, c.modalities, c.timestamps)
    try:
        first = 28 * 34_560
        got = mars_amd.graph_knn_range(dg, 8, first, 2048)
        u, r = mars_amd.graph_knn_report(dg)
        assert r == u and u <= 20
        idx = np.sort(np.concatenate([np.arange(0, 528, 11), np.random.default_rng(7).choice(np.arange(528, 2048), 52, replace=False)]))
        check_lists(c.embeddings, first + idx, got[idx])
    finally:
        mars_amd.free_device(dg)


def test_tied_rows_are_scanned_again():
    c = corpus.make_corpus(6000, D, seed=17)
    emb = c.embeddings.copy()
    dups = np.arange(1000, 1080)                        # 80 copies of row 1000
    emb[dups] = emb[1000]
    dg = device_graph(emb, c.modalities, c.timestamps)
    try:
        got = mars_amd.graph_knn(dg, 8)
        u, r = dg.knn_report
        assert u >= 80 and r == u, (u, r)
        for node in dups:
            assert set(got[node].tolist()) <= set(dups.tolist()) - {int(node)}
        check_lists(emb, np.arange(0, 6000, 7), got[::7])
    finally:
        mars_amd.free_device(dg)


def test_blocked_build_counts_only():
    c = corpus.make_corpus(6000, D, seed=18)
    emb = c.embeddings.copy()
    emb[10:30] = emb[10]                                 # ties inside block 0
    dg = device_graph(emb, c.modalities, c.timestamps)
    try:
        got = mars_amd.graph_knn(dg, 8, block_rows=2000)
        u, r = dg.knn_report
        assert u >= 20 and r == 0, (u, r)
        for b in range(3):                              # lists stay inside their block
            assert np.all((got[2000 * b:2000 * (b + 1)] // 2000) == b)
    finally:
        mars_amd.free_device(dg)


def test_blocked_build_with_a_nan_row():
    """A row with a NaN (dots that no threshold test may drop or rank): its block's other lists
    are exact over the other rows, the row's own list is the block's first ids, the other block
    is untouched, and nothing is certified."""
    n, bad = 6000, 1700
    c = corpus.make_corpus(n, D, seed=19)
    emb = c.embeddings.copy()
    emb[bad, 5] = np.nan
    dg = device_graph(emb, c.modalities, c.timestamps)
    try:
        got = mars_amd.graph_knn(dg, 8, block_rows=3000)
        assert dg.knn_report == (n, 0)
        assert np.array_equal(got[bad], np.arange(8)) and not np.any(got == bad)
        nodes = np.setdiff1d(np.arange(0, 3000, 13), [bad])
        keep = np.setdiff1d(np.arange(3000), [bad])
        check_lists(c.embeddings[keep], np.searchsorted(keep, nodes), np.searchsorted(keep, got[nodes]))
        nodes = np.arange(3000, 6000, 13)
        check_lists(c.embeddings[3000:], nodes - 3000, got[nodes] - 3000)
    finally:
        mars_amd.free_device(dg)


# all-pairs sizes around the tile (256), the smallest MFMA build (1024 queries), the group
# splits over the XCDs (5, 10, 20 and 40 groups), and two launches (10,241); ranges whose
# groups do not divide evenly
@pytest.mark.parametrize("n, first, count", [(1024, 0, 0), (1025, 0, 0), (1281, 0, 0), (2561, 0, 0), (5121, 0, 0),
                                             (10_240, 0, 0), (10_241, 0, 0), (3000, 1400, 1600), (50_001, 7, 2_817),
                                             (50_001, 44_000, 6_001)])
def test_build_grids(n, first, count):
    c = corpus.make_corpus(n, 256, seed=n)
    dg = device_graph(c.embeddings, c.modalities, c.timestamps)
    try:
        got = mars_amd.graph_knn_range(dg, 8, first, count) if count else mars_amd.graph_knn(dg, 8)
        u, r = dg.knn_report if not count else mars_amd.graph_knn_report(dg)
        assert r == u and u <= max(4, len(got) // 100)
        idx = np.unique(np.r_[np.arange(0, len(got), 37), len(got) - 1])
        check_lists(c.embeddings, first + idx, got[idx])
    finally:
        mars_amd.free_device(dg)


@pytest.mark.parametrize("k", [1, 3, 4, 8, 15, 16])
def test_rescoring_that_stops_early_is_exact(k):
    """Rows spaced so that fp16 scores order some candidates wrongly (copies with perturbations
    near the fp16 step) among well separated ones: every list equals the oracle's, whether the
    rescoring ran through all 16 candidates or stopped after the first k."""
    c = corpus.make_corpus(2100, 512, seed=23)
    emb = c.embeddings.copy()
    rng = np.random.default_rng(24)
    for base in range(0, 2000, 50):
        e = emb[base] + rng.uniform(0, 6e-4, (20, 1)).astype(np.float32) * rng.standard_normal((20, 512)).astype(np.float32)
        emb[base + 1:base + 21] = e / np.linalg.norm(e, axis=1, keepdims=True)
    dg = device_graph(emb, c.modalities, c.timestamps)
    try:
        got = mars_amd.graph_knn(dg, k)
        u, r = dg.knn_report
        assert r == u
    finally:
        mars_amd.free_device(dg)
    s = emb.astype(np.float64) @ emb.astype(np.float64).T
    np.fill_diagonal(s, -np.inf)
    kth = np.sort(s, axis=1)[:, -k]
    took = np.take_along_axis(s, got, axis=1)
    assert np.all(took >= kth[:, None] - 1e-6)              # fp32 sums of 512 products of unit rows
    assert all(len(set(row)) == k for row in got.tolist())
