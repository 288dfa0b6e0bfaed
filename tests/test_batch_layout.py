"""Layouts of the batched scoring's scratch (mars::batch_grid), on the CPU: its size is bounded over every
batch size and row count, a growing graph's scratch is allocated a bounded number of times, and an insert's
search keeps to its share of the chip."""
from __future__ import annotations

import ctypes as C

import pytest

from mars_amd import _lib

SCORE_WORDS = 6 << 20             # the most 64-bit words of a layout that keeps every row's score (48 MiB)
LISTS = 256 * 16                  # the most of a query's lists: 256 ranges of 16


class Grid(C.Structure):
    _fields_ = [("n_rranges", C.c_int32), ("n_qblocks", C.c_int32), ("rows_per_range", C.c_int64), ("part", C.c_int64),
                ("scores", C.c_int32)]


def check(g, n, q, kp):
    assert g.n_qblocks == (q + 63) // 64
    assert g.n_rranges * g.rows_per_range >= n and (g.n_rranges - 1) * g.rows_per_range < n
    assert g.part == g.n_qblocks * 64 * g.n_rranges * (8 if g.scores else kp)
    assert g.rows_per_range == 16 or not g.scores
    return g


@pytest.fixture(scope="module")
def so():
    so = C.CDLL(str(_lib.LIB_PATH))
    so._ZN4mars10batch_gridElibiib.restype = Grid
    so._ZN4mars11insert_gridEli.restype = Grid
    so._ZN4mars15batch_part_roomEll.restype = C.c_int64
    return so


def grid(so, n, q, plain, kp, rq64=False, cap=256):
    return check(so._ZN4mars10batch_gridElibiib(C.c_int64(n), C.c_int32(q), C.c_bool(plain), C.c_int32(kp), C.c_int32(cap),
                                                C.c_bool(rq64)), n, q, kp)


ROWS = [1, 15, 16, 17, 1024, 1025, 1400, 1537, 4096, 6307, 12_288, 12_289, 20_000, 24_576, 45_056, 45_057, 300_007,
        1_000_000, 13_000_000]


@pytest.mark.parametrize("kp", [8, 16])
@pytest.mark.parametrize("plain", [False, True])
@pytest.mark.parametrize("q", [1, 64, 65, 128, 256, 512, 700, 1023, 1024, 4096, 65_536, 100_000, 1_000_000])
def test_scratch_is_bounded(so, q, plain, kp):
    for n in ROWS:
        for rq64 in ([False, True] if q <= 64 else [False]):
            g = grid(so, n, q, plain, kp, rq64)
            assert g.part <= (SCORE_WORDS if g.scores else g.n_qblocks * 64 * LISTS), (n, q, plain, kp)
            assert g.n_rranges <= 256 or g.scores


# products that once kept a key of every row, whatever their size; and the largest that keep scores
@pytest.mark.parametrize("q,n,scores", [(100_000, 1400, 0), (1_000_000, 1400, 0), (65_536, 1535, 0), (256, 45_056, 1),
                                        (512, 22_528, 1), (1023, 11_264, 1), (2000, 11_264, 0)])
def test_large_products_keep_lists(so, q, n, scores):
    assert grid(so, n, q, False, 16).scores == scores


def test_growing_graph_allocates_a_few_times(so):
    held, times = 0, 0
    for n in range(100, 46_000, 16):
        need = grid(so, n, 128, False, 16).part
        if need > held:
            held, times = so._ZN4mars15batch_part_roomEll(C.c_int64(held), C.c_int64(need)), times + 1
            assert need <= held <= max(SCORE_WORDS, need)
    assert times <= 12


@pytest.mark.parametrize("q", [1, 64, 65, 128, 200, 900, 1023, 1024])
def test_inserts_keep_to_a_quarter_of_the_chip(so, q):
    """At most 64 ranges per query group, whose buffer does not grow with the graph."""
    for n in ROWS:
        g = check(so._ZN4mars11insert_gridEli(C.c_int64(n), C.c_int32(q)), n, q, 16)
        assert g.n_rranges <= (64 if n <= 2_000_000 else 256), (n, q, g.n_rranges)


# up to 64 queries: rows, row length, results, one time
@pytest.mark.parametrize("q,n,d,k,uniform,rq", [
    (64, 45_056, 768, 16, False, True), (64, 45_057, 768, 16, False, False), (1, 32_768, 256, 8, False, True),
    (1, 32_769, 256, 8, True, False), (64, 1_000_000, 768, 8, True, False), (64, 13_000_000, 768, 9, True, True),
    (1, 1 << 19, 256, 10, True, True), (1, (1 << 19) + 1, 256, 10, True, False), (33, 1 << 20, 512, 10, True, True),
    (33, (1 << 20) + 1, 384, 10, True, False), (65, 1000, 768, 10, True, False)])
def test_small_batches_take_the_faster_kernel(so, q, n, d, k, uniform, rq):
    f = so._ZN4mars14batch_small_rqEiliib
    f.restype = C.c_bool
    assert f(C.c_int32(q), C.c_int64(n), C.c_int32(d), C.c_int32(k), C.c_bool(uniform)) == rq
