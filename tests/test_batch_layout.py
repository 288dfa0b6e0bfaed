"""Layouts of the batched scoring's partial keys (mars::batch_grid), on the CPU: their number is bounded over
every batch size and row count, a growing graph's scratch is allocated a bounded number of times, and an
insert's search keeps to its share of the chip."""
from __future__ import annotations

import ctypes as C

import pytest

from mars_amd import _lib

ALL_KEYS = 6 << 20                # the most keys of a layout that keeps every row's (48 MiB)
LISTS = 256 * 16                  # the most of a query's lists: 256 ranges of 16


@pytest.fixture(scope="module")
def so():
    so = C.CDLL(str(_lib.LIB_PATH))
    so._ZN4mars10batch_gridElibPiS0_Pliib.restype = None
    so._ZN4mars15batch_part_roomEll.restype = C.c_int64
    return so


def grid(so, n, q, plain, kp, rq64=False, cap=256):
    rr, qb, rows = C.c_int32(), C.c_int32(), C.c_int64()
    so._ZN4mars10batch_gridElibPiS0_Pliib(C.c_int64(n), C.c_int32(q), C.c_bool(plain), C.byref(rr), C.byref(qb),
                                          C.byref(rows), C.c_int32(cap), C.c_int32(kp), C.c_bool(rq64))
    assert qb.value == (q + 63) // 64 and rr.value * rows.value >= n and (rr.value - 1) * rows.value < n
    return rr.value, rows.value, qb.value * 64 * rr.value * kp


ROWS = [1, 15, 16, 17, 1400, 1537, 4096, 6307, 12_288, 12_289, 20_000, 45_056, 45_057, 300_007, 1_000_000, 13_000_000]


@pytest.mark.parametrize("kp", [8, 16])
@pytest.mark.parametrize("plain", [False, True])
@pytest.mark.parametrize("q", [1, 64, 65, 128, 256, 512, 700, 1023, 1024, 4096, 65_536, 100_000, 1_000_000])
def test_partial_keys_are_bounded(so, q, plain, kp):
    padded = (q + 63) // 64 * 64
    for n in ROWS:
        for rq64 in ([False, True] if q <= 64 else [False]):
            rr, rows, keys = grid(so, n, q, plain, kp, rq64)
            # the ranges of a batch this large without its keys kept
            lists = padded * kp * grid(so, n, q, plain, 0)[0]
            assert lists <= padded * LISTS
            assert keys <= max(ALL_KEYS, lists), (n, q, plain, kp, keys)


# the sizes that kept up to eleven times the keys of the lists, without a bound
@pytest.mark.parametrize("q,n", [(256, 45_056), (100_000, 1400), (1_000_000, 1400), (65_536, 1535)])
def test_large_products_keep_lists(so, q, n):
    rr, rows, keys = grid(so, n, q, False, 16)
    assert keys <= (q + 63) // 64 * 64 * LISTS and rows > 16 and rr <= 256


def test_growing_graph_allocates_a_few_times(so):
    held, times = 0, 0
    for n in range(100, 46_000, 16):
        need = grid(so, n, 128, False, 16)[2]
        if need > held:
            held, times = so._ZN4mars15batch_part_roomEll(C.c_int64(held), C.c_int64(need)), times + 1
            assert need <= held <= max(ALL_KEYS, need)
    assert times <= 12


@pytest.mark.parametrize("q", [1, 64, 65, 128, 200, 900, 1023, 1024])
def test_inserts_keep_to_a_quarter_of_the_chip(so, q):
    """At most 64 ranges per query group, whose buffer does not grow with the graph."""
    f = so._ZN4mars11insert_gridEliPiS0_Pl
    f.restype = None
    for n in ROWS:
        rr, qb, rows = C.c_int32(), C.c_int32(), C.c_int64()
        f(C.c_int64(n), C.c_int32(q), C.byref(rr), C.byref(qb), C.byref(rows))
        assert rr.value * rows.value >= n and (rr.value - 1) * rows.value < n
        assert rr.value <= (64 if n <= 2_000_000 else 256), (n, q, rr.value)
