"""The rule that picks the int8 GEMMs' tile (lg_prefill_tile), on the CPU: where
each tile is taken, and that a tile is never taken for more rounds of longer
work than the wide ones need."""
import ctypes as C

import pytest

from ligguf_amd import lib as L


def tile(rows, cols, T, t=L.Q4_K):
    out = [C.c_int() for _ in range(3)]
    L.check(L.load().lg_prefill_tile(t, rows, cols, T, *(C.byref(o) for o in out)))
    return tuple(o.value for o in out)


@pytest.mark.parametrize("t", [L.Q2_K, L.Q3_K, L.Q4_K, L.Q5_K, L.Q6_K, L.Q8_0, L.Q1_0])
@pytest.mark.parametrize("cols", [4096, 12288])
@pytest.mark.parametrize("T", [257, 289, 320, 321, 353, 384, 385, 417, 448, 449, 512])
def test_wide_tile_that_fills_the_chip_once_stays(cols, T, t):
    """4096 rows: 128 x 64 with K in two is one round of the 256 CUs up to 512
    tokens; 64 x 32 tiles would take two and unpack each weight twice as often
    (Q5_K, 400 tokens: 58 us against 42)."""
    assert tile(4096, cols, T, t) == (128, 64, 2)


@pytest.mark.parametrize("rows,cols,T,want", [
    (24576, 4096, 512, (128, 64, 1)), (6144, 4096, 512, (128, 64, 1)), (6144, 4096, 200, (128, 64, 2)),
    (4096, 4096, 200, (64, 32, 2)), (4096, 12288, 200, (64, 32, 2)), (4096, 12288, 77, (64, 32, 4)),
    (4096, 12288, 16, (32, 32, 4)), (600, 2048, 96, (32, 32, 4))])
@pytest.mark.parametrize("t", [L.Q4_K, L.Q1_G])
def test_tile_by_shape(rows, cols, T, want, t):
    assert tile(rows, cols, T, t) == want


def test_tile_by_type():
    """the two tables: Q1_G rows cost about as much alone on a CU as in pairs"""
    assert tile(4096, 4096, 129) == (32, 32, 4) and tile(4096, 4096, 129, L.Q1_G) == (64, 32, 2)


@pytest.mark.parametrize("T", [1, 33, 100, 200, 512])
@pytest.mark.parametrize("rows", [33, 288, 768, 4096, 12288])
@pytest.mark.parametrize("cols", [32, 256, 288, 512])
@pytest.mark.parametrize("t", [L.Q8_0, L.Q1_G])
def test_narrow_matrices_take_no_empty_parts(rows, cols, T, t):
    """one or two steps of 256 values: at most two parts of K (a part of four
    would compute nothing and still load, hold LDS and be summed)"""
    assert tile(rows, cols, T, t)[2] <= 2


def test_bad_arguments():
    lib = L.load()
    o = C.c_int()
    for rows, cols, T in ((0, 256, 1), (32, 0, 1), (32, 256, 0)):
        assert lib.lg_prefill_tile(L.Q4_K, rows, cols, T, C.byref(o), C.byref(o), C.byref(o)) == -1
    assert lib.lg_prefill_tile(L.Q4_K, 32, 256, 1, None, C.byref(o), C.byref(o)) == -1
    for t in (L.F16, L.F32, 99):
        assert lib.lg_prefill_tile(t, 32, 256, 1, C.byref(o), C.byref(o), C.byref(o)) == -1
