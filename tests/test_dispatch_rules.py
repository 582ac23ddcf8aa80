"""Dispatch rules that the library answers on the host: each is held to a model
of its launch and to the points at which both sides were measured."""
from __future__ import annotations

import pytest


@pytest.fixture(scope="module")
def lib():
    from rwkv7mi import _lib

    return _lib.load()


def _cd(a, b):
    return -(-a // b)


def _prefill_splits(lib, k, rows, I, O):
    part = lib.rwkv7mi_mm8t_gemm_prefill_split_ws_bytes(k, rows, I, O) - lib.rwkv7mi_mm8t_gemm_prefill_ws_bytes(k, I, O)
    return max(1, part // (k * rows * _cd(O, 32) * 32 * 4))


def _fullest_xcd(rows, O):
    """256 x 256 tiles on the fullest of the eight XCDs: groups of 4 x 8 tiles,
    padded to whole groups, each XCD a contiguous eighth of their order."""
    mt, nt = _cd(rows, 256), _cd(O, 256)
    gm, gn = min(mt, 4), min(nt, 8)
    order = [(m, c) for m0 in range(0, mt, gm) for c0 in range(0, nt, gn)
             for m in range(m0, m0 + gm) for c in range(c0, c0 + gn)]
    per = _cd(len(order), 8)
    return max(sum(m < mt and c < nt for m, c in order[x * per:(x + 1) * per]) for x in range(8))


@pytest.mark.parametrize("k", [1, 2, 3])
@pytest.mark.parametrize("I,O", [(8192, 2048), (2048, 2048), (10240, 2560), (2560, 2560), (16384, 4096), (4096, 4096),
                                 (4096, 1000), (3072, 768), (2560, 10240)])
def test_prefill_splits_shorten_the_fullest_xcd(lib, k, I, O):
    """A K split is taken where the steps that the fullest XCD's CUs run one
    after the other fall by a sixth or more; 32 CUs an XCD."""
    steps = I // 64
    for rows in (257, 300, 513, 768, 1025, 1100, 1281, 1500, 1537, 2304, 2500, 3000, 3072, 4000, 6000):
        S = _prefill_splits(lib, k, rows, I, O)
        if S > 1:
            most = k * _fullest_xcd(rows, O)
            assert _cd(most * S, 32) * _cd(steps, S) <= 5 / 6 * _cd(most, 32) * steps, (rows, S)


def test_prefill_splits_at_measured_points(lib):
    assert _prefill_splits(lib, 1, 2500, 10240, 2560) == 1  # 262 us in two, 199 in one
    assert _prefill_splits(lib, 1, 1025, 8192, 2048) == 4   # 114 us in five (two rounds), 84.6 in four
    assert _prefill_splits(lib, 1, 1100, 4096, 4096) == 2   # 104.6 us in three, 83.8 in two


@pytest.mark.parametrize("k,rows,I,O,pays", [
    (3, 1000, 2048, 2048, 0),    # 64 us, 58 on the dequantised weight
    (3, 512, 2048, 2048, 1), (1, 1000, 2048, 8192, 1), (1, 768, 16384, 4096, 1), (3, 600, 4096, 4096, 1),
    (1, 600, 4096, 16384, 0),    # two rounds of its tiles
])
def test_middle_row_kernel_against_the_prefill_gemm(lib, k, rows, I, O, pays):
    """Above 256 rows by the two estimates; an unsplit launch is priced with its own epilogue and pre-pass."""
    assert lib.rwkv7mi_mm8t_rows_pays(k, rows, I, O, 1) == pays


def test_middle_row_kernel_splits_before_it_runs_an_epilogue(lib):
    """2048 -> 8192 at 512 rows: 53.7 us unsplit, 41.8 in two K ranges."""
    x = 512 * 2048 * 2 + 512 * 16
    assert lib.rwkv7mi_mm8t_rows_workspace_bytes(1, 512, 2048, 8192) >= x + 2 * 512 * 8192 * 4


@pytest.mark.parametrize("rows,I,O,pays", [
    (128, 8192, 4096, 0), (128, 4096, 8192, 0),     # 31.0 and 32.2 us; 28.5 and 29.6 on the 64-row tiles
    (129, 8192, 4096, 1), (256, 4096, 8192, 1),     # 33.0 and 38.4 us; 38.8 and 45.5
    (65, 10240, 4096, 1), (128, 16384, 4096, 1),    # 29.1 and 42.0 us; 40.2 and 44.0
    (64, 16384, 4096, 0), (200, 2560, 10240, 0),
])
def test_middle_row_kernel_against_the_64_row_tiles(lib, rows, I, O, pays):
    assert lib.rwkv7mi_mm8t_rows_pays(1, rows, I, O, 1) == pays


@pytest.mark.parametrize("rows,I,O,aff,dt,split", [
    (128, 1024, 1024, 0, 1, True), (512, 2048, 2048, 0, 1, True),      # 16.6 and 28.1 us unsplit, 11 and 20 split
    (96, 2048, 8192, 1, 2, True),                                      # 46.9 us unsplit, 24.6 split
    (128, 768, 768, 0, 1, False),                                      # six blocks: 13.8 us in one launch
    (384, 4096, 16384, 0, 1, False), (1000, 4096, 4096, 0, 1, False),  # the tiles fill the chip
])
def test_w4_splits(lib, rows, I, O, aff, dt, split):
    assert (lib.rwkv7mi_w4_workspace_bytes(rows, O, I, 128, aff, dt) > 0) is split


@pytest.mark.parametrize("rows,I,O,aff,dt,few", [
    (17, 4096, 4096, 0, 1, True), (32, 2048, 8192, 0, 1, True), (17, 2560, 2560, 1, 2, True), (64, 2048, 2048, 0, 1, True),
    (17, 4096, 4096, 0, 2, False), (17, 4096, 16384, 0, 1, False), (33, 4096, 4096, 0, 1, False), (65, 2048, 2048, 0, 1, False),
])
def test_w4_few_rows_of_small_weights_take_no_scratch(lib, rows, I, O, aff, dt, few):
    """They run on the 64-row launches of the GEMV's kernel; the others here split K."""
    assert (lib.rwkv7mi_w4_workspace_bytes(rows, O, I, 128, aff, dt) == 0) is few


@pytest.mark.parametrize("B,T,H,two", [
    (1, 256, 48, 1), (1, 8192, 48, 1), (1, 240, 12, 0), (1, 288, 64, 0), (2, 320, 32, 0), (5, 400, 12, 1),
    (1, 1000, 64, 1), (2, 4096, 32, 1), (2, 1000, 40, 0),
])
def test_scan_takes_the_two_kernel_form(lib, B, T, H, two):
    """One launch wins again where 49 to 64 heads meet few chunks (64 heads: 320
    tokens 30.2 us against 31.8) and, by type, very many."""
    assert (lib.rwkv7mi_wkv7_chunk_workspace_bytes(B, T, H) > 0) == bool(two)
