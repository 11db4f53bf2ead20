# SPDX-License-Identifier: Apache-2.0
"""The rules that pick a kernel by a call's sizes (csrc/dsv4_choose.h),
compiled for the host: the forms that were measured to be the faster ones, and
the forms that the GPU tests of the kernels rely on reaching."""
import ctypes as C
import os
import subprocess

import pytest

from conftest import PKG_DIR

SHIM = """
#include "dsv4_choose.h"
using namespace dsv4;
extern "C" {
int c_gemm_mid_tile(int M, int N, int K) { return gemm_mid_tile(M, N, K); }
int c_dense8_tile(int M, long slabs) { long c = 0; return dense8_tile(M, slabs, &c); }
int c_mmq_takes_seam(int nt, int rows, int cols) { return mmq_takes_seam(nt, rows, cols, true); }
int c_grouped_form(long pairs, int ne, int hidden, int inter, int stream)
{ return grouped_form(pairs, ne, hidden, inter, stream != 0); }
int c_grouped_splits(long pairs, int form, int hidden, int inter) { return grouped_splits(pairs, form, hidden, inter); }
long c_grouped_fat_tiles(long pairs) { return grouped_fat_tiles(pairs); }
int c_fat(int which) { return which ? GROUPED_FAT_MIN : GROUPED_FAT_ROWS; }
int c_mx_wide_k(int K) { return mx_wide_k(K); }
int c_bf16_form(int rows, int cols, int nt) { return bf16_form(rows, cols, nt); }
}
"""
STREAM = 5
SMALL, ROWS, GEMM, WAVE = 1, 2, 3, 4


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("choice")
    src, so = d / "shim.cpp", d / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I",
                    os.path.join(PKG_DIR, "csrc"), str(src), "-o", str(so)], check=True)
    lib = C.CDLL(str(so))
    lib.c_dense8_tile.argtypes = [C.c_int, C.c_long]
    lib.c_grouped_splits.argtypes = [C.c_long, C.c_int, C.c_int, C.c_int]
    lib.c_grouped_fat_tiles.argtypes, lib.c_grouped_fat_tiles.restype = [C.c_long], C.c_long
    lib.c_grouped_form.argtypes = [C.c_long, C.c_int, C.c_int, C.c_int, C.c_int]
    return lib


@pytest.mark.parametrize("tokens,rows,cols,tile", [
    (8, 1024, 4096, 2), (300, 1024, 4096, 2), (300, 4096, 4096, 4), (700, 4096, 4096, 8), (1500, 4096, 4096, 0),
    (300, 1024, 8320, 0),                                  # more weight scales than a register holds
])
def test_gemm_tile(rules, tokens, rows, cols, tile):
    assert rules.c_gemm_mid_tile(tokens, rows, cols) == tile


@pytest.mark.parametrize("tokens,rows,tile", [(77, 4096, 1), (333, 4096, 3), (700, 4096, 6)])
def test_dense_tile(rules, tokens, rows, tile):
    assert rules.c_dense8_tile(tokens, rows // 128) == tile


@pytest.mark.parametrize("tokens,rows,cols,seam", [
    (1500, 4096, 4096, 0), (2000, 4096, 4096, 1), (2048, 1024, 4096, 0), (500, 15360, 4096, 1), (333, 4096, 4096, 0),
    (3708, 1280, 384, 1), (1751, 15360, 640, 1), (1737, 10240, 768, 1), (2059, 4352, 512, 1), (3000, 2048, 128, 1),
    (2803, 3072, 640, 1),
    (1000, 1280, 128, 0), (2000, 1280, 2048, 0),
])
def test_many_token_matmul(rules, tokens, rows, cols, seam):
    assert rules.c_mmq_takes_seam(tokens, rows, cols) == seam


@pytest.mark.parametrize("rows,cols,tokens", [(3200, 256, 1280), (2432, 512, 1337), (2560, 1280, 1700), (2048, 128, 4096),
                                              (2176, 640, 2050), (4224, 384, 1337)])
def test_shapes_of_the_seam_tests(rules, rows, cols, tokens):
    """The seam GEMM's GPU tests run it, and dense tiles beside it."""
    assert rules.c_mmq_takes_seam(tokens, rows, cols) and not rules.c_mmq_takes_seam(500, rows, cols)


def test_dense_tile_heights_of_the_seam_tests(rules):
    """Every height among the cases of the same-bits test."""
    cases = {(2048, 128): (32, 33, 129, 257, 300, 513, 600, 1000, 1290), (2176, 640): (32, 47, 300, 500, 700, 1290),
             (4224, 384): (40, 500, 700)}
    heights = {rules.c_dense8_tile(n, r // 128) for (r, c), ns in cases.items() for n in ns if not rules.c_mmq_takes_seam(n, r, c)}
    assert heights == {1, 2, 3, 4, 6}
    assert not rules.c_mmq_takes_seam(1290, 2560, 1280)
    assert [rules.c_dense8_tile(n, 32) for n in (150, 96)] == [2, 1]


@pytest.mark.parametrize("tokens,experts,hidden,inter,form", [
    (7, 256, 4096, 2048, STREAM), (64, 256, 4096, 2048, STREAM), (701, 256, 4096, 2048, STREAM),
    (1500, 256, 4096, 2048, 8), (60, 64, 4096, 512, 1), (700, 64, 4096, 512, 8),
])
def test_expert_tiles_top6(rules, tokens, experts, hidden, inter, form):
    assert rules.c_grouped_form(6 * tokens, experts, hidden, inter, 1) == form


@pytest.mark.parametrize("pairs,experts,hidden,inter,form", [
    (50, 1, 4096, 2048, STREAM), (400, 1, 4096, 2048, STREAM), (200, 2, 4096, 2048, STREAM), (400, 4, 4096, 2048, STREAM),
    (1600, 1, 4096, 2048, 8), (1120, 8, 4096, 2048, 8), (3200, 16, 4096, 2048, 8),
    (100, 1, 2048, 512, 1), (800, 1, 2048, 512, 1), (400, 8, 2048, 512, 1), (800, 2, 512, 512, 1),
    (4097, 1, 512, 512, 8),                                # past GROUPED_FEW_PAIRS
    (3200, 64, 4096, 2048, 8), (2240, 32, 2048, 512, 8),   # tiles enough for every CU
    (1100, 64, 4096, 512, 1), (2048, 64, 4096, 512, 1), (2100, 64, 4096, 512, 8), (4096, 128, 2048, 512, 1),   # short rows
    (4800, 256, 2048, 512, 8), (4800, 512, 2048, 512, 1),
])
def test_expert_tiles_few_experts(rules, pairs, experts, hidden, inter, form):
    """A few experts' 128-row tiles leave the device idle: 16-row tiles until
    there are pairs enough."""
    assert rules.c_grouped_form(pairs, experts, hidden, inter, 1) == form


def test_large_buckets_leave_the_16_row_tiles(rules):
    """Above 4,096 pairs, whatever the mean bucket: 6,000 pairs may sit on 8 of
    256 experts."""
    for pairs, experts, inter in ((4206, 256, 2048), (6000, 256, 2048), (7168, 256, 2048), (8000, 512, 512)):
        form = rules.c_grouped_form(pairs, experts, 4096, inter, 1)
        assert form in (1, STREAM) and rules.c_grouped_splits(pairs, form, 4096, inter)
    assert not rules.c_grouped_splits(4096, STREAM, 4096, 2048)
    assert not rules.c_grouped_splits(9000, 8, 4096, 2048)
    assert not rules.c_grouped_splits(6000, STREAM, 1024, 1024)      # small experts: from the caches


def test_fat_tile_bound(rules):
    """The room for the large buckets' tile records holds their tiles, whatever
    the buckets: each bucket's alone, and the one that fits least."""
    rows, least = rules.c_fat(0), rules.c_fat(1)
    worst = min(range(least + 1, 40 * rows), key=lambda c: c / -(-c // rows))
    for c in range(least + 1, 40 * rows):
        for m in (1, 7):                       # m buckets of c rows and one of the worst kind
            assert m * -(-c // rows) + -(-worst // rows) <= rules.c_grouped_fat_tiles(m * c + worst)


@pytest.mark.parametrize("cols,wide", [(512, 0), (1024, 0), (1536, 0), (2048, 1), (2304, 0), (2560, 1), (4096, 1)])
def test_mx_scales_four_stages_at_a_time(rules, cols, wide):
    """Only rows long enough for the wide form's start, and of whole groups."""
    assert rules.c_mx_wide_k(cols) == wide


@pytest.mark.parametrize("rows,cols,tokens,form", [
    (256, 4096, 1, SMALL), (256, 4096, 8, SMALL), (129280, 4096, 1, ROWS), (16384, 4096, 4, ROWS), (4096, 4096, 4, GEMM),
    (256, 4096, 700, GEMM),
    (8553, 440, 1, WAVE), (103825, 232, 1, WAVE), (8137, 2024, 1, WAVE), (5492, 544, 2, WAVE), (2048, 136, 1, WAVE),
    (16384, 2024, 1, ROWS), (8192, 2056, 1, SMALL), (1024, 440, 1, SMALL), (16384, 768, 2, ROWS), (4096, 440, 2, SMALL),
    (12000, 64, 3, ROWS), (12000, 136, 3, GEMM),
])
def test_bf16_form(rules, rows, cols, tokens, form):
    assert rules.c_bf16_form(rows, cols, tokens) == form
