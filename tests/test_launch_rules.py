"""The rules that pick a kernel by the sizes (csrc/launch_rules.h, plain C++), asked on the CPU: that the sizes of the GPU tests are
on the kernels these tests are about, and that dealing units out to the XCDs leaves none out."""
import ctypes
import shutil
import subprocess
from pathlib import Path

import pytest

import test_gpu_experts as G
from piper_amd import _lib

CUS = 256
GATE_UP, DOWN, DX, DX_TRANSPOSED, DH, DH_SCALED = range(6)
TILES, RUNS, RING, BIG = range(4)
SOURCE = """
#include "launch_rules.h"
using namespace pk_rules;
extern "C" {
int rows(int what, int64_t A, int64_t E, int64_t cols, int64_t K, int64_t cus) { return unit_rows((Product)what, A, E, cols, K, cus); }
int wgrad(int64_t A, int64_t H, int64_t I, int64_t E, int64_t n, int acc, int64_t cus) { return wgrad_kernel(A, H, I, E, n, acc != 0, cus); }
int run(int64_t A, int64_t E, int64_t tiles, int64_t per_cu) { return wgrad_run(A, E, tiles, per_cu); }
int64_t chunk(int64_t units, int64_t per_expert) { return deal_chunk(units, per_expert); }
int64_t blocks(int64_t units, int64_t chunk) { return dealt_blocks(units, chunk); }
int absent(int gate_up, int64_t A, int64_t E, int64_t rows, int64_t cols, int64_t k, int64_t cus) { return absent_rows_left_out(gate_up != 0, A, E, rows, cols, k, cus); }
int unit(int block, int chunk) { return dealt_unit(block, chunk); }
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("no g++")
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(SOURCE)
    csrc = Path(_lib.__file__).resolve().parent / "csrc"
    subprocess.run([gxx, "-std=c++17", "-O1", "-shared", "-fPIC", f"-I{csrc}", str(d / "rules.cpp"), "-o", str(d / "rules.so")], check=True,
                   timeout=120)
    lib = ctypes.CDLL(str(d / "rules.so"))
    i64 = ctypes.c_int64
    lib.rows.argtypes = [ctypes.c_int] + [i64] * 5
    lib.wgrad.argtypes = [i64] * 5 + [ctypes.c_int, i64]
    lib.run.argtypes = [i64] * 4
    lib.absent.argtypes = [ctypes.c_int] + [i64] * 6
    lib.chunk.argtypes = lib.blocks.argtypes = [i64, i64]
    lib.chunk.restype = lib.blocks.restype = i64
    return lib


def test_the_160_row_tests_are_on_160_row_units(rules):
    H, I, E, A = 768, 1024, 8, 21504
    assert rules.rows(GATE_UP, A, E, I // 128, H, CUS) == 160
    assert rules.rows(DOWN, A, E, H // 256, I, CUS) == 160
    assert rules.rows(DX, A, E, H // 256, I, CUS) == 160
    for H in (128, 256):
        assert rules.rows(GATE_UP, 64 * 260, 64, 1280 // 128, H, CUS) == 160
    assert [rules.rows(GATE_UP, E * 260, E, 1280 // 128, 2048, CUS) for E in (64, 16)] == [160, 128]


def test_units_of_the_other_heights(rules):
    """The benchmark's region: 128 experts 2048 x 768 with 256 and 1,024 rows each, and 64 rows."""
    assert [rules.rows(p, 128 * 256, 128, c, k, CUS) for p, c, k in ((GATE_UP, 6, 2048), (DOWN, 8, 768), (DX, 8, 768), (DH_SCALED, 3, 2048))] == \
        [160, 160, 160, 128]
    assert [rules.rows(p, 128 * 1024, 128, c, k, CUS) for p, c, k in ((GATE_UP, 6, 2048), (DOWN, 8, 768), (DX_TRANSPOSED, 8, 768), (DH, 3, 2048))] == \
        [160, 256, 256, 256]
    assert [rules.rows(p, 128 * 64, 128, c, k, CUS) for p, c, k in ((GATE_UP, 6, 2048), (DOWN, 8, 768), (DX, 8, 768))] == [128] * 3


def test_the_weight_gradient_tests_are_on_their_kernels(rules):
    want = [(RUNS, 1), (RUNS, 2), (RUNS, 4), (BIG, 1), (RING, 1), (RING, 1), (RUNS, 1), (RUNS, 1), (BIG, 1), (RUNS, 1), (RING, 1), (BIG, 1)]
    chunks = {6: 3, 7: 7, 8: 2}
    assert len(want) == len(G.RUN_CASES)
    for i, ((counts, H, I), (kernel, run)) in enumerate(zip(G.RUN_CASES, want)):
        A, E, tiles = sum(counts), len(counts), (H // 256) * (I // 256)
        assert rules.wgrad(A, H, I, E, 3, 0, CUS) == kernel, i
        assert rules.wgrad(A, H, I, E, 3, 1, CUS) == (RUNS if kernel == RING else kernel), i
        if kernel == RUNS:
            assert rules.run(A, E, tiles, E * tiles * 3 // CUS) == run, i
        if i in chunks:
            assert rules.chunk(E * tiles * 3 // run, tiles * 3 // run) == chunks[i], i


@pytest.mark.parametrize("units,per_expert", [(1, 1), (7, 1), (162, 18), (360, 45), (432, 27), (900, 75), (768, 24), (9216, 72), (1000003, 19)])
def test_every_unit_is_dealt_out_once(rules, units, per_expert):
    chunk = rules.chunk(units, per_expert)
    assert 1 <= chunk <= per_expert
    if units >= 128:
        assert units // (8 * chunk) >= 16          # chunks of an XCD
    blocks = rules.blocks(units, chunk)
    dealt = sorted(rules.unit(b, chunk) for b in range(blocks))
    assert dealt == list(range(blocks)) and blocks >= units


@pytest.mark.parametrize("gate_up,E,rows,col_tiles,k_tiles,want", [
    (1, 24, 8, 6, 32, True), (1, 96, 8, 8, 32, True), (1, 100, 8, 8, 32, False), (1, 128, 16, 12, 64, False),
    (0, 64, 8, 16, 48, True), (0, 80, 20, 16, 32, False), (0, 64, 32, 16, 48, True), (0, 64, 33, 16, 48, False),
    (0, 64, 8, 16, 12, True), (0, 64, 8, 16, 11, False), (0, 128, 16, 8, 32, True), (0, 128, 8, 12, 64, False),
])
def test_which_fp32_products_leave_out_absent_rows(rules, gate_up, E, rows, col_tiles, k_tiles, want):
    assert bool(rules.absent(gate_up, E * rows, E, 64, col_tiles, k_tiles, CUS)) == want
    if rows == 8 and want:
        assert rules.absent(gate_up, 3, E, 64, col_tiles, k_tiles, CUS) == 1      # fewer rows than experts
        assert rules.absent(gate_up, E * 17, E, 32, col_tiles, k_tiles, CUS) == 0
