"""The size rules of the automatic kernel choice (vela_amd/csrc/dispatch_rules.h), compiled with the host compiler:
shapes on both sides of each line, every one of them timed on both of the kernels it lies between."""
import ctypes
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
EXPORTS = """
#include "dispatch_rules.h"
extern "C" int x32_wide_tiles(int M, int N, int Kp) { return vk::x32_wide_tiles(M, N, Kp); }
extern "C" int stripe_shift_rows(int epi, int M, int N, int Kp) { return vk::stripe_shift_rows(vk::ShiftEpi(epi), M, N, Kp); }
extern "C" int norm_tiles(int gn, long long M, int RT, long long row_cap) {
    return vk::norm_tiles_per_block(M, RT, row_cap, gn ? vk::GN_APPLY_COST : vk::LNORM_COST);
}
extern "C" int attn_form(int Tkp) { const vk::AttnForm f = vk::attn_form(Tkp); return f.multi ? 0 : 10 * f.waves + f.tiles; }
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    (d / "rules.cpp").write_text(EXPORTS)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-I", str(ROOT / "vela_amd" / "csrc"), str(d / "rules.cpp"),
                    "-o", str(d / "rules.so")], check=True)
    return ctypes.CDLL(str(d / "rules.so"))


@pytest.mark.parametrize("M,N,K,wide", [
    (32768, 320, 1280, True), (24576, 320, 1280, True), (8192, 1280, 1280, True), (14400, 1280, 1280, True), (6144, 1280, 2560, True),
    (32768, 320, 640, True), (24576, 320, 640, True), (32768, 320, 320, True), (28672, 320, 320, True), (14336, 640, 512, True),
    (7168, 1280, 640, True),
    # slower on the wide tiles (64 x 128 / 64 x 320, us): shallow K ...
    (24576, 320, 64, False),       # 20.7 / 21.7
    (32768, 300, 64, False), (61440, 320, 160, False), (24576, 320, 320, False),   # 38.2 / 42.2 in 64-bit integers
    # ... and last rounds of several columns of tiles that are not full
    (14400, 1280, 64, False),      # 34.0 / 39.2
    (14400, 1280, 320, False),     # 44.3 / 49.4
    (14400, 1280, 640, False),     # 59.5 / 61.5
    (8192, 1280, 320, False),      # 41.1 / 42.9 in 64-bit integers
    (65536, 300, 320, False),
    # few tiles, padding columns
    (16384, 320, 1280, False), (24512, 320, 1280, False), (32768, 192, 1280, False),
])
def test_int32_rows_on_wide_tiles(rules, M, N, K, wide):
    assert bool(rules.x32_wide_tiles(M, N, K)) == wide


@pytest.mark.parametrize("epi,M,N,K,row_stationary", [
    (1, 32768, 2560, 320, True), (1, 4096, 2560, 320, True), (1, 3520, 2560, 320, True), (1, 6592, 2560, 320, True), (0, 32768, 320, 320, True),
    (0, 16384, 1280, 320, True), (0, 3136, 2560, 320, True), (0, 7040, 1280, 320, True), (0, 12352, 640, 320, True), (0, 20544, 320, 160, True),
    (0, 64000, 320, 320, True), (1, 65536, 256, 192, True),
    (0, 61568, 64, 320, True), (1, 38400, 640, 320, True), (1, 76083, 640, 304, True), (1, 30374, 640, 320, True), (0, 12867, 2104, 128, True), (2, 69866, 320, 304, True),
    (2, 7040, 1280, 320, True), (2, 9932, 2560, 96, True), (2, 13120, 1280, 64, True),
    # slower there (tile kernels / row-stationary, us): one chunk a block, grids just past a whole number of rounds
    (0, 61568, 72, 320, False),      # 16.5 / 20.6
    (1, 61568, 128, 320, False),     # 21.0 / 23.7
    (0, 14080, 640, 320, False),     # 19.8 / 20.4, 22.4 in double
    (0, 16640, 640, 320, False),     # 21.9 / 23.2, 26.1 in double
    (1, 23488, 328, 320, False),     # 20.5 / 22.0
    (0, 24576, 512, 320, False),     # 23.4 / 25.3 in double
    (1, 2944, 2568, 320, False),     # 16.1 / 17.1 in double
    (1, 4713, 2560, 320, False),     # 24.7 / 25.2, 27.8 in double
    # five K steps whatever Kp is
    (1, 34188, 640, 128, False),   # 1.13 times in double
    (1, 61568, 72, 64, False), (0, 24576, 512, 64, False), (1, 3136, 2560, 64, False), (1, 10844, 2560, 96, False), (2, 3136, 2560, 64, False),
    # few rows, few tiles
    (0, 16384, 320, 320, False), (1, 1000, 8000, 320, False), (1, 1400, 2560, 320, False),
])
def test_rows_with_shifts(rules, epi, M, N, K, row_stationary):
    """epi 0 PLAIN, 1 GEGLU, 2 GELU."""
    assert bool(rules.stripe_shift_rows(epi, M, N, K)) == row_stationary


@pytest.mark.parametrize("gn,M,RT,tiles", [
    # few rows: one tile a wave
    (0, 64, 1, 4), (0, 2048, 2, 4), (0, 1024, 4, 4), (1, 256, 1, 4), (1, 2048, 2, 4), (1, 4096, 4, 4),
    # whole numbers of blocks a CU (12 tiles a block, 1360 blocks, 77.7 -> 91.8 us of GroupNorm + SiLU, 16320 x 1920)
    (0, 16320, 1, 16), (1, 16320, 1, 32), (1, 16320, 4, 8), (1, 23108, 4, 8), (1, 32720, 4, 8), (0, 32720, 2, 16), (1, 13716, 2, 16),
    # between them, fewer rows a block
    (1, 11528, 4, 4), (0, 9688, 1, 8), (1, 9688, 1, 20), (1, 18000, 1, 12), (1, 13716, 1, 28), (1, 131072, 4, 8),
])
def test_norm_tiles(rules, gn, M, RT, tiles):
    assert rules.norm_tiles(gn, ctypes.c_longlong(M), RT, ctypes.c_longlong(1 << 20)) == tiles


@pytest.mark.parametrize("T", [1, 2, 3, 5, 7, 100])
@pytest.mark.parametrize("RT", [1, 2, 4, 8])
def test_norm_tiles_span(rules, T, RT):
    """A block of the GroupNorm apply spans at most eight samples, so at most 6 T + 1 rows (or one tile)."""
    for M in (T, 1000 * T + 1, 40000 * T):
        t = rules.norm_tiles(1, ctypes.c_longlong(M), RT, ctypes.c_longlong(6 * T + 1))
        assert 1 <= t and (t == 1 or t * RT <= min(32, 6 * T + 1))


@pytest.mark.parametrize("Tkp", range(64, 1280, 64))
def test_attention_form(rules, Tkp):
    """The kept forms hold every tile of the keys, and up to 256 keys no more than the next power of two of them."""
    f = rules.attn_form(Tkp)
    assert (f == 0) == (Tkp > 1024)
    if f:
        waves, tiles = f // 10, f % 10
        assert waves * tiles * 64 >= Tkp
        assert waves * tiles * 64 < 2 * Tkp
