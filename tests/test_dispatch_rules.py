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
