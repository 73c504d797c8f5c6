"""The prefill GEMM's choice of tile and K splits (csrc/gemm_rule.h, host
arithmetic), compiled by itself: no GPU."""
import ctypes as C
import os
import subprocess

import pytest

from webgllm_amd.self_check import PLAIN_TUNING

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "webgllm_amd",
                    "csrc")
ZK = {"q4_0": 0, "u8": 1, "f16": 2, "q8": 3}
CUS = 256
SIZES = [(M, N, K) for M in (9, 33, 45, 100, 131, 257, 300, 512, 1024, 2048)
         for N in (64, 256, 896, 1152, 2048, 4096, 6144, 9728, 14336, 28672)
         for K in (64, 256, 576, 768, 2048, 4096, 4864, 8192, 8448, 14336)]


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    d = tmp_path_factory.mktemp("rule")
    src, so = d / "rule.cpp", d / "rule.so"
    src.write_text(f'#include "{CSRC}/gemm_rule.h"\n'
                   'extern "C" int tile(int zk, int M, int N, int K, int cus, int residual,'
                   ' int groups, int splits) {\n'
                   '  return wg::gemm_tile_for(zk, M, N, K, cus, residual, groups, splits);\n}\n')
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-o",
                    str(so), str(src)], check=True)
    return C.CDLL(str(so))


def test_plain_settings_take_no_wave_groups(rule):
    """The self-check's simplest forms split no K, between waves or between
    workgroups (the library passes groups = (gemm_splits == 0))."""
    assert PLAIN_TUNING["gemm_splits"] == 1
    for zk in ZK.values():
        for M, N, K in SIZES:
            assert max(rule.tile(zk, M, N, K, CUS, r, 0, 0) for r in (0, 1)) <= 3, (zk, M, N, K)
    assert any(rule.tile(0, M, N, K, CUS, 0, 1, 1) >= 4 for M, N, K in SIZES)


# (form, M, N, K, the tile where splits may run, the tile under capture): each
# a shape beside a line, where the tile on its other side takes longer
@pytest.mark.parametrize("zk,M,N,K,tile,captured", [
    # one 64 x 64 a compute unit, not two 32 x 64
    ("f16", 300, 2048, 8192, 5, 5), ("q4_0", 33, 9728, 8192, 5, 5), ("u8", 45, 9728, 4864, 5, 5),
    ("u8", 33, 9728, 8192, 1, 5), ("q4_0", 131, 6144, 8192, 7, 7), ("q4_0", 700, 896, 768, 7, 7),
    # 64 x 128 in two groups only while the splits of one are slower
    ("q4_0", 100, 9728, 8192, 1, 4), ("q4_0", 1024, 1152, 8192, 1, 4),
    ("u8", 300, 4096, 8192, 1, 4), ("u8", 300, 4096, 4096, 4, 4),
    ("f16", 1500, 896, 8192, 2, 4), ("f16", 131, 9728, 8192, 4, 4),
    ("q8", 1024, 1152, 8192, 2, 4), ("q8", 131, 6144, 8192, 7, 7),
    # from 256 deep on
    ("q4_0", 45, 1152, 256, 6, 6), ("q8", 300, 1536, 512, 7, 7), ("q4_0", 45, 1152, 192, 1, 1),
    # half zero points' 64 x 128 to 1536 deep
    ("f16", 2048, 2048, 2048, 2, 2), ("q4_0", 2048, 2048, 2048, 1, 1),
    # 128 rows past 8192 deep: a split more, a costly dequant
    ("f16", 300, 4096, 14336, 2, 1), ("q8", 300, 4096, 14336, 2, 1),
    ("f16", 300, 9728, 8448, 2, 2), ("q4_0", 300, 4096, 14336, 1, 1), ("q8", 257, 6144, 8448, 1, 1),
    ("f16", 300, 1152, 14336, 1, 1), ("q4_0", 400, 1152, 8448, 1, 1)])
def test_lines(rule, zk, M, N, K, tile, captured):
    assert rule.tile(ZK[zk], M, N, K, CUS, 0, 1, 1) == tile
    assert rule.tile(ZK[zk], M, N, K, CUS, 0, 1, 0) == captured


# (form, M, N, K, the tile where a residual is added, without one)
@pytest.mark.parametrize("zk,M,N,K,tile,plain", [
    ("q4_0", 700, 1024, 4608, 7, 5), ("q4_0", 400, 2048, 8192, 7, 5), ("q8", 700, 1024, 4608, 5, 5),
    ("f16", 300, 2048, 6144, 7, 5), ("f16", 300, 2048, 7168, 5, 5), ("u8", 300, 2048, 7168, 7, 1),
    ("u8", 300, 2048, 8192, 1, 1), ("q4_0", 100, 9728, 4096, 4, 1), ("q4_0", 1024, 1152, 5632, 4, 1),
    ("f16", 1500, 896, 8192, 4, 2), ("q8", 1024, 1152, 8192, 4, 2), ("f16", 2048, 2048, 2048, 1, 2),
    ("u8", 64, 8704, 7168, 1, 1), ("q4_0", 64, 8704, 4096, 5, 5), ("q4_0", 65, 8192, 4096, 7, 5),
    ("q8", 65, 9216, 2048, 4, 7), ("q8", 65, 9216, 2560, 7, 7), ("q8", 400, 4096, 8448, 1, 2),
    ("q8", 400, 5120, 8448, 2, 2), ("u8", 300, 4096, 14336, 1, 2), ("f16", 400, 4096, 8448, 2, 2)])
def test_lines_of_a_residual(rule, zk, M, N, K, tile, plain):
    assert rule.tile(ZK[zk], M, N, K, CUS, 1, 1, 1) == tile
    assert rule.tile(ZK[zk], M, N, K, CUS, 0, 1, 1) == plain


def test_tiles_divide_the_columns(rule):
    """Every tile's columns divide N (a multiple of 64)."""
    cols = {0: 64, 1: 128, 2: 128, 3: 256, 4: 128, 5: 64, 6: 32, 7: 64, 8: 128}
    for zk in ZK.values():
        for M, N, K in SIZES + [(M, N + 64, K) for M, N, K in SIZES]:
            for form in ((0, 1, 1), (1, 1, 1), (0, 1, 0), (1, 1, 0), (0, 0, 0)):
                assert N % cols[rule.tile(zk, M, N, K, CUS, *form)] == 0
