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
                   'extern "C" int tile(int zk, int M, int N, int K, int cus, int groups) {\n'
                   '  return wg::gemm_tile_for(zk, M, N, K, cus, groups != 0);\n}\n')
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-o",
                    str(so), str(src)], check=True)
    return C.CDLL(str(so))


def test_plain_settings_take_no_wave_groups(rule):
    """The self-check's simplest forms split no K, between waves or between
    workgroups (the library passes groups = (gemm_splits == 0))."""
    assert PLAIN_TUNING["gemm_splits"] == 1
    for zk in ZK.values():
        for M, N, K in SIZES:
            assert rule.tile(zk, M, N, K, CUS, 0) <= 3, (zk, M, N, K)
    assert any(rule.tile(0, M, N, K, CUS, 1) >= 4 for M, N, K in SIZES)
