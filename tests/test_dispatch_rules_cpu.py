"""Each rule that chooses between two kernels by a call's sizes, against times
measured on an MI355X with either kernel: where the two differ by more than the
measurement's noise (3%), the rule takes the faster one. The rules are the header's own, compiled
here with g++.
"""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

SOURCE = """
#include "rules.hpp"
extern "C" {
int rowproj_f32_by_token(int64_t T, int r) { return mc::rowproj_f32_by_token(T, r); }
}
"""


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    d = tmp_path_factory.mktemp("rules")
    src, so = d / "rules.cpp", d / "rules.so"
    src.write_text(SOURCE)
    inc = os.path.join(ROOT, "metal-candle_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", inc, str(src), "-o", str(so)],
                   check=True)
    return ctypes.CDLL(str(so))


# A forward without W (projection and a product of 64 columns), us: workgroup per token, per 16 tokens.
@pytest.mark.parametrize("r,K,T,by_token,by_16", [
    (1, 768, 32, 7.4, 9.2), (1, 3584, 512, 9.9, 17.0), (1, 3584, 1024, 11.0, 17.1), (1, 8960, 256, 11.9, 29.2),
    (4, 128, 256, 7.3, 7.6), (4, 768, 32, 7.7, 9.0), (4, 768, 512, 8.5, 9.5), (4, 1536, 128, 8.5, 11.4),
    (4, 3584, 256, 11.0, 17.0), (4, 8960, 32, 14.8, 28.6), (4, 8960, 512, 23.6, 29.3),
    (1, 3584, 4096, 23.8, 20.6), (1, 128, 4096, 9.5, 8.0), (4, 768, 1024, 10.1, 9.6), (4, 8960, 1024, 39.8, 31.3),
    (4, 8960, 4096, 134.4, 41.1),
])
def test_rowproj_f32_by_token(rules, r, K, T, by_token, by_16):
    chosen = by_token if rules.rowproj_f32_by_token(ctypes.c_int64(T), r) else by_16
    assert chosen <= 1.03 * min(by_token, by_16)
