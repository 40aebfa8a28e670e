"""Every load of the fp32 ring GEMM's [k][N] operand stays inside it.

The kernel keeps each lane's offset in a VGPR and passes a full step's advance
(32 k rows) in soffset. Only the VGPR offset is sure to be range-checked, so a
lane whose VGPR offset passes the check must land inside the operand after the
advance; the last, ragged step adds the advance to the VGPR offset. The offsets
are the header's own (compiled here with g++), the loop is gemm_f32_tiled's.
"""
import ctypes
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
STEP = 32


@pytest.fixture(scope="module")
def offset(tmp_path_factory):
    d = tmp_path_factory.mktemp("ring")
    src, so = d / "ring.cpp", d / "ring.so"
    src.write_text('#include "ring_offsets.hpp"\nextern "C" uint32_t off(int w, int l, int j, uint32_t ldb, int64_t cols)'
                   " { return mc::nn_chunk_offset(w, l, j, ldb, cols); }\n")
    inc = os.path.join(ROOT, "metal-candle_amd", "csrc")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", inc, str(src), "-o", str(so)], check=True)
    f = ctypes.CDLL(str(so)).off
    f.restype = ctypes.c_uint32
    f.argtypes = [ctypes.c_int] * 3 + [ctypes.c_uint32, ctypes.c_int64]
    return f


@pytest.mark.parametrize("k", [4, 32, 36, 64, 1024])  # one ragged step, one full, both, full last steps
@pytest.mark.parametrize("N", [4, 36, 64, 100, 800, 1000])  # 800: a last tile of 32 columns
def test_nn_loads_stay_inside_the_operand(offset, k, N):
    for n0 in range(0, N, 64):
        cols = N - n0
        size = ((k - 1) * N + cols) * 4  # bytes from element [0][n0] to the operand's end
        seen = set()
        steps = range((k + STEP - 1) // STEP)
        lanes = [(w, l, j, offset(w, l, j, N, cols)) for w in range(4) for j in range(2) for l in range(64)]
        for kt in sorted({steps[0], steps[-1], max(len(steps) - 2, 0)}):
            adv = kt * STEP * N * 4
            for w, l, j, off in lanes:
                row, col = 8 * w + 4 * j + l // 16, 4 * ((l % 16) ^ (8 * j))
                if kt < k // STEP:  # full step: the check sees the VGPR offset only
                    fetched, at = off < size, off + adv
                else:
                    fetched, at = off + adv < size, off + adv
                if fetched:
                    assert at + 16 <= size, (n0, kt, w, l, j)
                if kt * STEP + row < k and col < cols:
                    assert fetched and at == ((kt * STEP + row) * N + col) * 4
                    seen.add((kt, row, col))
        full = sum(min(STEP, k - kt * STEP) for kt in sorted({steps[0], steps[-1], max(len(steps) - 2, 0)}))
        assert len(seen) == full * ((min(cols, 64) + 3) // 4)
