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
int xent_stream_gradients(int64_t rows, int64_t vocab, int elem_size) {
    return mc::xent_stream_gradients(rows, vocab, elem_size);
}
int xent_wide_rows(int64_t rows, int64_t vocab, int elem_size) { return mc::xent_wide_rows(rows, vocab, elem_size); }
int softmax_ragged_vectors(int64_t rows, int64_t dim, int causal, int elem_size, int backward) {
    return mc::softmax_ragged_vectors(rows, dim, causal != 0, elem_size, backward != 0);
}
int attention_f32_tiles_fit(int64_t S, int64_t bh) { return mc::attention_f32_tiles_fit(S, bh); }
int attention_f32_rows_fwd(int64_t S, int D) { return mc::attention_f32_rows_fwd(S, D); }
int attention_f32_rows_bwd(int64_t S, int D, int rep) { return mc::attention_f32_rows_bwd(S, D, rep); }
int lora_few_tokens(int64_t T, int64_t N, int r) { return mc::lora_few_tokens(T, N, r); }
int rowproj_f32_by_token(int64_t T, int r) { return mc::rowproj_f32_by_token(T, r); }
int colreduce_f32_tile(int64_t T, int64_t cols, int r) {
    const mc::ColF32Tile t = mc::colreduce_f32_tile(T, cols, r);
    return 10 * t.rt + t.ct;
}
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


# A projection's forward, us: few-token kernels, tiled path, the tiled path before it had tiles for small
# grids. Up to 16 tokens the rule may leave 10% to the tiled path.
@pytest.mark.parametrize("T,K,N,r,few,tiled,former", [
    (8, 1536, 1536, 8, 9.4, 16.6, 27.3), (8, 3584, 18944, 64, 50.1, 56.4, 65.9), (16, 1536, 8960, 8, 18.7, 17.0, 27.6),
    (16, 18944, 3584, 64, 59.2, 135.0, 198.4), (17, 896, 896, 8, 9.4, 11.5, 19.2), (17, 1536, 8960, 8, 19.3, 17.1, 28.0),
    (17, 3584, 18944, 64, 65.3, 57.3, 66.3), (20, 8960, 1536, 64, 47.1, 71.0, 98.9), (24, 1536, 8960, 64, 31.7, 29.0, 34.9),
    (24, 3584, 18944, 8, 51.5, 47.6, 66.5), (24, 3584, 3584, 64, 29.5, 39.8, 51.5), (28, 3584, 512, 8, 20.6, 31.6, 50.6),
    (32, 896, 128, 64, 19.4, 23.9, 27.6), (32, 1536, 1536, 64, 23.3, 28.0, 33.4), (32, 1536, 18944, 64, 48.2, 40.2, 41.6),
    (32, 896, 28672, 48, 39.4, 33.4, 33.8), (32, 3584, 18944, 64, 71.7, 60.7, 67.1), (32, 18944, 3584, 8, 77.9, 125.4, 190.4),
])
def test_lora_few_tokens(rules, T, K, N, r, few, tiled, former):
    chosen = few if rules.lora_few_tokens(ctypes.c_int64(T), ctypes.c_int64(N), r) else tiled
    assert chosen <= (1.1 if T <= 16 else 1.03) * min(few, tiled)
    assert chosen <= former


def test_lora_few_tokens_limits(rules):
    for T, N, r, want in ((16, 1 << 20, 64, 1), (16, 8, 65, 0), (17, 8192, 64, 1), (17, 8200, 1, 0), (32, 8192, 64, 1),
                          (33, 8, 1, 0)):
        assert rules.lora_few_tokens(ctypes.c_int64(T), ctypes.c_int64(N), r) == want


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


# dB of one projection, us, by tile (10 rt + ct).
@pytest.mark.parametrize("r,cols,T,us", [
    (4, 128, 2048, {11: 8.1, 14: 15.6}), (4, 4608, 2048, {11: 22.9, 14: 18.5}), (4, 8960, 512, {11: 10.7, 14: 7.8}),
    (16, 128, 4096, {11: 15.9, 14: 28.0}), (16, 768, 32, {11: 2.9, 14: 4.5}), (16, 2304, 2048, {11: 10.9, 14: 16.9}),
    (16, 4608, 32, {11: 3.2, 14: 4.5}), (16, 4608, 2048, {11: 25.8, 14: 20.6}), (16, 8960, 4096, {11: 74.1, 14: 43.2}),
    (32, 128, 512, {11: 4.4, 14: 6.3, 21: 5.7, 24: 10.2}), (32, 2304, 2048, {11: 15.5, 14: 17.0, 21: 17.2, 24: 31.3}),
    (32, 4608, 2048, {11: 29.7, 14: 20.0, 21: 33.7, 24: 35.7}), (32, 8960, 4096, {11: 104.9, 14: 72.4, 21: 96.5, 24: 67.7}),
    (64, 128, 512, {11: 4.5, 14: 6.3, 24: 10.3, 44: 17.6}), (64, 768, 4096, {11: 16.6, 14: 29.1, 24: 56.0, 44: 92.0}),
    (64, 1536, 32, {11: 3.2, 14: 4.6, 24: 6.5, 44: 10.6}), (64, 1536, 2048, {11: 15.7, 14: 17.4, 24: 31.3, 44: 50.9}),
    (64, 2304, 2048, {11: 22.9, 14: 17.8, 24: 31.7, 44: 51.2}), (64, 4608, 2048, {11: 50.2, 14: 33.0, 24: 35.9, 44: 56.2}),
    (64, 8960, 2048, {11: 94.1, 14: 59.1, 24: 57.5, 44: 57.6}), (64, 8960, 4096, {11: 187.9, 14: 110.4, 24: 107.4, 44: 103.1}),
    (128, 768, 4096, {11: 26.0, 14: 29.1, 24: 56.5, 44: 91.8}), (128, 4608, 4096, {11: 189.1, 14: 85.8, 24: 102.2, 44: 99.7}),
    (128, 8960, 2048, {11: 180.2, 14: 98.1, 24: 82.5, 44: 104.4}),
])
def test_colreduce_f32_tile(rules, r, cols, T, us):
    tile = rules.colreduce_f32_tile(ctypes.c_int64(T), ctypes.c_int64(cols), r)
    assert us[tile] <= 1.03 * min(us.values())


# fp32 attention, time on the 32 x 32 tiles over time on the row kernels, by sequence (the worse of causal or
# not for whichever side the rule takes; 10% either way around the crossing).
@pytest.mark.parametrize("D,rep,fwd,bwd", [
    (32, 1, {1: 1.73, 2: 1.38, 3: 1.18, 8: 0.74, 16: 0.45}, {1: 1.62, 2: 1.40, 3: 1.25, 10: 0.79, 16: 0.58}),
    (64, 1, {1: 2.10, 3: 1.51, 6: 1.07, 10: 0.84, 16: 0.59}, {1: 2.21, 5: 1.49, 8: 1.20, 16: 0.88, 24: 0.70}),
    (64, 6, {1: 2.03, 3: 1.50, 6: 1.06, 10: 0.84, 16: 0.59}, {1: 2.00, 2: 1.48, 3: 1.16, 5: 0.92, 8: 0.67}),
    (128, 6, {1: 3.01, 4: 1.65, 8: 1.08, 12: 0.90, 24: 0.51}, {1: 2.79, 3: 1.45, 5: 1.02, 8: 0.83, 16: 0.47}),
    (128, 7, {1: 2.81, 4: 1.65, 8: 1.07, 12: 0.90, 24: 0.27}, {1: 2.43, 3: 1.36, 4: 1.06, 6: 0.94, 8: 0.69}),
    (96, 1, {1: 3.08, 4: 1.68, 8: 1.08, 12: 0.91, 24: 0.51}, {1: 3.57, 8: 1.62, 12: 1.27, 24: 0.89}),
])
def test_attention_f32_rows(rules, D, rep, fwd, bwd):
    for S, ratio in fwd.items():
        rows = rules.attention_f32_rows_fwd(ctypes.c_int64(S), D)
        assert (ratio if not rows else 1 / ratio) <= 1.1, ("forward", S)
    for S, ratio in bwd.items():
        rows = rules.attention_f32_rows_bwd(ctypes.c_int64(S), D, rep)
        assert (ratio if not rows else 1 / ratio) <= 1.1, ("backward", S)


# Softmax rows of S elements, 56 heads of S x S and 112 causal ones, us: (elements, covering vectors) of each.
@pytest.mark.parametrize("size,backward,S,plain,causal", [
    (4, 0, 9, (2.3, 2.6), (2.4, 2.7)), (4, 0, 33, (2.4, 2.8), (2.8, 3.3)), (4, 0, 65, (3.0, 3.1), (3.8, 4.1)),
    (4, 0, 99, (3.7, 3.5), (5.4, 5.1)), (4, 0, 201, (8.4, 5.3), (11.7, 8.2)), (4, 0, 777, (113.0, 44.1), (176.8, 75.3)),
    (4, 1, 33, (2.2, 2.8), (2.4, 3.5)), (4, 1, 99, (3.5, 4.0), (5.0, 5.7)), (4, 1, 161, (6.5, 5.5), (7.7, 7.7)),
    (4, 1, 301, (17.6, 13.5), (24.8, 19.4)), (4, 1, 777, (122.4, 76.8), (148.1, 111.0)),
    (2, 0, 33, (2.4, 3.1), (2.9, 3.8)), (2, 0, 99, (3.5, 4.2), (5.0, 6.0)), (2, 0, 201, (8.0, 6.2), (11.0, 10.2)),
    (2, 0, 777, (92.8, 32.4), (120.0, 54.9)), (2, 1, 33, (2.2, 3.1), (2.4, 3.8)), (2, 1, 77, (2.7, 4.0), (3.7, 5.5)),
    (2, 1, 129, (4.0, 4.9), (5.9, 7.5)), (2, 1, 257, (8.8, 7.3), (12.5, 11.6)), (2, 1, 1023, (132.7, 101.8), (192.2, 189.7)),
])
def test_softmax_ragged_vectors(rules, size, backward, S, plain, causal):
    for heads, c, us in ((56, 0, plain), (112, 1, causal)):
        vectors = rules.softmax_ragged_vectors(ctypes.c_int64(heads * S), ctypes.c_int64(S), c, size, backward)
        assert us[vectors] <= 1.03 * min(us)


# 65536 rows, no mask.
@pytest.mark.parametrize("size,dim,forward,backward", [
    (4, 33, (14.6, 15.0), (11.1, 17.8)), (4, 77, (20.7, 15.0), (21.3, 19.0)), (4, 129, (30.9, 16.8), (31.1, 27.4)),
    (2, 33, (14.2, 21.3), (10.8, 19.2)), (2, 77, (20.4, 21.1), (15.7, 19.1)), (2, 129, (26.6, 21.2), (27.3, 20.9)),
    (2, 301, (52.1, 23.6), (47.8, 29.9)),
])
def test_softmax_ragged_vectors_many_rows(rules, size, dim, forward, backward):
    for b, us in enumerate((forward, backward)):
        vectors = rules.softmax_ragged_vectors(ctypes.c_int64(65536), ctypes.c_int64(dim), 0, size, b)
        assert us[vectors] == min(us)


# Cross-entropy forward and backward, us: 256 threads, 1024 threads, by rows.
@pytest.mark.parametrize("size,V,us", [
    (4, 4096, {64: (11.4, 12.5), 512: (14.2, 17.3), 1000: (17.5, 25.2)}),
    (4, 8001, {64: (15.9, 14.0), 200: (16.7, 15.4)}),
    (2, 10001, {64: (13.1, 13.5), 128: (14.7, 14.5)}),
    (4, 8192, {64: (13.8, 13.6), 256: (15.7, 15.3), 384: (16.3, 19.0), 640: (19.1, 24.9), 1000: (23.9, 30.5)}),
    (4, 16384, {128: (19.6, 16.7), 256: (20.4, 19.2), 384: (22.4, 24.4), 512: (24.7, 27.6)}),
    (4, 32000, {64: (28.5, 18.7), 256: (30.3, 25.8), 384: (40.2, 36.8), 640: (52.9, 54.7)}),
    (4, 151936, {64: (110.8, 44.5), 384: (165.7, 132.4), 512: (183.3, 165.2), 1023: (339.8, 338.8)}),
    (2, 8192, {64: (11.7, 12.9), 256: (13.6, 14.2), 512: (15.3, 18.0), 1000: (19.1, 26.4)}),
    (2, 16384, {64: (15.3, 15.0), 256: (16.6, 16.0), 384: (17.9, 19.7), 1000: (25.4, 32.2)}),
    (2, 32000, {128: (22.8, 19.5), 256: (23.8, 21.1), 512: (27.7, 29.4), 1000: (44.6, 50.4)}),
    (2, 50257, {64: (28.6, 20.6), 384: (36.3, 34.8), 512: (41.3, 39.9), 768: (51.9, 53.9)}),
    (2, 151936, {64: (63.7, 35.9), 512: (115.6, 95.3), 768: (134.8, 131.3), 896: (153.1, 154.6)}),
])
def test_xent_wide_rows(rules, size, V, us):
    for rows, t in us.items():
        wide = rules.xent_wide_rows(ctypes.c_int64(rows), ctypes.c_int64(V), size)
        assert t[wide] <= 1.04 * min(t), rows


# Cross-entropy forward and backward in a loop over three inputs, us: ordinary stores, streamed.
@pytest.mark.parametrize("size,V,us", [
    (4, 32000, {20: (25.7, 25.3), 50: (35.0, 35.2), 85: (55.3, 50.6), 100: (69.4, 61.8), 140: (95.2, 81.7)}),
    (4, 151936, {20: (38.6, 38.7), 60: (41.5, 41.1), 70: (47.2, 42.4), 85: (55.8, 46.7), 120: (81.7, 63.5)}),
    (2, 32000, {10: (25.2, 25.5), 50: (42.4, 42.3), 70: (45.9, 43.9), 100: (69.7, 60.1), 140: (101.3, 87.4)}),
    (2, 151936, {20: (36.9, 35.5), 60: (39.6, 38.9), 85: (65.9, 63.1), 100: (77.2, 67.7), 140: (100.4, 87.1)}),
])
def test_xent_stream_gradients_alone(rules, size, V, us):
    for mb, t in us.items():
        stream = rules.xent_stream_gradients(ctypes.c_int64(mb * 10**6 // size // V), ctypes.c_int64(V), size)
        assert t[stream] <= 1.04 * min(t), mb


# The same on logits not seen before, with the LoRA backward that reads the gradients behind it, us.
@pytest.mark.parametrize("size,rows,V,us", [
    (4, 200, 32000, (129.9, 141.3)), (4, 200, 50257, (179.4, 234.6)), (4, 64, 151936, (487.5, 536.6)),
    (2, 64, 32000, (143.7, 165.1)), (2, 500, 32000, (172.3, 187.5)), (2, 64, 151936, (559.6, 690.6)),
    (2, 200, 151936, (656.3, 715.7)), (2, 1500, 151936, (492.1, 476.2)), (4, 4096, 8192, (143.6, 141.4)),
])
def test_xent_stream_gradients_with_reader(rules, size, rows, V, us):
    stream = rules.xent_stream_gradients(ctypes.c_int64(rows), ctypes.c_int64(V), size)
    assert us[stream] == min(us)


def test_xent_stream_gradients_line(rules):
    assert not rules.xent_stream_gradients(ctypes.c_int64(64 << 10), ctypes.c_int64(512), 2)
    assert rules.xent_stream_gradients(ctypes.c_int64((64 << 10) + 1), ctypes.c_int64(512), 2)


def test_attention_f32_tiles_fit(rules):
    """One launch holds at most 2^32 - 1 work-items; calls that the tiles would
    take past that stay with the row kernels."""
    for S, bh, want in ((2, 16777215, 1), (2, 16777216, 0), (33, 8388607, 1), (33, 8388608, 0), (1 << 20, 511, 1)):
        assert rules.attention_f32_tiles_fit(ctypes.c_int64(S), ctypes.c_int64(bh)) == want
        if want:
            assert (S + 31) // 32 * bh * 256 < 1 << 32
