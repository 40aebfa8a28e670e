"""The bf16 GEMM's tiles for small grids: 64 x 64 tiles and two 128 x 128
workgroups per CU, at ragged rows, columns and reductions, with the rank-r
columns filling and not filling the last step, forward (single and grouped) and
backward.

Against the composite in float64, y, dX within 1e-2 of the largest value (bf16
results), dA, dB within 1e-4 (fp32 sums over operands split to ~16 bits).
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float((a.double() - b).abs().max() / b.abs().max())


def make(dev, T, K, N, r, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    return dict(x=rnd(T, K).bfloat16(), W=(rnd(N, K) * 0.05).bfloat16(), A=rnd(K, r) * K ** -0.5, B=rnd(r, N) * 0.2,
                bias=rnd(N).bfloat16(), dY=rnd(T, N).bfloat16())


def reference(c, s):
    x, W, A, B, dY = (c[k].double() for k in ("x", "W", "A", "B", "dY"))
    h, g = x @ A, s * (dY @ B.t())
    return x @ W.t() + c["bias"].double() + s * (h @ B), dY @ W + g @ A.t(), x.t() @ g, s * (h.t() @ dY)


@pytest.mark.parametrize("T,K,N,r", [
    (65, 64, 64, 8), (65, 72, 136, 16), (100, 328, 3592, 16), (127, 1000, 1000, 5), (129, 56, 2048, 64),
    (463, 1536, 256, 64), (1243, 200, 520, 24), (8192, 136, 128, 16),      # 64 x 64
    (777, 200, 8960, 16), (777, 1536, 8952, 8), (300, 264, 18944, 16), (1025, 64, 3848, 70),  # 128 x 128 pairs
])
def test_gemm_small_grid_tiles(mc, dev, T, K, N, r):
    c = make(dev, T, K, N, r, T + K + N)
    y, h = mc.lora_forward(c["x"], c["A"], c["B"], 2.0, W=c["W"], bias=c["bias"])
    dX, dA, dB = mc.lora_backward(c["x"], c["A"], c["B"], c["dY"], 2.0, W=c["W"], h_save=h)
    y_ref, dX_ref, dA_ref, dB_ref = reference(c, 2.0)
    assert rel(y, y_ref) <= 1e-2 and rel(dX, dX_ref) <= 1e-2
    assert rel(dA, dA_ref) <= 1e-4 and rel(dB, dB_ref) <= 1e-4


@pytest.mark.parametrize("T,K,Ns,r", [(200, 896, [896, 128, 136], 8), (515, 264, [1536, 256, 256], 16),
                                      (600, 136, [4096, 4104], 64)])
def test_gemm_small_grid_group(mc, dev, T, K, Ns, r):
    cs = [make(dev, T, K, N, r, 11 * N + T) for N in Ns]
    x = cs[0]["x"]
    projs = [dict(W=c["W"], bias=c["bias"], A=c["A"], B=c["B"], Wt=mc.transpose_weight(c["W"])) for c in cs]
    ys, hs = mc.lora_group_forward(x, projs, 2.0)
    dX, dAs, dBs = mc.lora_group_backward(x, projs, [c["dY"] for c in cs], 2.0, h_saves=hs)
    total = 0.0
    for c, y, dA, dB in zip(cs, ys, dAs, dBs):
        c["x"] = x
        y1, _ = mc.lora_forward(x, c["A"], c["B"], 2.0, W=c["W"], bias=c["bias"])
        y_ref, dX_ref, dA_ref, dB_ref = reference(c, 2.0)
        assert torch.equal(y, y1) and rel(y, y_ref) <= 1e-2
        assert rel(dA, dA_ref) <= 1e-4 and rel(dB, dB_ref) <= 1e-4
        total = total + dX_ref
    assert rel(dX, total) <= 1e-2
