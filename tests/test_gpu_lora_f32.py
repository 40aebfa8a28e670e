"""The float32 LoRA linear at the sizes where its kernels change: products of
enough 64 x 64 tiles for the LDS-ring GEMM (ragged tiles, ragged last k steps,
one to several 64-rank blocks) next to shapes that stay on the 32 x 32 one, and
the rank-r products at the edges of their tiles.

Reference: the same composite in float64 on the GPU. Tolerance as in
test_gpu_lora.py: max|out - ref| / max|ref| <= 1e-5.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = 1e-5


def close(got, want, name):
    err = float((got.double() - want).abs().max() / want.abs().max())
    assert err <= TOL, f"{name}: {err:.2e}"


def lora_case(dev, T, K, N, r, p, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    mask = (torch.rand(T, r, generator=g, device=dev) >= p).to(torch.uint8) if p > 0 else None
    return dict(x=rnd(T, K), W=rnd(N, K) * 0.05, A=rnd(K, r) * 0.1, B=rnd(r, N) * 0.1, bias=rnd(N), dY=rnd(T, N), mask=mask)


def check_lora(mc, c, scale, p):
    y, h = mc.lora_forward(c["x"], c["A"], c["B"], scale, W=c["W"], bias=c["bias"], mask=c["mask"], dropout_p=p)
    dX, dA, dB = mc.lora_backward(c["x"], c["A"], c["B"], c["dY"], scale, W=c["W"], mask=c["mask"], dropout_p=p, h_save=h)
    x, W, A, B, dY = (c[k].double() for k in ("x", "W", "A", "B", "dY"))
    keep = 1.0 if c["mask"] is None else c["mask"].double() / (1.0 - p)
    H = (x @ A) * keep
    G = scale * (dY @ B.t()) * keep
    close(h.t(), H, "h")
    close(y, x @ W.t() + c["bias"].double() + scale * (H @ B), "y")
    close(dX, dY @ W + G @ A.t(), "dX")
    close(dA, x.t() @ G, "dA")
    close(dB, scale * (H.t() @ dY), "dB")


@pytest.mark.parametrize("T,K,N,r,p", [
    (1024, 896, 896, 8, 0.0),       # whole tiles and steps
    (1000, 900, 908, 16, 0.1),      # ragged tiles, last step of 4 k
    (2036, 256, 1536, 5, 0.0),      # few steps
    (4100, 64, 1000, 64, 0.0),      # two steps: less than the ring
    (4100, 32, 1000, 7, 0.0),       # one step
    (4100, 1000, 36, 1, 0.0),       # the backward's reduction of one ragged step
    (4100, 1000, 1024, 8, 0.0),     # ragged columns whose last k row is in a full step
    (4100, 1000, 100, 130, 0.0),    # three blocks of ranks, the last of two
    (1030, 1028, 1028, 65, 0.1),
])
def test_lora_f32_ring_gemm(mc, dev, T, K, N, r, p):
    check_lora(mc, lora_case(dev, T, K, N, r, p, T + K + N + r), 2.0, p)


@pytest.mark.parametrize("T,K,N,r", [(1024, 897, 896, 8), (1024, 896, 898, 8), (1023, 770, 1030, 3), (64, 768, 768, 8),
                                     (1, 4, 4, 1)])
def test_lora_f32_other_shapes(mc, dev, T, K, N, r):
    """Widths whose rows are not whole 16-byte chunks, and small products."""
    check_lora(mc, lora_case(dev, T, K, N, r, 0.0, T + K), 0.5, 0.0)


@pytest.mark.parametrize("r", [1, 15, 16, 17, 32, 33, 64, 65, 129])
@pytest.mark.parametrize("T,K,N", [(1, 5, 7), (17, 31, 33), (33, 64, 65), (250, 66, 127), (257, 1000, 130)])
def test_lora_f32_rank_products(mc, dev, T, K, N, r):
    """The rank-r products on the matrix cores: ranks around the 16-rank tiles
    and 64-rank groups, tokens and columns around the 16-token and 32- / 64-
    column blocks, rows that are not 16-byte aligned, dropout."""
    check_lora(mc, lora_case(dev, T, K, N, r, 0.1, T + K + r), 2.0, 0.1)


@pytest.mark.parametrize("T,K,N,r", [(65, 3070, 67, 16), (300, 3001, 130, 7), (32, 6300, 65, 40), (33, 6300, 65, 40),
                                     (270, 6211, 90, 33), (4099, 6211, 90, 64), (4096, 6200, 64, 65)])
def test_lora_f32_column_tiles(mc, dev, T, K, N, r):
    """The column reductions' other tiles (64 columns by 16, 32 and 64 ranks):
    wide inputs of ragged columns, tokens and ranks."""
    check_lora(mc, lora_case(dev, T, K, N, r, 0.1, T + K + r), 2.0, 0.1)


@pytest.mark.parametrize("T,K,N,r", [(2048, 300, 7, 1), (2049, 300, 7, 1), (33, 1030, 513, 3), (512, 255, 257, 4),
                                     (513, 256, 255, 4), (256, 8960, 512, 2)])
def test_lora_f32_projection_by_token(mc, dev, T, K, N, r):
    """The row projection with a workgroup per token, and just past it: up to 4
    ranks and 2048 tokens over the ranks, columns around a pass of 256."""
    check_lora(mc, lora_case(dev, T, K, N, r, 0.1, T + K + r), 2.0, 0.1)


def test_lora_f32_ring_gemm_sees_only_its_rows(mc, dev):
    """A non-finite token reaches its own row of y and dX and no other, and a
    non-finite weight row its own column of y."""
    c = lora_case(dev, 1030, 900, 900, 8, 0.0, 5)
    y, _ = mc.lora_forward(c["x"], c["A"], c["B"], 1.0, W=c["W"])
    dX, _, _ = mc.lora_backward(c["x"], c["A"], c["B"], c["dY"], 1.0, W=c["W"], need_dA=False, need_dB=False)
    x2, d2, W2 = c["x"].clone(), c["dY"].clone(), c["W"].clone()
    x2[1029], d2[1029] = float("inf"), float("nan")
    y2, _ = mc.lora_forward(x2, c["A"], c["B"], 1.0, W=c["W"])
    dX2, _, _ = mc.lora_backward(c["x"], c["A"], c["B"], d2, 1.0, W=c["W"], need_dA=False, need_dB=False)
    assert torch.equal(y[:1029], y2[:1029]) and torch.equal(dX[:1029], dX2[:1029])
    W2[899] = float("nan")
    y3, _ = mc.lora_forward(c["x"], c["A"], c["B"], 1.0, W=W2)
    assert torch.equal(y[:, :899], y3[:, :899]) and torch.isnan(y3[:, 899]).all()
