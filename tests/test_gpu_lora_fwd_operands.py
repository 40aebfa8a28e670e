"""The bf16 LoRA forward whose hidden and B^T operands come from one launch
(lora_fwd_operands): tokens around its 16-token tiles and the limits of its
rule, ranks around its 16-rank tiles and its limit, reductions around its
64-column blocks and 1024-column rounds, dropout, and groups.

Against the composite in float64: y within bf16 rounding of it (1e-2 of the
largest value), the fp32 hidden within 1e-5.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


def fwd_case(dev, T, K, N, r, p, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    return dict(x=rnd(T, K).bfloat16(), W=(rnd(N, K) * 0.05).bfloat16(), bias=rnd(N).bfloat16(), A=rnd(K, r) * K ** -0.5,
                B=rnd(r, N) * 0.2, mask=(torch.rand(T, r, generator=g, device=dev) >= p).to(torch.uint8) if p > 0 else None)


@pytest.mark.parametrize("T", [33, 48, 63, 4095, 4096, 4097])
@pytest.mark.parametrize("K,N,r,p", [(8, 8, 1, 0.0), (72, 40, 16, 0.1), (1032, 24, 17, 0.0), (2048, 136, 32, 0.1),
                                     (1088, 64, 33, 0.0), (4088, 16, 5, 0.0)])
def test_lora_fwd_one_launch(mc, dev, T, K, N, r, p):
    c = fwd_case(dev, T, K, N, r, p, T + K + N + r)
    x, A, B = c["x"].double(), c["A"].double(), c["B"].double()
    H = x @ A
    if c["mask"] is not None:
        H = H * c["mask"].double() / (1.0 - p)
    for W in (c["W"], None):
        y, h = mc.lora_forward(c["x"], c["A"], c["B"], 2.0, W=W, bias=c["bias"] if W is not None else None,
                               mask=c["mask"], dropout_p=p)
        want = 2.0 * (H @ B)
        if W is not None:
            want = want + x @ W.double().t() + c["bias"].double()
        assert float((h.t().double() - H).abs().max()) <= 1e-5 * float(H.abs().max())
        assert float((y.double() - want).abs().max()) <= 1e-2 * float(want.abs().max())


@pytest.mark.parametrize("T,r", [(100, 8), (4096, 20)])
def test_lora_fwd_one_launch_group_equals_single(mc, dev, T, r):
    Ns = [152, 24, 64]
    cs = [fwd_case(dev, T, 1160, N, r, 0.1, 7 + N) for N in Ns]
    x = cs[0]["x"]
    projs = [dict(W=c["W"], bias=c["bias"], A=c["A"], B=c["B"], mask=c["mask"]) for c in cs]
    projs[1]["W"] = projs[1]["bias"] = None
    ys, hs = mc.lora_group_forward(x, projs, 2.0, dropout_p=0.1)
    for pr, y, h in zip(projs, ys, hs):
        y1, h1 = mc.lora_forward(x, pr["A"], pr["B"], 2.0, W=pr["W"], bias=pr["bias"], mask=pr["mask"], dropout_p=0.1)
        assert torch.equal(y, y1) and torch.equal(h, h1)
