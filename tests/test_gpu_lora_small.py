"""The bf16 LoRA forward of a few tokens (lora_small.hip): tokens around its
16-token tiles and its limit, ranks around the 16-rank tiles and its limit,
reductions and outputs around its steps and splits, dropout, no base weight,
and the saved hidden that the backward reads.

Against the composite in float64: y within bf16 rounding of it (1e-2 of the
largest value), the fp32 hidden within 1e-5.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


def small_case(dev, T, K, N, r, p, bias, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device=dev)
    return dict(x=rnd(T, K).bfloat16(), W=(rnd(N, K) * 0.05).bfloat16(), A=rnd(K, r) * K ** -0.5, B=rnd(r, N) * 0.2,
                bias=rnd(N).bfloat16() if bias else None,
                mask=(torch.rand(T, r, generator=g, device=dev) >= p).to(torch.uint8) if p > 0 else None)


def check_small(mc, c, W, p, scale=2.0):
    y, h = mc.lora_forward(c["x"], c["A"], c["B"], scale, W=W, bias=c["bias"] if W is not None else None,
                           mask=c["mask"], dropout_p=p)
    x, A, B = c["x"].double(), c["A"].double(), c["B"].double()
    H = x @ A
    if c["mask"] is not None:
        H = H * c["mask"].double() / (1.0 - p)
    want = scale * (H @ B)
    if W is not None:
        want = want + x @ W.double().t()
        if c["bias"] is not None:
            want = want + c["bias"].double()
    assert float((h.t().double() - H).abs().max()) <= 1e-5 * float(H.abs().max())
    assert float((y.double() - want).abs().max()) <= 1e-2 * float(want.abs().max())
    return y, h


@pytest.mark.parametrize("T", [1, 2, 15, 16, 17, 31, 32, 33])
@pytest.mark.parametrize("K,N,r,p,bias", [(896, 128, 8, 0.0, True), (1536, 1536, 16, 0.1, False), (64, 24, 1, 0.0, True),
                                          (8, 8, 17, 0.0, False), (64, 16400, 5, 0.0, True), (1032, 1000, 33, 0.0, True), (4096, 40, 64, 0.1, True),
                                          (3592, 520, 64, 0.0, False), (520, 1544, 65, 0.0, True),
                                          (100, 50, 7, 0.0, True)])
def test_lora_few_tokens(mc, dev, T, K, N, r, p, bias):
    c = small_case(dev, T, K, N, r, p, bias, T + K + N + r)
    y, h = check_small(mc, c, c["W"], p)
    check_small(mc, c, None, p)
    y2, _ = mc.lora_forward(c["x"], c["A"], c["B"], 2.0, W=c["W"], bias=c["bias"], mask=c["mask"], dropout_p=p,
                            save_hidden=False)
    assert torch.equal(y, y2)


@pytest.mark.parametrize("T", [1, 5, 30])
def test_lora_few_tokens_group_equals_single(mc, dev, T):
    Ns = [1536, 256, 248]
    cs = [small_case(dev, T, 1536, N, 16, 0.1, True, 7 + N) for N in Ns]
    x = cs[0]["x"]
    projs = [dict(W=c["W"], bias=c["bias"], A=c["A"], B=c["B"], mask=c["mask"]) for c in cs]
    projs[1]["W"] = projs[1]["bias"] = None
    ys, hs = mc.lora_group_forward(x, projs, 2.0, dropout_p=0.1)
    for pr, y, h in zip(projs, ys, hs):
        y1, h1 = mc.lora_forward(x, pr["A"], pr["B"], 2.0, W=pr["W"], bias=pr["bias"], mask=pr["mask"], dropout_p=0.1)
        assert torch.equal(y, y1) and torch.equal(h, h1)


@pytest.mark.parametrize("T", [1, 16, 17, 32])
@pytest.mark.parametrize("Ns,r", [((8960, 8952, 24), 16), ((8184, 8192, 24), 64), ((24, 8200, 1000, 8960), 33)])
def test_lora_few_tokens_wide_group_equals_single(mc, dev, T, Ns, r):
    """Groups of 16384 or more columns take the wide kernels where each of their
    projections alone takes the narrow ones, and past 16 tokens projections of
    more than 8192 columns go another way than the rest of the group."""
    K = 264
    cs = [small_case(dev, T, K, N, r, 0.1, i % 2 == 0, 11 + N + T) for i, N in enumerate(Ns)]
    x = cs[0]["x"]
    projs = [dict(W=c["W"], bias=c["bias"], A=c["A"], B=c["B"], mask=c["mask"]) for c in cs]
    ys, hs = mc.lora_group_forward(x, projs, 2.0, dropout_p=0.1)
    for c, pr, y, h in zip(cs, projs, ys, hs):
        c["x"] = x
        y1, h1 = check_small(mc, c, c["W"], 0.1)
        assert torch.equal(y, y1) and torch.equal(h, h1)
    ys2, _ = mc.lora_group_forward(x, projs, 2.0, dropout_p=0.1, save_hidden=False)
    assert all(torch.equal(a, b) for a, b in zip(ys, ys2))


def test_lora_few_tokens_are_timed_by_class(mc, dev):
    """The timing hook books the hidden's launches as low-rank work and the
    product with W as a GEMM, as on the tiled path."""
    T, K, N, r = 5, 1032, 1000, 8
    c = small_case(dev, T, K, N, r, 0.0, False, 4)
    L = mc._lib.lib()
    mc._lib.check(L.mc_profile_reset())
    mc._lib.check(L.mc_profile_enable(1))
    try:
        mc.lora_forward(c["x"], c["A"], c["B"], 1.0, W=c["W"])
        mc.lora_forward(c["x"], c["A"], c["B"], 1.0)
    finally:
        mc._lib.check(L.mc_profile_enable(0))
    mc._lib.check(L.mc_profile_collect())
    low, gemm = mc._lib.profile_read("lowrank"), mc._lib.profile_read("gemm")
    mc._lib.check(L.mc_profile_reset())
    assert low[1] == gemm[1] == 2 and low[0] > 0 and gemm[0] > 0
    assert low[2] == 2 * (2 * T * K * r) and gemm[2] == 2 * T * N * K + 2 * T * N * r


def test_lora_few_tokens_are_apart(mc, dev):
    """A non-finite token or weight row reaches its own outputs only."""
    c = small_case(dev, 5, 1032, 1000, 8, 0.0, True, 3)
    y, _ = mc.lora_forward(c["x"], c["A"], c["B"], 1.0, W=c["W"], bias=c["bias"])
    x2, W2 = c["x"].clone(), c["W"].clone()
    x2[4], W2[999] = float("nan"), float("inf")
    y2, _ = mc.lora_forward(x2, c["A"], c["B"], 1.0, W=W2, bias=c["bias"])
    assert torch.equal(y[:4, :999], y2[:4, :999])
    assert torch.isnan(y2[4]).all() and not torch.isfinite(y2[:, 999]).any()
