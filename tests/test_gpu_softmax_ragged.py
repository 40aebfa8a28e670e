"""Softmax rows that are not whole 16-byte vectors: the one-wave kernels over
the aligned vectors that cover a row (shared with its neighbours), at every
start of a row inside a vector, the shortest and longest such rows, and the
scalar kernels on both sides of them.

Against the oracle, tolerances as in test_gpu_rowops.py (fp32 1e-5, bf16 2e-2
of the largest value), and each element against float64: 1e-5 of its terms (the
exponential of an fp32 difference of at most 27: 2e-6, and the fp32 sums), plus,
in bf16, the rounding of the result, 2^-8 of it.
"""
import pytest
import torch

import oracle
from conftest import rel_err

pytestmark = pytest.mark.gpu

DIMS = {torch.float32: [1, 2, 3, 5, 7, 63, 65, 95, 97, 98, 99, 159, 161, 253, 255, 257, 777, 1025, 2045, 2046, 2051],
        torch.bfloat16: [1, 3, 7, 9, 12, 63, 65, 175, 177, 223, 225, 226, 227, 228, 229, 230, 231, 509, 513, 777, 1023, 4082, 4083, 4089]}


def check_elements(got, want, terms, dtype):
    bound = 1e-5 * terms + (0.0 if dtype == torch.float32 else 2.0 ** -8) * want.abs()
    bad = ~((got.double() - want).abs() <= bound)  # a NaN, too
    assert not bad.any(), f"{int(bad.sum())} elements, the first at {bad.nonzero()[0].tolist()}"


def check_exact(s, p, dp, ds, S, dtype):
    """p against the softmax of s, ds against its gradient at p, whole tensors."""
    rows, dim = s.shape
    x = s.double()
    if S:
        lim = torch.arange(rows, device=s.device)[:, None] % S + (dim - S)
        x = x.masked_fill(torch.arange(dim, device=s.device)[None, :] > lim, float("-inf"))
    want = torch.softmax(x, -1)
    check_elements(p, want, want, dtype)
    q, g = p.double(), dp.double()
    terms = q * (g.abs() + (q * g).abs().sum(-1, keepdim=True))
    check_elements(ds, q * (g - (q * g).sum(-1, keepdim=True)), terms, dtype)


@pytest.mark.parametrize("dtype,dim", [(t, d) for t, ds in DIMS.items() for d in ds])
@pytest.mark.parametrize("causal", [False, True])
def test_softmax_ragged_rows(mc, dev, nan_outputs, dtype, dim, causal):
    g = torch.Generator().manual_seed(dim)
    rows = 11 if dim > 300 else 37
    S = min(dim, 6) if causal else 0
    s = (torch.randn(rows, dim, generator=g) * 3).to(dtype)
    dp = torch.randn(rows, dim, generator=g).to(dtype)
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    p = mc.softmax_forward(s.to(dev), S)
    p_ref = oracle.softmax_fwd(s.float().numpy(), causal_rows=S)
    assert rel_err(p, p_ref) <= tol
    ds = mc.softmax_backward(p, dp.to(dev), S)
    ds_ref = oracle.softmax_bwd(p.float().cpu().numpy(), dp.float().numpy(), causal_rows=S)
    assert rel_err(ds, ds_ref) <= tol
    check_exact(s.to(dev), p, dp.to(dev), ds, S, dtype)
    if causal:
        keep = torch.arange(dim)[None, :] <= (torch.arange(rows) % S)[:, None] + (dim - S)
        assert not p.cpu()[~keep].any() and not ds.cpu()[~keep].any()


@pytest.mark.parametrize("dtype,dim", [(torch.float32, 63), (torch.float32, 65), (torch.bfloat16, 111),
                                       (torch.bfloat16, 113)])
@pytest.mark.parametrize("rows", [32767, 32769])
def test_softmax_ragged_many_rows(mc, dev, nan_outputs, dtype, dim, rows):
    """Both sides of the rule for many unmasked rows, whole tensors."""
    g = torch.Generator(device=dev).manual_seed(dim)
    s = (torch.randn(rows, dim, generator=g, device=dev) * 3).to(dtype)
    dp = torch.randn(rows, dim, generator=g, device=dev).to(dtype)
    p = mc.softmax_forward(s)
    ds = mc.softmax_backward(p, dp)
    check_exact(s, p, dp, ds, 0, dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("dim", [3, 61, 777])
def test_softmax_ragged_rows_are_apart(mc, dev, dtype, dim):
    """A row without a finite maximum reaches its own unmasked columns only."""
    g = torch.Generator(device=dev).manual_seed(dim)
    s = torch.randn(24, dim, generator=g, device=dev).to(dtype)
    dp = torch.randn(24, dim, generator=g, device=dev).to(dtype)
    S = 3
    p = mc.softmax_forward(s, S)
    ds = mc.softmax_backward(p, dp, S)
    s2, p2 = s.clone(), p.clone()
    s2[7], s2[13], s2[15] = float("nan"), float("inf"), float("-inf")
    p2[7] = float("nan")
    q = mc.softmax_forward(s2, S)
    ok = [i for i in range(24) if i not in (7, 13, 15)]
    assert torch.equal(q[ok], p[ok])
    e = mc.softmax_backward(p2, dp, S)
    ok = [i for i in range(24) if i != 7]
    assert torch.equal(e[ok], ds[ok])
    for i in (7, 13, 15):
        lim = i % S + dim - S
        assert torch.isnan(q[i, :lim + 1]).any() and not q[i, lim + 1:].any()
