"""Softmax rows that are not whole 16-byte vectors: the one-wave kernels over
the aligned vectors that cover a row (shared with its neighbours), at every
start of a row inside a vector, the shortest and longest such rows, and the
scalar kernels on both sides of them.

Against the oracle, tolerances as in test_gpu_rowops.py (fp32 1e-5, bf16 2e-2
of the largest value).
"""
import pytest
import torch

import oracle
from conftest import rel_err

pytestmark = pytest.mark.gpu

DIMS = {torch.float32: [1, 2, 3, 5, 7, 63, 65, 95, 97, 98, 99, 159, 161, 253, 255, 257, 777, 1025, 2045, 2046, 2051],
        torch.bfloat16: [1, 3, 7, 9, 12, 63, 65, 175, 177, 223, 225, 226, 227, 228, 229, 230, 231, 509, 513, 777, 1023, 4082, 4083, 4089]}


@pytest.mark.parametrize("dtype,dim", [(t, d) for t, ds in DIMS.items() for d in ds])
@pytest.mark.parametrize("causal", [False, True])
def test_softmax_ragged_rows(mc, dev, dtype, dim, causal):
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
    if causal:
        keep = torch.arange(dim)[None, :] <= (torch.arange(rows) % S)[:, None] + (dim - S)
        assert not p.cpu()[~keep].any() and not ds.cpu()[~keep].any()


@pytest.mark.parametrize("dtype,dim", [(torch.float32, 63), (torch.float32, 65), (torch.bfloat16, 111),
                                       (torch.bfloat16, 113)])
@pytest.mark.parametrize("rows", [32767, 32769])
def test_softmax_ragged_many_rows(mc, dev, dtype, dim, rows):
    """Both sides of the rule for many unmasked rows, whole tensors."""
    g = torch.Generator(device=dev).manual_seed(dim)
    s = (torch.randn(rows, dim, generator=g, device=dev) * 3).to(dtype)
    dp = torch.randn(rows, dim, generator=g, device=dev).to(dtype)
    p = mc.softmax_forward(s)
    ds = mc.softmax_backward(p, dp)
    want = torch.softmax(s.double(), -1)
    q = p.double()
    wds = q * (dp.double() - (q * dp.double()).sum(-1, keepdim=True))
    tol = 1e-5 if dtype == torch.float32 else 2e-2
    assert float((q - want).abs().max()) <= tol * float(want.max())
    assert float((ds.double() - wds).abs().max()) <= tol * float(wds.abs().max())


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
