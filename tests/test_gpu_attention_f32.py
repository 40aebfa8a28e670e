"""The float32 matrix-core attention (attention_f32.hip) at its edges: sequence
lengths around the 32-row blocks and the 4-way split of the blocks over a
workgroup's waves, head dims that fill and do not fill the 32 / 64 / 128-wide
tiles, every grouping of a K/V head's query heads in dK/dV, masks, and rows
that a causal query must not see even when they are not finite.

Tolerance as in test_gpu_attention.py: max|out - ref| / max|ref| <= 1e-5
against the oracle (fp32 sums of at most a few hundred terms).
"""
import pytest
import torch

from inputs import gen
from test_gpu_attention import case, check, check_bwd, ref, ref_bwd, run, run_bwd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("S", [1, 31, 32, 33, 64, 97, 128, 161, 290])
@pytest.mark.parametrize("D,causal,masked", [(64, True, False), (128, False, False), (32, True, True), (20, False, True),
                                             (36, True, False), (100, True, True), (4, False, False)])
def test_attention_f32_blocks(mc, dev, S, D, causal, masked):
    q, k, v, mask = case(S + D, 2, 4, 2, S, D, torch.float32, masked)
    o, lse = run(mc, dev, q, k, v, mask, causal)
    o_ref, lse_ref = ref(q, k, v, mask, causal)
    check(o, lse, o_ref, lse_ref, torch.float32)
    dout = torch.randn(2, S, 4 * D, generator=gen(S))
    got = run_bwd(mc, dev, q, k, v, mask, causal, dout)
    check_bwd(got, ref_bwd(q, k, v, mask, causal, dout), torch.float32)


@pytest.mark.parametrize("D,S", [(32, 4), (32, 5), (32, 6), (64, 7), (64, 8), (64, 11), (64, 12), (128, 9), (128, 10),
                                 (100, 15), (100, 16)])
@pytest.mark.parametrize("causal,masked", [(True, False), (False, True)])
def test_attention_f32_short(mc, dev, D, S, causal, masked):
    """Sequences around the lengths from which the tiles take the forward and,
    separately, the backward (whose workspace changes with them)."""
    q, k, v, mask = case(S + D, 2, 4, 4, S, D, torch.float32, masked)
    o, lse = run(mc, dev, q, k, v, mask, causal)
    o_ref, lse_ref = ref(q, k, v, mask, causal)
    check(o, lse, o_ref, lse_ref, torch.float32)
    dout = torch.randn(2, S, 4 * D, generator=gen(S))
    check_bwd(run_bwd(mc, dev, q, k, v, mask, causal, dout), ref_bwd(q, k, v, mask, causal, dout), torch.float32)


@pytest.mark.parametrize("B,H,Hkv,S", [(8, 8, 4, 1000), (8, 16, 4, 500), (8, 24, 4, 400), (1, 6, 1, 100), (2, 3, 3, 70)])
def test_attention_f32_bwd_groups(mc, dev, B, H, Hkv, S):
    """One, two, three and all query heads' partials per K/V head (the groups
    grow until the grid has 1024 workgroups)."""
    D = 8
    q, k, v, _ = case(S, B, H, Hkv, S, D, torch.float32)
    dout = torch.randn(B, S, H * D, generator=gen(S + 1))
    got = run_bwd(mc, dev, q, k, v, None, True, dout)
    check_bwd(got, ref_bwd(q, k, v, None, True, dout), torch.float32)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_attention_f32_unseen_rows_may_be_anything(mc, dev, D, bad):
    """Rows of k, v, q and dout that are not finite reach the causal results
    that see them and no other: the queries before row t0, and the keys after
    it for q and dout, get what they get from finite rows, bit for bit."""
    B, H, Hkv, S, t0 = 1, 4, 2, 75, 45
    q, k, v, _ = case(D, B, H, Hkv, S, D, torch.float32)
    dout = torch.randn(B, S, H * D, generator=gen(D + 3))
    o, lse = run(mc, dev, q, k, v, None, True)
    dq, dk, dv = run_bwd(mc, dev, q, k, v, None, True, dout)
    k2, v2 = k.clone(), v.clone()
    k2[:, :, t0], v2[:, :, t0] = bad, bad
    o2, lse2 = run(mc, dev, q, k2, v2, None, True)
    dq2, _, _ = run_bwd(mc, dev, q, k2, v2, None, True, dout)
    assert torch.equal(o[:, :t0], o2[:, :t0]) and torch.equal(lse[..., :t0], lse2[..., :t0])
    assert torch.equal(dq[:, :, :t0], dq2[:, :, :t0])
    assert not torch.isfinite(o2[:, t0:]).any()
    q2, d2 = q.clone(), dout.clone()
    q2[:, :, t0], d2[:, t0] = bad, bad
    _, dk2, dv2 = run_bwd(mc, dev, q2, k, v, None, True, d2)
    assert torch.equal(dk[:, :, t0 + 1:], dk2[:, :, t0 + 1:]) and torch.equal(dv[:, :, t0 + 1:], dv2[:, :, t0 + 1:])
    assert not torch.isfinite(dk2[:, :, :t0 + 1]).any() and not torch.isfinite(dv2[:, :, :t0 + 1]).any()
