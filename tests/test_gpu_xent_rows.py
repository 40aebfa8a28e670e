"""Cross-entropy rows of any length and start: vocabularies around the vector
and thread counts of the row kernels (256 threads, 1024 where rows are few and
long), rows that start anywhere inside a 16-byte vector, logits that are
themselves not 16-byte aligned, targets in the edges, ignored and non-finite
rows.

Against the composite in float64; the loss to 1e-5, the gradient to 1e-5 (fp32)
and 1e-2 (bf16) of its largest value, and each element of it to 1e-5 of its
terms (p is the exponential of a difference of two fp32 numbers of about 20,
each rounded to 2^-24 of itself: 2.4e-6, and as much again from the fp32
log-sum-exp) plus, in bf16, the rounding of the result, 2^-8 of it.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


def reference(x, t, ignore, eps):
    x = x.double()
    lp = torch.log_softmax(x, -1)
    counted = torch.ones_like(t, dtype=torch.bool) if ignore is None else t != ignore
    n = counted.sum()
    nll = -lp.gather(1, t[:, None].long())[:, 0][counted].sum() / n
    loss = (1 - eps) * nll + eps * -lp.mean()
    p = lp.exp()
    onehot = torch.zeros_like(p).scatter_(1, t[:, None].long(), 1.0)
    a, b = (1 - eps) * counted[:, None] / n, eps / x.shape[0]
    terms = (a * (p + onehot)).add_(b * p).add_(b / x.shape[1])
    return loss, a * (p - onehot) + b * (p - 1.0 / x.shape[1]), torch.logsumexp(x, -1), terms


def check_elements(d, want, terms, dtype):
    bound = 1e-5 * terms + (0.0 if dtype == torch.float32 else 2.0 ** -8) * want.abs()
    bad = ~((d.double() - want).abs() <= bound)  # a NaN, too
    assert not bad.any(), f"{int(bad.sum())} elements, the first at {bad.nonzero()[0].tolist()}"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("V", [1, 2, 7, 9, 17, 255, 1023, 2049, 4096, 8192, 8193, 16384, 33001])
@pytest.mark.parametrize("offset,rows,ignore,eps", [(0, 5, None, 0.0), (3, 33, 0, 0.1), (5, 1030, 0, 0.0)])
def test_xent_rows(mc, dev, nan_outputs, dtype, V, offset, rows, ignore, eps):
    if ignore is not None and V == 1:
        pytest.skip("every target would be ignored")
    g = torch.Generator(device=dev).manual_seed(V + offset)
    buf = torch.randn(rows * V + offset, generator=g, device=dev).mul_(2.0).to(dtype)
    x = buf[offset:].view(rows, V)
    t = torch.randint(0, V, (rows,), generator=g, device=dev, dtype=torch.int32)
    t[0], t[-1] = V - 1, min(1, V - 1)
    loss, stats = mc.cross_entropy_forward(x, t, ignore, eps)
    d = mc.cross_entropy_backward(x, t, stats, None, ignore, eps)
    loss_ref, d_ref, lse_ref, terms = reference(x, t, ignore, eps)
    assert abs(float(loss) - float(loss_ref)) <= 1e-5 * max(1.0, abs(float(loss_ref)))
    assert float((stats[:-1].double() - lse_ref).abs().max()) <= 1e-5 * max(1.0, float(lse_ref.abs().max()))
    tol = 1e-5 if dtype == torch.float32 else 1e-2
    assert float((d.double() - d_ref).abs().max()) <= tol * max(float(d_ref.abs().max()), 1e-30)
    check_elements(d, d_ref, terms, dtype)


@pytest.mark.parametrize("dtype,rows,V,offset", [(torch.bfloat16, 1017, 33001, 3), (torch.bfloat16, 1016, 33001, 3),
                                                 (torch.float32, 2, 8388609, 1), (torch.float32, 2, 8388607, 1)])
def test_xent_gradients_streamed(mc, dev, nan_outputs, dtype, rows, V, offset):
    """Both sides of 64 MB of gradients, past which they are stored past the caches."""
    g = torch.Generator(device=dev).manual_seed(rows)
    x = torch.randn(rows * V + offset, generator=g, device=dev).mul_(2.0).to(dtype)[offset:].view(rows, V)
    t = torch.randint(0, V, (rows,), generator=g, device=dev, dtype=torch.int32)
    loss, stats = mc.cross_entropy_forward(x, t, None, 0.1)
    d = mc.cross_entropy_backward(x, t, stats, None, None, 0.1)
    loss_ref, d_ref, _, terms = reference(x, t, None, 0.1)
    assert abs(float(loss) - float(loss_ref)) <= 1e-5 * abs(float(loss_ref))
    check_elements(d, d_ref, terms, dtype)


@pytest.mark.parametrize("rows,V", [(40, 20001), (1100, 777)])
def test_xent_rows_are_apart(mc, dev, rows, V):
    g = torch.Generator(device=dev).manual_seed(V)
    x = torch.randn(rows, V, generator=g, device=dev)
    t = torch.randint(0, V, (rows,), generator=g, device=dev, dtype=torch.int32)
    _, s0 = mc.cross_entropy_forward(x, t)
    x2 = x.clone()
    x2[7], x2[9] = float("nan"), float("-inf")
    x2[11, V - 1] = float("inf")
    loss, s1 = mc.cross_entropy_forward(x2, t)
    ok = [i for i in range(rows) if i not in (7, 9, 11)]
    assert torch.equal(s0[ok], s1[ok]) and torch.isnan(loss).all()
    assert torch.isnan(s1[7]) and not torch.isfinite(s1[9]) and torch.isnan(s1[11])
