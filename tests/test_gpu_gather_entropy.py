"""Gathered log-probabilities and entropy in one pass (``nrl_gather_entropy_*``) against the fp32 oracle."""

import pytest
import torch

from oracle import distill as OD

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _ops():
    from rl_amd import ops  # noqa: F401  (registers torch.ops.rl_amd)

    return torch.ops.rl_amd


# vocabularies around a vector, a 256-lane step and the four-deep main loop; K of one, of a wave and past the on-chip list
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("vocab,k", [(1, 1), (7, 3), (2047, 64), (8192, 65), (8201, 512), (20011, 513)])
@pytest.mark.parametrize("entropy", [False, True])
def test_gather_entropy_matches_oracle(dtype, vocab, k, entropy):
    g = torch.Generator().manual_seed(vocab + k)
    b, s, n = 2, 4, 3
    logits = (torch.randn(b, s, vocab, generator=g) * 3).to(dtype)
    idx = torch.randint(0, vocab, (b, s, k), generator=g)
    idx[..., -1] = idx[..., 0]  # a repeated index
    up = torch.randn(b, n, k, generator=g)
    up_h = torch.randn(b, n, generator=g)
    up[1, 1], up_h[1, 1] = 0, 0  # a row without any upstream gradient
    xo = logits.float().requires_grad_(True)
    want = OD.gather_logprob(xo[:, :n], idx[:, :n])
    want_h = OD.neg_entropy(xo[:, :n])
    total = (want * up).sum() + ((want_h * up_h).sum() if entropy else 0.0)
    total.backward()

    x = logits.to(DEV)
    out, h, lse = _ops().gather_entropy_fwd(x, idx.to(DEV), n, entropy)
    # fp32 sums over the row in both: 2^-24 of the largest intermediate (|lse| < 32), a few steps deep
    assert (out.cpu() - want.detach()).abs().max().item() <= 1e-5
    if entropy:
        assert (h.cpu() - want_h.detach()).abs().max().item() <= 1e-5
    d = _ops().gather_entropy_bwd(x, idx.to(DEV), n, lse, h if entropy else None, up_h.to(DEV) if entropy else None, up.to(DEV))
    assert d.dtype == dtype and d.shape == logits.shape
    err = (d.float().cpu() - xo.grad).abs()
    # one narrowing to the logits' dtype (half a unit in the last place), fp32 arithmetic of terms as large as the sum of
    # the row's upstream gradients
    scale = up.abs().sum(-1, keepdim=True) + up_h.abs().unsqueeze(-1) * 16
    ulp = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[dtype]
    bound = ulp * xo.grad.abs() + 1e-7 + torch.cat([scale, torch.zeros(b, s - n, 1)], 1) * 4e-6
    assert bool((err <= bound).all()), (err - bound).max()
    assert bool((d[:, n:] == 0).all()) and bool((d[1, 1] == 0).all())


def test_gather_entropy_of_rows_off_the_16_byte_grid():
    g = torch.Generator().manual_seed(5)
    big = torch.randn(2, 5, 3003, generator=g).to(torch.bfloat16)
    view = big.to(DEV)[:, 1:4, 3:3000]
    idx = torch.randint(0, 2997, (2, 3, 8), generator=g)
    out, h, lse = _ops().gather_entropy_fwd(view, idx.to(DEV), 3, True)
    ref = big[:, 1:4, 3:3000].float().requires_grad_(True)
    want, want_h = OD.gather_logprob(ref, idx), OD.neg_entropy(ref)
    assert (out.cpu() - want.detach()).abs().max().item() <= 1e-5
    assert (h.cpu() - want_h.detach()).abs().max().item() <= 1e-5
    up, up_h = torch.randn(2, 3, 8, generator=g), torch.randn(2, 3, generator=g)
    ((want * up).sum() + (want_h * up_h).sum()).backward()
    d = _ops().gather_entropy_bwd(view, idx.to(DEV), 3, lse, h, up_h.to(DEV), up.to(DEV))
    assert bool(((d.float().cpu() - ref.grad).abs() <= 2.0 ** -8 * ref.grad.abs() + 2e-4).all())


def test_minus_infinity_logits_have_no_entropy_and_no_gradient():
    x = torch.tensor([[[0.0, float("-inf"), 1.0, float("-inf")]]], device=DEV)
    idx = torch.zeros(1, 1, 1, dtype=torch.int64, device=DEV)
    out, h, lse = _ops().gather_entropy_fwd(x, idx, 1, True)
    p = torch.softmax(torch.tensor([0.0, 1.0]), -1)
    assert abs(h.item() - (p * p.log()).sum().item()) <= 1e-6
    d = _ops().gather_entropy_bwd(x, idx, 1, lse, h, torch.ones(1, 1, device=DEV), torch.ones(1, 1, 1, device=DEV))
    assert bool(torch.isfinite(d).all()) and d[0, 0, 1].item() == 0.0 and d[0, 0, 3].item() == 0.0


@pytest.mark.parametrize("dtype,value", [(torch.float32, v) for v in (-1e6, 1e12, -1e12, -6e29, -1e30, 3e38, torch.finfo(torch.float32).min)]
                         + [(torch.bfloat16, v) for v in (1e12, -7e29, -1e30, torch.finfo(torch.bfloat16).min)]
                         + [(torch.float16, torch.finfo(torch.float16).min)])
@pytest.mark.parametrize("vocab", [8192, 8201])
def test_flat_rows_of_any_magnitude(dtype, value, vocab):
    """A row whose logits are all alike, as one masked whole is, and the same with one ordinary logit."""
    x = torch.full((1, 2, vocab), value, dtype=dtype, device=DEV)
    x[0, 1, 5] = 1.0 if value < 0 else torch.finfo(dtype).max
    idx = torch.tensor([[[0, 5], [0, 5]]], device=DEV)
    out, h, lse = _ops().gather_entropy_fwd(x, idx, 2, True)
    flat, log_v = x[0, 0, 0].double().item(), torch.tensor(float(vocab)).log().item()
    unit = abs(flat) * 2.0 ** -23  # the log-sum-exp is one fp32 number of this size, the logprobs are differences from it
    assert abs(h[0, 0].item() + log_v) <= 1e-5 and abs(lse[0, 0].double().item() - flat - log_v) <= unit + 1e-5
    assert bool(((out[0, 0].double() + log_v).abs() <= max(unit, log_v if unit > 1 else 0.0) + 1e-5).all())
    assert h[0, 1].item() == 0.0 and lse[0, 1].item() == x[0, 1, 5].float().item() and out[0, 1, 1].item() == 0.0


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_long_rows_keep_the_precision_of_fp32(dtype):
    """2-norm of the error against 64 bits: the log-sum-exp and the difference from it round once each, 2^-24 of numbers up to
    1.5 times the results; sums of 262144 terms must not add to that."""
    g = torch.Generator(device=DEV).manual_seed(9)
    x = (torch.randn(1, 64, 262144, generator=g, device=DEV) * torch.linspace(2, 6, 64, device=DEV).view(1, 64, 1)).to(dtype)
    idx = torch.randint(0, 262144, (1, 64, 32), generator=g, device=DEV)
    out, h, _ = _ops().gather_entropy_fwd(x, idx, 64, True)
    lp = x.double().log_softmax(-1)
    for got, want in ((out, lp.gather(-1, idx)), (h, (lp.exp() * lp).sum(-1))):
        assert ((got.double() - want).norm() / want.norm()).item() <= 2.0 ** -23
