"""The fused lm_head where its products are cut into k ranges and its forward into many vocabulary shares: few tiles and a
long k, tile and slab remainders, a chunk whose tokens are all dead.  Bounds: see ``test_gpu_lmhead.narrowing_bounds``."""

import pytest
import torch

from test_gpu_lmhead import narrowing_bounds

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _ops():
    from rl_amd import ops  # noqa: F401

    return torch.ops.rl_amd


# (tokens, hidden, vocab): dH in many ranges of a ragged k; dH of one token; three token blocks; dW in ranges (few
# vocabulary tiles, thousands of tokens); both products cut, a hidden size off the 64-wide slab
@pytest.mark.parametrize("n,h,v", [(512, 256, 40009), (1, 64, 20000), (700, 128, 9000), (4100, 128, 700), (2050, 72, 4099)])
@pytest.mark.parametrize("keep", [False, True])
def test_split_products_match_oracle(n, h, v, keep):
    g = torch.Generator().manual_seed(n + v)
    hid = torch.randn(n, h, generator=g).to(torch.bfloat16)
    w = (torch.randn(v, h, generator=g) * 0.05).to(torch.bfloat16)
    tgt = torch.randint(0, v, (n,), generator=g)
    up = torch.randn(n, generator=g) * 1e-3
    up[::5] = 0 if n > 1 else 1e-3
    lp, lse, kept = _ops().lmhead_logprob_fwd(hid.to(DEV), w.to(DEV), tgt.to(DEV), 0, v, keep)
    logits = (hid.float() @ w.float().T)
    want = torch.log_softmax(logits, -1).gather(-1, tgt.unsqueeze(-1)).squeeze(-1)
    # one bf16 rounding of every logit (2^-9 of its size), of the target's and averaged in the log-sum-exp
    assert (lp.cpu() - want).abs().max().item() <= 2.0 ** -7 * logits.abs().max().item() + 2e-3
    dh, dw = _ops().lmhead_logprob_bwd(hid.to(DEV), w.to(DEV), tgt.to(DEV), lse, up.to(DEV), 0, v, kept if keep else None)
    o_dh, o_dw, b_dh, b_dw = narrowing_bounds(hid, w, tgt, up)
    assert bool(((dh.cpu() - o_dh).abs() <= b_dh).all())
    assert bool(((dw.float().cpu() - o_dw).abs() <= b_dw).all())
    again = _ops().lmhead_logprob_bwd(hid.to(DEV), w.to(DEV), tgt.to(DEV), lse, up.to(DEV), 0, v, kept if keep else None)
    assert torch.equal(again[0], dh) and torch.equal(again[1], dw)  # partial products are added in a fixed order


# edges of core T's tiles, slabs and fragments: ids, tokens and hidden sizes on either side of 16, 32, 64 and 256
@pytest.mark.parametrize("n,h,v", [(1, 8, 1), (31, 8, 17), (33, 72, 63), (64, 264, 65), (65, 248, 255), (257, 256, 257), (255, 8, 1030), (129, 520, 40)])
@pytest.mark.parametrize("keep", [False, True])
def test_products_at_the_edges_of_tiles(n, h, v, keep):
    g = torch.Generator().manual_seed(n * 1000 + v)
    hid = torch.randn(n, h, generator=g).to(torch.bfloat16)
    w = (torch.randn(v, h, generator=g) * 0.1).to(torch.bfloat16)
    tgt = torch.randint(0, v, (n,), generator=g)
    up = torch.randn(n, generator=g) * 1e-2
    up[1::4] = 0
    _, lse, kept = _ops().lmhead_logprob_fwd(hid.to(DEV), w.to(DEV), tgt.to(DEV), 0, v, keep)
    dh, dw = _ops().lmhead_logprob_bwd(hid.to(DEV), w.to(DEV), tgt.to(DEV), lse, up.to(DEV), 0, v, kept if keep else None)
    o_dh, o_dw, b_dh, b_dw = narrowing_bounds(hid, w, tgt, up)
    assert bool(((dh.cpu() - o_dh).abs() <= b_dh).all())
    assert bool(((dw.float().cpu() - o_dw).abs() <= b_dw).all())


def test_products_of_a_shard_leave_other_ranks_targets_out():
    """A rank that holds ids 100 .. 399: targets elsewhere have a softmax part but no one-hot term."""
    g = torch.Generator().manual_seed(9)
    n, h, v, first = 90, 64, 300, 100
    hid = torch.randn(n, h, generator=g).to(torch.bfloat16)
    w = (torch.randn(v, h, generator=g) * 0.1).to(torch.bfloat16)
    tgt = torch.randint(0, 500, (n,), generator=g)
    up = torch.randn(n, generator=g) * 1e-2
    _, lse, kept = _ops().lmhead_logprob_fwd(hid.to(DEV), w.to(DEV), tgt.to(DEV), first, first + v, True)
    inside = ((tgt >= first) & (tgt < first + v)).float()
    one = torch.nn.functional.one_hot((tgt - first).clamp(0, v - 1), v).float() * inside.unsqueeze(-1)
    p = torch.softmax((hid @ w.T).float(), -1)
    grad = (one - p) * up.unsqueeze(-1)
    mag = (one + 2 * p) * up.abs().unsqueeze(-1)
    for k in (kept, None):
        dh, dw = _ops().lmhead_logprob_bwd(hid.to(DEV), w.to(DEV), tgt.to(DEV), lse, up.to(DEV), first, first + v, k)
        # G narrowed to bf16 (2^-8) from logits narrowed to bf16 (as much again); dW narrowed once more
        assert bool(((dh.cpu() - grad @ w.float()).abs() <= 2.0 ** -7 * ((p * up.abs().unsqueeze(-1)) @ w.float().abs()) + 1e-6).all())
        want = grad.T @ hid.float()
        assert bool(((dw.float().cpu() - want).abs() <= 2.0 ** -7 * (mag.T @ hid.float().abs()) + 2.0 ** -8 * want.abs() + 1e-6).all())


@pytest.mark.parametrize("n,h,v", [(300, 128, 20000), (4096, 64, 600)])
def test_no_live_token_gives_zero_gradients(n, h, v):
    hid = torch.randn(n, h, device=DEV).to(torch.bfloat16)
    w = torch.randn(v, h, device=DEV).to(torch.bfloat16)
    tgt = torch.zeros(n, dtype=torch.int64, device=DEV)
    _, lse, _ = _ops().lmhead_logprob_fwd(hid, w, tgt, 0, v)
    dh, dw = _ops().lmhead_logprob_bwd(hid, w, tgt, lse, torch.zeros(n, device=DEV), 0, v)
    assert bool((dh == 0).all()) and bool((dw == 0).all())


@pytest.mark.parametrize("h", [64, 72])            # both gradient kernels that recompute logits
@pytest.mark.parametrize("v", [4096, 65536])       # dH in one k range and in several
def test_the_one_hot_term_of_dh_is_added_once(h, v):
    """All logits are 0, so G is -g / V exactly (the bf16 nearest to exp(-log V) is the power of two), and dH = g (W[target] -
    mean(W)).  The mean is below 1/2 next to a W[target] of 256 to 384: added to it once, the result is one rounding of 2^-16
    away, besides the short sum's own, 2^-24 of the mean in each of its V / 16 steps.  Inside the running sum every step would
    round at 256."""
    g = torch.Generator().manual_seed(h + v)
    n = 5
    hid = torch.zeros(n, h, dtype=torch.bfloat16)
    w = (torch.rand(v, h, generator=g) * 0.125).to(torch.bfloat16)
    tgt = torch.arange(n) * 17
    w[tgt] = 256 + 2 * torch.randint(0, 64, (n, h), generator=g).to(torch.bfloat16)
    up = torch.tensor([1.0, -1.0, 1.0, 0.0, -1.0])
    _, lse, kept = _ops().lmhead_logprob_fwd(hid.to(DEV), w.to(DEV), tgt.to(DEV), 0, v, True)
    mean = w.double().mean(0)
    want = up.double().unsqueeze(-1) * (w[tgt].double() - mean)
    bound = 2.0 ** -16 + v / 16 * 2.0 ** -24 * mean.max().item()
    for k in (kept, None):
        dh, _ = _ops().lmhead_logprob_bwd(hid.to(DEV), w.to(DEV), tgt.to(DEV), lse, up.to(DEV), 0, v, k)
        assert (dh.double().cpu() - want).abs().max().item() <= bound


@pytest.mark.parametrize("n,h,v,pad", [(300, 256, 2000, 8), (70, 264, 700, 248), (512, 64, 9001, 64), (5, 8, 65, 1016)])
@pytest.mark.parametrize("keep", [False, True])
def test_weights_and_hidden_states_with_rows_further_apart(n, h, v, pad, keep):
    """A weight that is a column slice of a wider one: dH's product reads it with its own row stride.  The same bits as of a copy."""
    g = torch.Generator().manual_seed(n + pad)
    hid = torch.randn(n, h + pad, generator=g).to(torch.bfloat16).to(DEV)[:, pad:]
    w = (torch.randn(v, h + pad, generator=g) * 0.05).to(torch.bfloat16).to(DEV)[:, pad:]
    assert w.stride(0) == h + pad and w.data_ptr() % 16 == 0
    tgt = torch.randint(0, v, (n,), generator=g).to(DEV)
    up = torch.randn(n, generator=g).to(DEV)
    up[1::4] = 0
    out = []
    for a, b in ((hid, w), (hid.contiguous(), w.contiguous())):
        lp, lse, kept = _ops().lmhead_logprob_fwd(a, b, tgt, 0, v, keep)
        out.append((lp, lse) + tuple(_ops().lmhead_logprob_bwd(a, b, tgt, lse, up, 0, v, kept if keep else None)))
    for x, y in zip(*out):
        assert torch.equal(x.view(torch.int16), y.view(torch.int16))
