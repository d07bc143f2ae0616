"""GPU parity: top-k / top-p filtered logprobs (K3) against the CPU oracle.

The oracle filters in fp32 (the training path casts the logits first); tolerances as for the
unfiltered logprobs.  Exact ties at the top-p boundary follow the documented rule (ascending
stable order: larger vocabulary indices survive), which is also what the oracle's stable sort does."""

import math

import pytest
import torch

from oracle import logprob as OL
from oracle import loss as O
from oracle import sampling as OS
from rl_amd.algorithms.logits_sampling_utils import TrainingSamplingParams, apply_top_k_top_p
from rl_amd.algorithms.loss import ClippedPGLossConfig, ClippedPGLossFn, prepare_loss_input
from rl_amd.distributed import model_utils as MU

pytestmark = pytest.mark.gpu
DEV = "cuda"

CASES = [(10, 1.0), (None, 0.9), (10, 0.9), (50, 0.95), (1, 1.0), (300, 0.5), (None, 0.3)]


def _check_grad(got, want_f32, dtype):
    got = got.float().cpu()
    scale = want_f32.abs().max().item() + 1e-30
    if dtype == torch.float32:
        assert (got - want_f32).abs().max().item() <= 1e-4 * scale
    else:
        ulp = 2.0 ** -8
        assert bool(((got - want_f32).abs() <= want_f32.abs() * (ulp + 1e-4) + 1e-4 * scale * ulp + 1e-30).all())


@pytest.mark.parametrize("k,p", CASES)
@pytest.mark.parametrize("dtype,vocab", [(torch.float32, 2003), (torch.bfloat16, 4096)])
def test_sampled_logprob_fwd_bwd_matches_oracle(k, p, dtype, vocab):
    g = torch.Generator().manual_seed(vocab + (k or 0))
    b, s = 2, 7
    logits = (torch.randn(b, s, vocab, generator=g) * 2.5).to(dtype)
    ids = torch.randint(0, vocab, (b, s), generator=g)
    # make most targets likely tokens so that a good share of them survives the filter
    top = logits.float().argmax(-1)
    ids[:, 1:] = torch.where(torch.rand(b, s - 1, generator=g) < 0.7, top[:, :-1], ids[:, 1:])
    up = torch.randn(b, s - 1, generator=g)
    xo = logits.to(torch.float32, copy=True).requires_grad_(True)
    want = OL.from_logits_to_logprobs(xo, ids, top_k=k, top_p=p)
    fin = torch.isfinite(want)
    assert fin.any()
    (torch.where(fin, want, torch.zeros_like(want)) * up).sum().backward()

    xg = logits.to(DEV).requires_grad_(True)
    got = MU.from_parallel_logits_to_logprobs(xg, ids.to(DEV), 0, vocab, None,
                                              sampling_params=TrainingSamplingParams(top_k=k, top_p=p))
    gc = got.cpu()
    assert torch.equal(torch.isfinite(gc), fin)            # the same targets are filtered out
    assert torch.all(gc[~fin] == -math.inf)
    assert (gc[fin] - want.detach()[fin]).abs().max().item() <= (1e-5 if dtype == torch.float32 else 2e-3)
    (torch.where(fin.to(DEV), got, torch.zeros_like(got)) * up.to(DEV)).sum().backward()
    _check_grad(xg.grad, xo.grad, dtype)
    # nothing outside the kept set receives gradient
    keep = OS.keep_mask_rows(logits.float().reshape(-1, vocab), k, p).reshape(b, s, vocab)
    assert torch.all(xg.grad.cpu()[:, :-1][~keep[:, :-1]] == 0)


@pytest.mark.parametrize("k,p", [(10, 1.0), (None, 0.9), (10, 0.9)])
def test_apply_top_k_top_p_standalone(k, p):
    g = torch.Generator().manual_seed(21)
    x = torch.randn(3, 5, 1500, generator=g) * 2
    want_f, want_keep = OS.apply_top_k_top_p(x, k, p)
    xg = x.to(DEV).requires_grad_(True)
    got_f, got_keep = apply_top_k_top_p(xg, k, p)
    assert got_keep.dtype == torch.bool and got_keep.shape == x.shape
    assert torch.equal(got_keep.cpu(), want_keep)
    assert torch.equal(got_f.detach().cpu(), want_f)
    assert torch.equal(got_keep, ~torch.isinf(got_f))
    up = torch.randn(3, 5, 1500, generator=g).to(DEV)
    torch.where(got_keep, got_f, torch.zeros_like(got_f)).mul(up).sum().backward()
    assert torch.equal(xg.grad.cpu(), (up.cpu() * want_keep))
    # switched off: the input comes back untouched
    same, none = apply_top_k_top_p(xg, None, 1.0)
    assert same is xg and none is None


def test_ties_at_the_boundaries():
    vocab = 64
    row = torch.full((vocab,), -5.0)
    row[[3, 17, 40]] = 2.0          # three-way tie for the 2nd..4th largest
    row[9] = 3.0
    x = row.view(1, 1, vocab).repeat(1, 2, 1)
    # top-k = 2 keeps every value tied with the 2nd largest
    _, keep = apply_top_k_top_p(x.to(DEV), 2, 1.0)
    assert sorted(torch.nonzero(keep[0, 0]).flatten().tolist()) == [3, 9, 17, 40]
    # top-p cutting through the tie keeps the larger indices first, like a stable ascending sort
    for p in (0.45, 0.65, 0.85):
        want_f, want_keep = OS.apply_top_k_top_p(x, None, p)
        _, keep = apply_top_k_top_p(x.to(DEV), None, p)
        assert torch.equal(keep.cpu(), want_keep), p


def test_c4_slice_bf16_temperature_topk_topp():
    """benchmark config 4 at reduced rows: V=151936 bf16, T=0.7 (divide in bf16), top_k=50, top_p=0.95."""
    g = torch.Generator().manual_seed(1004)
    vocab, b, s = 151936, 2, 6
    logits = (torch.randn(b, s, vocab, generator=g) * 3).to(torch.bfloat16)
    ids = torch.randint(0, vocab, (b, s), generator=g)
    scaled = (logits.float() * (1.0 / torch.tensor(0.7))).to(torch.bfloat16)   # what the GPU in-place divide yields
    top = scaled.float().argmax(-1)
    ids[:, 1:] = torch.where(torch.rand(b, s - 1, generator=g) < 0.8, top[:, :-1], ids[:, 1:])
    want = OL.from_logits_to_logprobs(scaled.float(), ids, top_k=50, top_p=0.95)
    got = MU.from_parallel_logits_to_logprobs(scaled.to(DEV), ids.to(DEV), 0, vocab, None,
                                              sampling_params=TrainingSamplingParams(top_k=50, top_p=0.95)).cpu()
    fin = torch.isfinite(want)
    assert torch.equal(torch.isfinite(got), fin) and fin.any()
    assert (got[fin] - want[fin]).abs().max().item() <= 2e-3
    # fused temperature at the op level gives the same rows from the unscaled logits
    from rl_amd._lib import NRL_TEMP_RCP

    lp, *_ = torch.ops.rl_amd.topk_topp_logprob_fwd(logits.to(DEV), ids[:, 1:].to(DEV), s - 1, 50, 0.95, 0.7, NRL_TEMP_RCP, False)
    assert torch.equal(lp.cpu(), got)


def _boundary_only(got_keep, want_keep, x, slack):
    """The two masks may differ only in a handful of elements whose values sit at the threshold: the
    oracle's running sum is sequential fp32 over tens of thousands of terms, the kernel's is double."""
    diff = got_keep ^ want_keep
    per_row = diff.reshape(-1, x.shape[-1]).sum(-1)
    assert int(per_row.max()) <= slack, per_row.tolist()
    for r in torch.nonzero(per_row).flatten().tolist():
        xr, dr, wr = x.reshape(-1, x.shape[-1])[r], diff.reshape(-1, x.shape[-1])[r], want_keep.reshape(-1, x.shape[-1])[r]
        thr = xr[wr].min()
        below = xr[~wr].max() if bool((~wr).any()) else thr
        # every disputed element is one of the smallest kept or largest dropped values
        assert float(xr[dr].max()) <= float(thr) + 1e-6 + abs(float(thr)) * 1e-2 and float(xr[dr].min()) >= float(below) - 1e-6 - abs(float(below)) * 1e-2


WIDE = [
    (None, 0.9, 50257, 2.5, torch.float32),      # nucleus of tens of thousands of tokens
    (None, 0.5, 65544, 2.5, torch.bfloat16),     # a small nucleus, but more candidates above the chunk bound than fit
    (None, 0.97, 151936, 1.0, torch.bfloat16),
    (None, 0.9, 151936, 4.0, torch.bfloat16),    # ~700 tokens: too many chunks pass the chunk maxima's bound, the row's own is used
    (None, 0.9, 151936, 5.0, torch.float32),     # ~100 tokens: the bound from the chunk maxima suffices
    (None, 0.9, 151936, 8.0, torch.bfloat16),    # a handful of tokens
    (3000, 1.0, 20000, 2.5, torch.float32),      # top_k beyond the candidate list's reach
    (3000, 0.8, 20000, 1.0, torch.float32),
    (5000, 0.9, 8199, 1.0, torch.bfloat16),      # bf16: many exact ties at both boundaries
    (None, 0.95, 40000, 1.0, torch.float16),     # fp16 keys: two 8-bit digits and one of three bits
    (6000, 0.9, 151936, 1.0, torch.float16),
    (8000, 0.7, 151936, 3.0, torch.bfloat16),    # the top-k and the top-p threshold lie in different leading digits
    (None, 0.999, 151936, 1.0, torch.float32),   # four digits, the threshold among the negative logits
    (20000, 0.6, 50257, 1.5, torch.float32),
]


@pytest.mark.parametrize("k,p,vocab,sigma,dtype", WIDE)
def test_kept_sets_beyond_the_candidate_list(k, p, vocab, sigma, dtype):
    """Rows whose kept set exceeds the 4096-entry on-chip list take the wide-row kernel (a radix descent over the order keys).  Same
    oracle; the top-p boundary may move by a few near-equal elements (see _boundary_only), which moves
    the kept mass by parts in 1e5, hence the 1e-4 bound on the logprobs."""
    g = torch.Generator().manual_seed(vocab + (k or 7))
    b, s = 2, 4
    logits = (torch.randn(b, s, vocab, generator=g) * sigma).to(dtype)
    ids = torch.randint(0, vocab, (b, s), generator=g)
    top = logits.float().argmax(-1)
    ids[:, 1:] = torch.where(torch.rand(b, s - 1, generator=g) < 0.5, top[:, :-1], ids[:, 1:])
    x32 = logits.float()
    want_keep = OS.keep_mask_rows(x32.reshape(-1, vocab), k, p).reshape(b, s, vocab)
    _, got_keep = apply_top_k_top_p(logits.to(DEV), k, p)
    got_keep = got_keep.cpu()
    if p >= 1.0:
        assert torch.equal(got_keep, want_keep)                  # top-k alone: no running sum, exact
    else:
        _boundary_only(got_keep, want_keep, x32, slack=8)
    # logprobs and gradient, judged on the targets both sides keep
    xo = x32.clone().requires_grad_(True)
    want = OL.from_logits_to_logprobs(xo, ids, top_k=k, top_p=p)
    xg = logits.to(DEV).requires_grad_(True)
    got = MU.from_parallel_logits_to_logprobs(xg, ids.to(DEV), 0, vocab, None,
                                              sampling_params=TrainingSamplingParams(top_k=k, top_p=p))
    gc = got.detach().cpu()
    tgt_keep_w = torch.isfinite(want.detach())
    tgt_keep_g = torch.isfinite(gc)
    both = tgt_keep_w & tgt_keep_g
    assert both.any() and int((tgt_keep_w ^ tgt_keep_g).sum()) <= 1
    assert (gc[both] - want.detach()[both]).abs().max().item() <= (1e-4 if dtype == torch.float32 else 2e-3)
    up = torch.randn(b, s - 1, generator=g)
    (torch.where(both, want, torch.zeros_like(want)) * up).sum().backward()
    (torch.where(both.to(DEV), got, torch.zeros_like(got)) * up.to(DEV)).sum().backward()
    gg, wg = xg.grad.float().cpu()[:, :-1], xo.grad[:, :-1]
    agree = ~(got_keep ^ want_keep)[:, :-1]
    scale = wg.abs().max().item() + 1e-30
    tol = 1e-4 if dtype == torch.float32 else 2.0 ** -7
    assert bool((((gg - wg).abs() <= wg.abs() * tol + 1e-4 * scale) | ~agree).all())
    assert torch.all(gg[~got_keep[:, :-1]] == 0)


def test_top_p_cut_at_multiples_of_the_wave_width():
    """The finish phase walks the sorted candidates 64 at a time; kept sets of exactly 64, 128, 192 ... entries
    put the cut on the first element of such a block.  Crafted rows (distinct descending values above a
    negligible floor) and seeded Gaussian rows whose nuclei happen to be 1024 and 576 tokens wide."""
    vocab = 5000
    for n_keep, n_top in ((64, 100), (128, 200), (192, 300), (256, 257), (63, 100), (65, 100)):
        # n_top tokens with probabilities ~ 1/n_top each (slightly decreasing), the rest negligible; the cut
        # 1 - p falls between the cumulative mass of n_top - n_keep and n_top - n_keep + 1 of the smallest
        logit = torch.full((vocab,), -60.0)
        vals = 2.0 + torch.linspace(0.0, 0.01, n_top)            # ascending, almost equal
        idx = torch.randperm(vocab, generator=torch.Generator().manual_seed(n_keep))[:n_top]
        logit[idx] = vals
        prob = torch.softmax(logit.double(), -1)[idx]             # ascending like vals
        cum = prob.cumsum(0)
        n_drop = n_top - n_keep
        cut = float((cum[n_drop - 1] + cum[n_drop]) / 2)
        p = 1.0 - cut
        x = logit.view(1, 1, vocab).repeat(1, 2, 1)
        want = OS.keep_mask_rows(x.reshape(-1, vocab), None, p).reshape(x.shape)
        assert int(want[0, 0].sum()) == n_keep
        _, keep = apply_top_k_top_p(x.to(DEV), None, p)
        assert torch.equal(keep.cpu(), want), n_keep
        _, keep_k = apply_top_k_top_p(x.to(DEV), n_top + 50, p)   # the same cut reached through the top-k path
        assert torch.equal(keep_k.cpu(), OS.keep_mask_rows(x.reshape(-1, vocab), n_top + 50, p).reshape(x.shape)), n_keep
    g = torch.Generator().manual_seed(0)
    x = (torch.randn(1, 32, 151936, generator=g) * 4.0).to(torch.bfloat16)
    want = OS.keep_mask_rows(x.float().reshape(-1, 151936), None, 0.9).reshape(x.shape)
    _, keep = apply_top_k_top_p(x.to(DEV), None, 0.9)
    assert torch.equal(keep.cpu(), want)


def test_wide_rows_with_masked_vocabulary_entries():
    """-inf logits (a masked part of the vocabulary) carry no mass and are never kept, also on the
    wide-row path; a top_k that reaches into them keeps only finite entries plus nothing else."""
    g = torch.Generator().manual_seed(77)
    vocab = 30011
    x = torch.randn(1, 3, vocab, generator=g) * 0.5
    x[..., torch.randperm(vocab, generator=g)[: vocab // 10]] = -math.inf
    ids = torch.randint(0, vocab, (1, 3), generator=g)
    for k, p in ((None, 0.9), (6000, 0.95), (6000, 1.0)):
        want_keep = OS.keep_mask_rows(x.reshape(-1, vocab), k, p).reshape(x.shape)
        _, keep = apply_top_k_top_p(x.to(DEV), k, p)
        keep = keep.cpu()
        assert not bool(keep[torch.isinf(x)].any())
        if p >= 1.0:
            assert torch.equal(keep, want_keep)
        else:
            _boundary_only(keep, want_keep, x, slack=8)
        want = OL.from_logits_to_logprobs(x, ids, top_k=k, top_p=p)
        got = MU.from_parallel_logits_to_logprobs(x.to(DEV), ids.to(DEV), 0, vocab, None,
                                                  sampling_params=TrainingSamplingParams(top_k=k, top_p=p)).cpu()
        both = torch.isfinite(want) & torch.isfinite(got)
        assert int((torch.isfinite(want) ^ torch.isfinite(got)).sum()) <= 1
        if both.any():
            assert (got[both] - want[both]).abs().max().item() <= 1e-4


def test_every_token_tied_under_top_p_alone():
    """151936 equal logits: the nucleus is ~144k tokens wide and the cut runs through one giant tie, where
    the smallest indices fall.  The oracle's sequential fp32 sum of 151936 equal terms drifts, so the
    count is compared with the exact one (drop floor((1 - p) V) tokens) and with the oracle loosely."""
    vocab, p = 151936, 0.95
    x = torch.zeros(1, 2, vocab, device=DEV)
    _, keep = apply_top_k_top_p(x, None, p)
    keep = keep[0, 0].cpu()
    n_drop = int((~keep).sum())
    cut = float(torch.tensor(1.0) - torch.tensor(p))           # 1 - p in fp32, as the kernel forms it
    assert abs(n_drop - math.floor(cut * vocab)) <= 1
    assert not keep[:n_drop].any() and keep[n_drop:].all()      # the dropped ones are the smallest indices
    want_keep = OS.keep_mask_rows(torch.zeros(1, vocab), None, p)[0]
    assert int((want_keep ^ keep).sum()) <= 64
    ids = torch.tensor([[5, vocab - 1]], device=DEV)
    lp = MU.from_parallel_logits_to_logprobs(x, ids, 0, vocab, None, sampling_params=TrainingSamplingParams(top_p=p)).cpu()
    assert abs(lp[0, 0].item() + math.log(vocab - n_drop)) <= 1e-5


def test_prepare_loss_input_with_sampling_and_kl():
    """loss/utils.py:97-118 of the reference: filtered logprobs with -inf masked to 0, plus unfiltered
    logprobs for the KL term; end-to-end loss and dlogits against the oracle."""
    g = torch.Generator().manual_seed(31)
    b, s, vocab = 3, 12, 777
    logits = torch.randn(b, s, vocab, generator=g) * 2
    ids = torch.randint(0, vocab, (b, s), generator=g)
    top = logits.argmax(-1)
    ids[:, 1:] = torch.where(torch.rand(b, s - 1, generator=g) < 0.6, top[:, :-1], ids[:, 1:])
    tm = torch.ones(b, s, dtype=torch.int64)
    tm[:, :3] = 0
    data = {"input_ids": ids, "token_mask": tm, "sample_mask": torch.ones(b), "advantages": torch.randn(b, s, generator=g),
            "prev_logprobs": -torch.rand(b, s, generator=g), "generation_logprobs": -torch.rand(b, s, generator=g),
            "reference_policy_logprobs": -torch.rand(b, s, generator=g) * 5}
    gs, gt = torch.tensor(float(b)), (tm[:, 1:]).sum().float()
    k, p = 20, 0.9
    xo = logits.clone().requires_grad_(True)
    lp_f = OL.next_token_logprobs(ids, xo, top_k=k, top_p=p)
    lp_f = OL.mask_out_neg_inf_logprobs(lp_f, (tm[:, 1:] * 1.0))
    lp_u = OL.next_token_logprobs(ids, xo)
    want, wm = O.clipped_pg_loss(O.LossConfig(reference_policy_kl_penalty=0.05), lp_f, {**data, "curr_logprobs_unfiltered": lp_u}, gs, gt)
    want.backward()

    fn = ClippedPGLossFn(ClippedPGLossConfig(reference_policy_kl_penalty=0.05))
    xg = logits.to(DEV).requires_grad_(True)
    ddev = {kk: v.to(DEV) for kk, v in data.items()}
    loss_input, ddev = prepare_loss_input(xg, ddev, fn, sampling_params=TrainingSamplingParams(top_k=k, top_p=p))
    assert "curr_logprobs_unfiltered" in ddev
    got, gm = fn(data=ddev, global_valid_seqs=gs.to(DEV), global_valid_toks=gt.to(DEV), **loss_input)
    got.backward()
    assert abs(got.item() - want.item()) <= 1e-4 * abs(want.item()) + 1e-6
    for kk in wm:
        assert abs(float(gm[kk]) - float(wm[kk])) <= 1e-4 * abs(float(wm[kk])) + 1e-6, kk
    scale = xo.grad.abs().max().item()
    assert (xg.grad.cpu() - xo.grad).abs().max().item() <= 1e-4 * scale


@pytest.mark.parametrize("pre_rolled", [False, True])
def test_packed_sequences_with_sampling(pre_rolled):
    g = torch.Generator().manual_seed(41)
    lens, vocab, smax = [9, 14, 0, 6], 600, 14
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    ids = torch.zeros(len(lens), smax, dtype=torch.int64)
    for i, n in enumerate(lens):
        ids[i, :n] = torch.randint(0, vocab, (n,), generator=g)
    logits = torch.randn(1, int(cu[-1]), vocab, generator=g) * 2
    targets = OL.pack_input_ids(ids, cu, cu, roll_shift=-1 if pre_rolled else 0)
    want = OL.packed_logits_to_logprobs(logits, targets, cu, smax, top_k=15, top_p=0.9, target_is_pre_rolled=pre_rolled)
    got = MU.from_parallel_logits_to_logprobs_packed_sequences(
        logits.to(DEV), targets.to(DEV), cu.to(DEV), smax, 0, vocab, None,
        sampling_params=TrainingSamplingParams(top_k=15, top_p=0.9), target_is_pre_rolled=pre_rolled).cpu()
    fin = torch.isfinite(want)
    assert torch.equal(torch.isfinite(got), fin)
    assert (got[fin] - want[fin]).abs().max().item() <= 1e-5


def test_sampling_autograd_classes():
    g = torch.Generator().manual_seed(51)
    vocab = 999
    x = torch.randn(2, 6, vocab, generator=g) * 2
    t = x.argmax(-1)
    want = OL.rows_logprob_sampled(x, t, 10, 0.9)
    xg = x.to(DEV).requires_grad_(True)
    a = MU.DistributedLogprobWithSampling.apply(xg, t.to(DEV), None, 10, 0.9, False)
    c = MU.ChunkedDistributedLogprobWithSampling.apply(xg, t.to(DEV), None, 10, 0.9, 2, False)
    assert torch.equal(a, c)
    torch.testing.assert_close(a.cpu(), want, rtol=0, atol=1e-5)
    ga, = torch.autograd.grad(a.sum(), xg)
    xo = x.clone().requires_grad_(True)
    OL.rows_logprob_sampled(xo, t, 10, 0.9).sum().backward()
    torch.testing.assert_close(ga.cpu(), xo.grad, rtol=1e-4, atol=1e-6)


@pytest.mark.parametrize("dtype,vocab", [(torch.float32, 2003), (torch.bfloat16, 4096), (torch.float16, 5001)])
@pytest.mark.parametrize("k,p,temperature", [(50, 0.95, 0.7), (10, 1.0, 1.0), (None, 0.9, 1.3), (100, 0.99, 1.0), (1, 1.0, 1.0)])
def test_backward_from_the_kept_set_record_equals_the_streaming_backward(dtype, vocab, k, p, temperature):
    """With the forward's record of the kept sets (count, indices, scaled logits per row) the backward writes a
    gradient row as zeros plus those entries and never reads the logits; without it, it streams the row.  Both
    must give the same bits (with ``top_k = 1`` the one kept entry of a row whose target survived is a zero whose
    sign is that of ``-g``: the scalar store of the record path and the vector store of the streaming path have to
    narrow a negative zero alike) -- also for rows whose kept set exceeds the record's capacity (here: a row of exact ties
    under top-k, a flat row under top-p), which fall back to streaming inside the same launch, and for rows with a
    zero upstream gradient."""
    from rl_amd._lib import NRL_TEMP_DIV, NRL_TEMP_RCP

    g = torch.Generator().manual_seed(vocab + (k or 0))
    b, s = 3, 9
    n = s - 1
    logits = (torch.randn(b, s, vocab, generator=g) * 3.0).to(dtype)
    logits[1, 2] = 0.5                      # every id tied: the kept set is the whole row (beyond any capacity)
    logits[2, 4] = (torch.randn(vocab, generator=g) * 0.01).to(dtype)   # flat: thousands of ids under top-p
    ids = torch.randint(0, vocab, (b, s), generator=g)
    top = logits.float().argmax(-1)
    ids[:, 1:] = torch.where(torch.rand(b, n, generator=g) < 0.7, top[:, :-1], ids[:, 1:])
    up = torch.randn(b, n, generator=g)
    up[0, 3] = 0.0
    x, t, u = logits.to(DEV), ids[:, 1:].contiguous().to(DEV), up.to(DEV)
    kk, pp = (k or 0), (p if p is not None else 1.0)
    ops = torch.ops.rl_amd
    for mode in (NRL_TEMP_RCP, NRL_TEMP_DIV):
        for cap in (8, 64, 128):
            lp, thr, tie, lse, _ = ops.topk_topp_logprob_fwd(x, t, n, kk, pp, temperature, mode, False)
            lp2, thr2, tie2, lse2, _, cnt, idx, val = ops.topk_topp_logprob_fwd_rec(x, t, n, kk, pp, temperature, mode, False, cap)
            assert torch.equal(lp, lp2) and torch.equal(thr, thr2) and torch.equal(tie, tie2) and torch.equal(lse, lse2)
            assert bool(((cnt >= -1) & (cnt <= cap)).all())
            if k is not None and cap >= k and dtype == torch.float32:   # (16-bit rows tie at the threshold: more than k kept)
                assert int(cnt[0, 0]) >= 1                       # an ordinary row is on record
                assert int(cnt[1, 2]) == -1                      # the all-tied row is not
            streamed = ops.topk_topp_logprob_bwd(x, t, thr, tie, lse, u, n, temperature, mode)
            recorded = ops.topk_topp_logprob_bwd(x, t, thr, tie, lse, u, n, temperature, mode, cnt, idx, val)
            assert torch.equal(streamed.view(torch.int16 if dtype != torch.float32 else torch.int32),
                               recorded.view(torch.int16 if dtype != torch.float32 else torch.int32))
            # the record is the kept set: as many entries as the streamed row has kept elements
            keep_rows = OS.keep_mask_rows((logits.float() / temperature if temperature != 1.0 else logits.float())
                                          .reshape(-1, vocab), k, p).reshape(b, s, vocab)[:, :-1]
            on_record = (cnt >= 0).cpu()
            if temperature == 1.0:
                assert torch.equal(cnt.cpu()[on_record].long(), keep_rows.sum(-1)[on_record])


def test_record_entries_outside_their_ranges_are_not_followed():
    """A count above the record's capacity is not a count the forward writes: that row is streamed like a row without
    a record.  An index outside the vocabulary is skipped.  Neither makes the backward write outside its row."""
    from rl_amd._lib import NRL_TEMP_RCP

    g = torch.Generator().manual_seed(77)
    b, s, vocab, cap = 2, 7, 3001, 64
    n = s - 1
    x = (torch.randn(b, s, vocab, generator=g) * 3.0).to(torch.bfloat16).to(DEV)
    t = x.float().argmax(-1)[:, :n].contiguous()
    u = torch.randn(b, n, generator=g).to(DEV)
    ops = torch.ops.rl_amd
    _, thr, tie, lse, _, cnt, idx, val = ops.topk_topp_logprob_fwd_rec(x, t, n, 20, 0.95, 1.0, NRL_TEMP_RCP, False, cap)
    streamed = ops.topk_topp_logprob_bwd(x, t, thr, tie, lse, u, n, 1.0, NRL_TEMP_RCP)
    assert int(cnt[0, 1]) > 0 and int(cnt[1, 3]) > 1
    bad_cnt = cnt.clone()
    bad_cnt[0, 1] = cap + 5
    got = ops.topk_topp_logprob_bwd(x, t, thr, tie, lse, u, n, 1.0, NRL_TEMP_RCP, bad_cnt, idx, val)
    assert torch.equal(got.view(torch.int16), streamed.view(torch.int16))
    bad_idx = idx.clone()
    skipped = int(bad_idx[1, 3, 1])
    bad_idx[1, 3, 1] = vocab + 12345
    got = ops.topk_topp_logprob_bwd(x, t, thr, tie, lse, u, n, 1.0, NRL_TEMP_RCP, cnt, bad_idx, val)
    want = streamed.clone()
    want[1, 3, skipped] = 0.0
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


@pytest.mark.parametrize("dtype,vocab", [(torch.bfloat16, 4096), (torch.float32, 2003)])
def test_record_backward_written_over_the_logits(dtype, vocab):
    """``dlogits`` may alias the logits, as for ``nrl_logprob_bwd``.  With the kept-set record the out-of-place call
    clears the gradient block first and only adds the entries; over the logits that would destroy the rows that are
    not on record (an all-tied row, a flat row) before they are streamed, so such a call must not clear: the in-place
    result equals the out-of-place one bit for bit."""
    import ctypes as C

    from rl_amd import _lib
    from rl_amd._lib import NRL_TEMP_RCP
    from rl_amd.ops import _ptr, _rows, _stream

    g = torch.Generator().manual_seed(vocab)
    b, s, cap = 3, 9, 64
    logits = (torch.randn(b, s, vocab, generator=g) * 3.0).to(dtype)
    logits[1, 2] = 0.5                      # every id tied: not on record
    logits[2, 4] = (torch.randn(vocab, generator=g) * 0.01).to(dtype)   # flat under top-p: not on record
    ids = torch.randint(0, vocab, (b, s), generator=g)
    ids[:, 1:] = torch.where(torch.rand(b, s - 1, generator=g) < 0.7, logits.float().argmax(-1)[:, :-1], ids[:, 1:])
    up = torch.randn(b, s - 1, generator=g)
    up[0, 3] = 0.0
    n = s - 1
    x, t, u = logits.to(DEV), ids[:, 1:].contiguous().to(DEV), up.to(DEV)
    ops = torch.ops.rl_amd
    _, thr, tie, lse, _, cnt, idx, val = ops.topk_topp_logprob_fwd_rec(x, t, n, 20, 0.95, 1.0, NRL_TEMP_RCP, False, cap)
    assert int(cnt[1, 2]) == -1 and int(cnt[0, 0]) >= 1
    want = ops.topk_topp_logprob_bwd(x, t, thr, tie, lse, u, n, 1.0, NRL_TEMP_RCP, cnt, idx, val)
    over = x.clone()
    rows = _rows(over, t, n, 0, vocab, 1.0, NRL_TEMP_RCP)
    with torch.cuda.device(over.device):
        code = _lib.load().nrl_topk_topp_logprob_bwd(
            C.byref(rows), _ptr(thr), _ptr(tie), _ptr(lse), _ptr(u), u.stride(0), u.stride(1),
            _ptr(cnt), _ptr(idx), _ptr(val), cap, _ptr(over), s, over.stride(0), over.stride(1), _stream())
    _lib.check(code, "nrl_topk_topp_logprob_bwd")
    torch.cuda.synchronize()
    bits = torch.int16 if dtype != torch.float32 else torch.int32
    assert torch.equal(over.view(bits), want.view(bits))


def test_wide_rows_come_out_the_same_every_time():
    """The histograms of the wide-row kernel are filled with LDS atomics in whatever order the waves arrive; its
    masses are integers, so the sums, and with them threshold, tie index and log-sum-exp, do not depend on that
    order: repeated calls agree bit for bit."""
    from rl_amd._lib import NRL_TEMP_RCP

    g = torch.Generator().manual_seed(5)
    vocab, n = 151936, 24
    x = torch.randn(1, n + 1, vocab, generator=g).to(torch.bfloat16).to(DEV)
    t = torch.randint(0, vocab, (1, n), generator=g).to(DEV)
    ops = torch.ops.rl_amd
    first = ops.topk_topp_logprob_fwd(x, t, n, 0, 0.95, 0.7, NRL_TEMP_RCP, True)
    assert bool((first[2] >= 0).all())                       # every row resolved
    for _ in range(4):
        again = ops.topk_topp_logprob_fwd(x, t, n, 0, 0.95, 0.7, NRL_TEMP_RCP, True)
        for a, b in zip(first, again):
            assert torch.equal(a.view(torch.int32), b.view(torch.int32))


@pytest.mark.parametrize("nucleus", [500, 512, 513, 700, 1300, 3900])
def test_nuclei_around_the_length_that_is_summed_in_double(nucleus):
    """Top-p alone with about `nucleus` kept ids, against 64-bit sums: the kept set is the heaviest ids, holds top_p of the mass and
    would not without its lightest (both up to 1e-5, the fp32 rounding of the log-sum-exp and of thousands of quotients), and
    logprobs are normalised over exactly that set."""
    from rl_amd.distributed.sampling_logprob import filter_logits, rows_logprob_sampled

    g = torch.Generator(device="cuda").manual_seed(nucleus)
    rows, vocab, top_p = 24, 30000, 0.95
    x = torch.randn(1, rows, vocab, generator=g, device="cuda") * 0.3 - 9.0
    heavy = torch.rand(rows, vocab, generator=g, device="cuda").topk(nucleus + 40, dim=-1).indices
    x[0].scatter_(1, heavy, torch.randn(rows, nucleus + 40, generator=g, device="cuda") * 0.3)
    _, keep = filter_logits(x, None, top_p)
    x64, keep = x[0].double(), keep[0]
    p = x64.softmax(-1)
    mass, lightest = (p * keep).sum(-1), p.masked_fill(~keep, 2.0).amin(-1)
    assert int(keep.sum(-1).amin()) > nucleus // 2
    assert bool((mass >= top_p - 1e-5).all()) and bool((mass - lightest <= top_p + 1e-5).all())
    assert bool((x64.masked_fill(keep, -1e9).amax(-1) <= x64.masked_fill(~keep, 1e9).amin(-1)).all())
    ids = x[0].argmax(-1)
    lp = rows_logprob_sampled(x, ids[None], rows, None, top_p, inference_only=True)[0]
    want = x64.gather(-1, ids[:, None])[:, 0] - x64.masked_fill(~keep, float("-inf")).logsumexp(-1)
    torch.testing.assert_close(lp.double(), want, rtol=0, atol=3e-6)  # fp32 logarithm and difference of values up to 9


@pytest.mark.parametrize("vocab", [900, 2048, 9001, 40000])
@pytest.mark.parametrize("top_k", [1, 50, 400, 2000])
def test_fp32_rows_that_share_their_leading_bits(vocab, top_k):
    """Logits around +-1e4 and 1e6 differ in their last bits only, logits of one value in none, logits at 1e-30 in all but their
    first: the k-th largest and its ties come out as a sort gives them."""
    g = torch.Generator().manual_seed(vocab + top_k)
    n = 9
    x = torch.randn(1, n + 1, vocab, generator=g) * 3
    for i, off in enumerate((0.0, 1e4, -1e4, 1e6, 30.0)):
        x[0, i] += off
    x[0, 5] = 2.5
    x[0, 6] *= 1e-30
    x[0, 7] = (x[0, 7] * 4).round() / 4 + 1e4
    x[0, 8, ::2] = float("-inf")
    x = x.to(DEV)
    from rl_amd import ops  # noqa: F401
    from rl_amd._lib import NRL_TEMP_RCP

    t = x[:, :n].argmax(-1)
    lp, thr, tie, lse, _ = torch.ops.rl_amd.topk_topp_logprob_fwd(x, t, n, top_k, 1.0, 1.0, NRL_TEMP_RCP, False)
    want = x[0, :n].topk(min(top_k, vocab), -1).values[:, -1]
    if top_k > vocab // 2:
        want[8] = x[0, 8][x[0, 8].isfinite()].min()   # -inf is never kept
    assert torch.equal(thr[0], want) and not bool(tie.any())
    z = x[0, :n].double()
    full = z.masked_fill(z < want[:, None], float("-inf")).logsumexp(-1)
    assert bool(((lse[0].double() - full).abs() <= 2.0 ** -23 * (2 + full.abs() + z.amax(-1).abs())).all())


def test_fp32_rows_around_1e4_take_no_longer():
    """A bound too coarse for such logits lets a whole row pass and sends it to the kernel for wide rows: 5 times as long."""
    from rl_amd import ops  # noqa: F401
    from rl_amd._lib import NRL_TEMP_RCP

    g = torch.Generator(device=DEV).manual_seed(1)
    n, vocab = 256, 151936
    x = torch.empty((1, n + 1, vocab), device=DEV).normal_(0, 3, generator=g)
    t = torch.randint(0, vocab, (1, n), generator=g, device=DEV)

    def shortest(x):
        times = []
        for _ in range(8):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(8):
                torch.ops.rl_amd.topk_topp_logprob_fwd(x, t, n, 50, 0.95, 1.0, NRL_TEMP_RCP, False)
            b.record()
            torch.cuda.synchronize()
            times.append(a.elapsed_time(b))
        return min(times)

    shortest(x)
    assert shortest(x + 1e4) < 2 * shortest(x)
