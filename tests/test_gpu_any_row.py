"""The single pass over rows off the 16-byte grid or longer than the chip holds, reached through the wrappers, against the
CPU oracle and the three-pass path.  They sum a row's exponentials in different orders (about 1e-6 in the log-sum-exp), and round a gradient
element to its type once: neighbouring 16-bit values may differ, fp32 values by 1e-4 of the largest as in test_gpu_fused."""

import pytest
import torch

from oracle import logprob as OL
from oracle import loss as O
from rl_amd.algorithms.logits_sampling_utils import TrainingSamplingParams
from rl_amd.algorithms.loss import (
    ClippedPGLossConfig,
    ClippedPGLossFn,
    SequencePackingFusionLossWrapper,
    prepare_loss_input,
    prepare_packed_loss_input,
    wrap_loss_fn_with_input_preparation,
)
from rl_amd.algorithms.loss.fused import any_row_fusable, any_row_fusable_packed, why_not_fusable
from rl_amd.temperature import apply_temperature_scaling, deferred_temperature
from test_gpu_fused import _batch, _close

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _same_gradient(got, want, dtype):
    got, want = got.float(), want.float()
    scale = want.abs().max().item()
    step = 0.0 if dtype == torch.float32 else 2.0 ** -7
    assert bool(((got - want).abs() <= want.abs() * (step + 1e-4) + 1e-4 * scale * (1.0 if dtype == torch.float32 else 2.0 ** -8)).all())


def _three_pass(x, data, fn, gs, gt, **kw):
    loss_input, d2 = prepare_loss_input(x, dict(data), fn, **kw)
    return fn(data=d2, global_valid_seqs=gs, global_valid_toks=gt, **loss_input)


def _setup(b, s, vocab, dtype):
    logits, data, gs, gt = _batch(b, s, vocab, dtype, seed=vocab)
    return logits.to(DEV), {k: v.to(DEV) for k, v in data.items()}, gs.to(DEV), gt.to(DEV)


SHAPES = [
    (torch.bfloat16, 513), (torch.bfloat16, 4103), (torch.bfloat16, 24581), (torch.bfloat16, 40961), (torch.bfloat16, 50257),
    (torch.bfloat16, 81927), (torch.bfloat16, 98305), (torch.bfloat16, 163841), (torch.bfloat16, 163848), (torch.bfloat16, 262144),
    (torch.bfloat16, 229381), (torch.float16, 50257), (torch.float16, 170003), (torch.float32, 257), (torch.float32, 20483),
    (torch.float32, 81921), (torch.float32, 81924), (torch.float32, 98308), (torch.float32, 151936), (torch.float32, 262143),
]


@pytest.mark.parametrize("dtype,vocab", SHAPES)
def test_rows_of_any_length_and_alignment(dtype, vocab):
    logits, data, gs, gt = _setup(3, 7, vocab, dtype)
    data["input_ids"][0, 4] = vocab - 1  # a target in the tail, and one in front of the first boundary of its row
    data["input_ids"][0, 5] = 0
    fn = ClippedPGLossFn(ClippedPGLossConfig())
    xf, xu = (logits.clone().requires_grad_(True) for _ in range(2))
    assert why_not_fusable(fn, xf, data) is not None and any_row_fusable(fn, xf, data)
    got, gm = wrap_loss_fn_with_input_preparation(xf, data, gs, gt, fn, prepare_loss_input)
    want, wm = _three_pass(xu, data, fn, gs, gt)
    assert _close(got.item(), want.item(), rel=1e-4)
    for k in wm:
        assert _close(float(gm[k]), float(wm[k])), k
    got.backward()
    want.backward()
    _same_gradient(xf.grad, xu.grad, dtype)


@pytest.mark.parametrize("dtype,vocab", [(torch.bfloat16, 1027), (torch.float32, 90001)])
def test_more_rows_than_workgroups_and_other_factors(dtype, vocab):
    """An upstream factor that is no power of two (rounded once), and a second backward through the same graph."""
    logits, data, gs, gt = _setup(4, 300 if vocab < 2000 else 90, vocab, dtype)
    fn = ClippedPGLossFn(ClippedPGLossConfig(reference_policy_kl_penalty=0.0, ratio_clip_min=0.2, ratio_clip_max=0.28))
    xf, xu = (logits.clone().requires_grad_(True) for _ in range(2))
    got, _ = wrap_loss_fn_with_input_preparation(xf, data, gs, gt, fn, prepare_loss_input)
    want, _ = _three_pass(xu, data, fn, gs, gt)
    for factor in (1.0, 0.3, 1.0):
        (df,) = torch.autograd.grad(got * factor, xf, retain_graph=True)
        (du,) = torch.autograd.grad(want * factor, xu, retain_graph=True)
        _same_gradient(df, du, dtype)
    (0.7 * got).backward()
    (0.7 * want).backward()
    _same_gradient(xf.grad, xu.grad, dtype)


@pytest.mark.parametrize("dtype,vocab", [(torch.bfloat16, 4099), (torch.float32, 81930)])
def test_temperature_strides_and_refusals(dtype, vocab):
    logits, data, gs, gt = _setup(3, 7, vocab, dtype)
    fn = ClippedPGLossFn(ClippedPGLossConfig())
    params = TrainingSamplingParams(temperature=0.7)
    xf, xu = (logits.clone().requires_grad_(True) for _ in range(2))
    with deferred_temperature():
        zf = apply_temperature_scaling(xf * 1.0, params)
        got, _ = wrap_loss_fn_with_input_preparation(zf, data, gs, gt, fn, prepare_loss_input)
    want, _ = _three_pass(apply_temperature_scaling(xu * 1.0, params), data, fn, gs, gt)
    got.backward()
    want.backward()
    assert _close(got.item(), want.item(), rel=1e-4)
    _same_gradient(xf.grad, xu.grad, dtype)
    # rows inside a wider buffer: alike modulo 16 bytes when the padding is a multiple of that, the general path otherwise
    per = 16 // logits.element_size()
    for pad, route in ((2 * per, True), (1, False)):
        wide = torch.zeros(3, 7, vocab + pad, dtype=dtype, device=DEV)
        wide[..., :vocab] = logits
        xw = wide[..., :vocab].requires_grad_(True)
        assert any_row_fusable(fn, xw, data) is route
        got, _ = wrap_loss_fn_with_input_preparation(xw, data, gs, gt, fn, prepare_loss_input)
        (dw,) = torch.autograd.grad(got, xw)
        xu = logits.clone().requires_grad_(True)
        (du,) = torch.autograd.grad(_three_pass(xu, data, fn, gs, gt)[0], xu)
        _same_gradient(dw, du, dtype)
    assert not any_row_fusable(fn, logits[..., 1:], data) and not any_row_fusable(fn, logits[..., :100], data)


@pytest.mark.parametrize("dtype,vocab", [(torch.bfloat16, 1029), (torch.bfloat16, 180003), (torch.float32, 82001)])
def test_packed_rows(dtype, vocab):
    logits, data, gs, gt = _setup(3, 8, vocab, dtype)
    lens, cuts = [8, 5, 1], [12, 6, 3]
    cu = torch.tensor([0, 8, 13, 14], dtype=torch.int32, device=DEV)
    cup = torch.tensor([0, 12, 18, 21], dtype=torch.int32, device=DEV)
    data["sample_mask"][:] = 1
    data["token_mask"][:] = 1
    for i, n in enumerate(lens):
        data["token_mask"][i, n:] = 0
    gt = data["token_mask"][:, 1:].sum()
    g = torch.Generator().manual_seed(3)
    x = (torch.randn(1, sum(cuts) + 2, vocab, generator=g) * 2).to(dtype).to(DEV)
    fn = ClippedPGLossFn(ClippedPGLossConfig(token_level_loss=False, reference_policy_kl_penalty=0.001))
    xf, xu = (x.clone().requires_grad_(True) for _ in range(2))
    got, gm = SequencePackingFusionLossWrapper(fn, prepare_packed_loss_input, cu, cup)(xf, data, gs, gt)
    loss_input, d2 = prepare_packed_loss_input(xu, dict(data), fn, cu, cup)
    want, wm = fn(data=d2, global_valid_seqs=gs, global_valid_toks=gt, **loss_input)
    assert _close(got.item(), want.item(), rel=1e-4)
    for k in wm:
        assert _close(float(gm[k]), float(wm[k])), k
    for factor in (1.0, 0.3):
        (df,) = torch.autograd.grad(got * factor, xf, retain_graph=True)
        (du,) = torch.autograd.grad(want * factor, xu, retain_graph=True)
        _same_gradient(df, du, dtype)


@pytest.mark.parametrize("vocab", [4099, 164000])
def test_masked_in_positions_beyond_a_packed_sequence(vocab):
    """They have no row: their logprob is 0 and they count in the loss and the metrics, as on the general path."""
    logits, data, gs, _ = _setup(4, 9, vocab, torch.bfloat16)
    data["token_mask"][:] = 1
    data["sample_mask"][:] = 1
    gt = data["token_mask"][:, 1:].sum()
    cu = torch.tensor([0, 8, 13, 13, 14], dtype=torch.int32, device=DEV)
    cup = torch.tensor([0, 12, 18, 18, 21], dtype=torch.int32, device=DEV)
    g = torch.Generator().manual_seed(4)
    x = (torch.randn(1, 23, vocab, generator=g) * 2).to(torch.bfloat16).to(DEV)
    for cfg in (dict(), dict(token_level_loss=False, reference_policy_kl_penalty=0.001), dict(reference_policy_kl_penalty=0.0)):
        fn = ClippedPGLossFn(ClippedPGLossConfig(**cfg))
        xf, xu = (x.clone().requires_grad_(True) for _ in range(2))
        assert any_row_fusable_packed(fn, xf, data)
        got, gm = SequencePackingFusionLossWrapper(fn, prepare_packed_loss_input, cu, cup)(xf, data, gs, gt)
        loss_input, d2 = prepare_packed_loss_input(xu, dict(data), fn, cu, cup)
        want, wm = fn(data=d2, global_valid_seqs=gs, global_valid_toks=gt, **loss_input)
        assert _close(got.item(), want.item(), rel=1e-4)
        for k in wm:
            assert _close(float(gm[k]), float(wm[k])), k
        got.backward()
        want.backward()
        _same_gradient(xf.grad, xu.grad, torch.bfloat16)


@pytest.mark.parametrize("dtype,vocab", [(torch.bfloat16, 4099), (torch.bfloat16, 4096), (torch.float32, 90000)])
@pytest.mark.parametrize("b,s", [(0, 9), (3, 1), (0, 1)])
def test_empty_microbatches(dtype, vocab, b, s):
    """No sequence, and sequences of one token: a zero loss and a zero gradient."""
    logits, data, gs, gt = _setup(3, 9, vocab, dtype)
    data = {k: v[:b] if v.dim() == 1 else v[:b, :s] for k, v in data.items()}
    fn = ClippedPGLossFn(ClippedPGLossConfig())
    x = logits[:b, :s].clone().requires_grad_(True)
    got, gm = wrap_loss_fn_with_input_preparation(x, data, gs, gt, fn, prepare_loss_input)
    want, wm = _three_pass(x, data, fn, gs, gt)
    assert got.item() == want.item() == 0.0
    for k in wm:
        assert float(gm[k]) == float(wm[k]) or (float(gm[k]) != float(gm[k]) and float(wm[k]) != float(wm[k])), k
    (d,) = torch.autograd.grad(got * 0.3, x)
    assert d.shape == x.shape and not bool(d.any())


@pytest.mark.parametrize("vocab", [4099, 4096])
def test_empty_packed_microbatches(vocab):
    logits, data, gs, gt = _setup(3, 9, vocab, torch.bfloat16)
    fn = ClippedPGLossFn(ClippedPGLossConfig())
    one = {k: v if v.dim() == 1 else v[:, :1] for k, v in data.items()}
    cu = torch.tensor([0, 1, 2, 3], dtype=torch.int32, device=DEV)
    x = logits[0, :4].clone().unsqueeze(0).requires_grad_(True)
    assert any_row_fusable_packed(fn, x, one)
    got, _ = SequencePackingFusionLossWrapper(fn, prepare_packed_loss_input, cu, cu)(x, one, gs, gt)
    (d,) = torch.autograd.grad(got, x)
    assert got.item() == 0.0 and d.shape == x.shape and not bool(d.any())


def _untouched_by_backward(x, loss, factor, want):
    """The gradient is the one the forward wrote: the logits it could be written again from are gone by then."""
    x.data.zero_()
    (d,) = torch.autograd.grad(loss, x)
    _same_gradient(d, want * factor, d.dtype)


@pytest.mark.parametrize("dtype,vocab", [(torch.bfloat16, 4099), (torch.float32, 82001)])
def test_a_named_factor_is_written_by_the_forward(dtype, vocab):
    from types import SimpleNamespace

    from rl_amd.models.automodel.train import LossPostProcessor as DTensorPost
    from rl_amd.models.megatron.train import LossPostProcessor as MegatronPost

    logits, data, gs, gt = _setup(3, 7, vocab, dtype)
    fn = ClippedPGLossFn(ClippedPGLossConfig())
    xu = logits.clone().requires_grad_(True)
    (want,) = torch.autograd.grad(_three_pass(xu, data, fn, gs, gt)[0], xu)
    want = want.float()

    def fresh():
        return logits.clone().requires_grad_(True)

    x = fresh()
    loss, _ = wrap_loss_fn_with_input_preparation(x, data, gs, gt, fn, prepare_loss_input, loss_scale=0.3)
    (again,) = torch.autograd.grad(loss * 0.7, x, retain_graph=True)  # not the one that was named
    _same_gradient(again, want * 0.7, dtype)
    x = fresh()
    loss, _ = wrap_loss_fn_with_input_preparation(x, data, gs, gt, fn, prepare_loss_input, loss_scale=0.3)
    _untouched_by_backward(x, loss * 0.3, 0.3, want)

    x = fresh()
    post = DTensorPost(fn, {}, None, None, None, 1, 4)
    loss, _ = post(x, dict(data), SimpleNamespace(), gs, gt)
    _untouched_by_backward(x, loss * post.dp_size * post.cp_size, 4.0, want)

    for n in (1, 8, 41):
        x = fresh()
        cfg = {"sequence_packing": {"enabled": False}}
        loss, _ = MegatronPost(fn, cfg, num_microbatches=n)(dict(data), None, gs, gt)(x)
        _untouched_by_backward(x, loss / n, 1.0, want)


def test_a_named_factor_of_packed_rows():
    from types import SimpleNamespace

    from rl_amd.models.megatron.train import LossPostProcessor

    logits, data, gs, gt = _setup(3, 8, 1029, torch.bfloat16)
    cu = torch.tensor([0, 8, 16, 24], dtype=torch.int32, device=DEV)
    flat = logits.reshape(1, 24, 1029)
    fn = ClippedPGLossFn(ClippedPGLossConfig())
    xu = flat.clone().requires_grad_(True)
    loss_input, d2 = prepare_packed_loss_input(xu, dict(data), fn, cu, cu)
    (want,) = torch.autograd.grad(fn(data=d2, global_valid_seqs=gs, global_valid_toks=gt, **loss_input)[0], xu)
    x = flat.clone().requires_grad_(True)
    loss, _ = SequencePackingFusionLossWrapper(fn, prepare_packed_loss_input, cu, cu)(x, data, gs, gt, loss_scale=0.3)
    _untouched_by_backward(x, loss * 0.3, 0.3, want.float())
    x = flat.clone().requires_grad_(True)
    post = LossPostProcessor(fn, {"sequence_packing": {"enabled": True, "fuse_loss": True}}, num_microbatches=41)
    loss, _ = post(dict(data), SimpleNamespace(cu_seqlens_q=cu, cu_seqlens_q_padded=cu), gs, gt)(x)
    _untouched_by_backward(x, loss / 41, 1.0, want.float())


# one length for every workgroup size and number of register slots, the form for rows longer than the chip holds last
@pytest.mark.parametrize("dtype,vocab", [(torch.bfloat16, 20003), (torch.bfloat16, 30001), (torch.bfloat16, 40961), (torch.bfloat16, 50257),
                                         (torch.bfloat16, 65003), (torch.bfloat16, 81919), (torch.bfloat16, 98305), (torch.bfloat16, 131075),
                                         (torch.bfloat16, 163841), (torch.float16, 50257), (torch.float32, 32003), (torch.float32, 151936)])
def test_rows_of_any_length_against_the_oracle(dtype, vocab):
    logits, data, gs, gt = _batch(4, 7, vocab, dtype, seed=vocab + 1)
    cfg = dict(reference_policy_kl_penalty=0.05)
    xo = logits.float().clone().requires_grad_(True)
    want, _ = O.clipped_pg_loss(O.LossConfig(**cfg), OL.next_token_logprobs(data["input_ids"], xo), data, gs, gt)
    want.backward()
    x = logits.to(DEV).requires_grad_(True)
    fn = ClippedPGLossFn(ClippedPGLossConfig(**cfg))
    dev = {k: v.to(DEV) for k, v in data.items()}
    assert any_row_fusable(fn, x, dev) and why_not_fusable(fn, x, dev) is not None
    got, _ = wrap_loss_fn_with_input_preparation(x, dev, gs.to(DEV), gt.to(DEV), fn, prepare_loss_input)
    got.backward()
    assert _close(got.item(), want.item(), rel=1e-4)
    # (the oracle's gradient is fp32: an fp16 one is rounded to multiples of 2^-24 where it is subnormal, half of that off)
    wanted = xo.grad if dtype != torch.float16 else torch.where((xo.grad - x.grad.cpu().float()).abs() <= 2.0 ** -25, x.grad.cpu().float(), xo.grad)
    _same_gradient(x.grad.cpu(), wanted, dtype)


def _many_rows(b, s, vocab, dtype, seed):
    """As ``_batch``, made on the GPU: every sequence but one carries tokens, behind a prompt of its own length."""
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = (torch.randn(b, s, vocab, generator=g, device=DEV) * 2.5).to(dtype)
    ids = torch.randint(0, vocab, (b, s), generator=g, device=DEV)
    lp = torch.stack([x[i, :-1].float().log_softmax(-1).gather(-1, ids[i, 1:, None]).squeeze(-1) for i in range(b)])
    cur = torch.cat([torch.zeros(b, 1, device=DEV), lp], 1)
    noise = lambda: 0.05 * torch.randn(b, s, generator=g, device=DEV)  # noqa: E731
    prompt = torch.randint(1, s // 3, (b, 1), generator=g, device=DEV)
    data = {"input_ids": ids, "token_mask": (torch.arange(s, device=DEV) >= prompt).long(), "sample_mask": torch.ones(b, device=DEV),
            "advantages": torch.randn(b, 1, generator=g, device=DEV).expand(b, s).contiguous(), "prev_logprobs": cur + noise(),
            "generation_logprobs": cur + noise(), "reference_policy_logprobs": cur + noise()}
    data["sample_mask"][b // 2] = 0
    return x, data, data["sample_mask"].sum(), (data["token_mask"][:, 1:] * data["sample_mask"][:, None]).sum()


# more rows than workgroups are resident (1024 of 256 threads, 512 of 512, 256 of 1024), so that a workgroup goes from one row to
# others with another head and tail; the aligned lengths are the longest of their workgroup size
WALKS = [(1100, 20003), (600, 50257), (600, 81919), (300, 98305), (300, 163003), (300, 164001), (1100, 40960), (600, 81920), (300, 163840)]


@pytest.mark.parametrize("rows,vocab", WALKS)
@pytest.mark.parametrize("packed", [False, True])
def test_a_workgroup_walks_several_rows(rows, vocab, packed):
    b = 4
    logits, data, gs, gt = _many_rows(b, rows // b, vocab, torch.bfloat16, seed=vocab)
    fn = ClippedPGLossFn(ClippedPGLossConfig(reference_policy_kl_penalty=0.05))
    if packed:
        cu = torch.arange(0, rows + 1, rows // b, dtype=torch.int32, device=DEV)
        xf, xu = (logits.reshape(1, rows, vocab).clone().requires_grad_(True) for _ in range(2))
        got, _ = SequencePackingFusionLossWrapper(fn, prepare_packed_loss_input, cu, cu)(xf, data, gs, gt)
        loss_input, d2 = prepare_packed_loss_input(xu, dict(data), fn, cu, cu)
        want, _ = fn(data=d2, global_valid_seqs=gs, global_valid_toks=gt, **loss_input)
    else:
        xf, xu = (logits.clone().requires_grad_(True) for _ in range(2))
        got, _ = wrap_loss_fn_with_input_preparation(xf, data, gs, gt, fn, prepare_loss_input)
        want, _ = _three_pass(xu, data, fn, gs, gt)
    assert _close(got.item(), want.item(), rel=1e-4)
    got.backward()
    want.backward()
    _same_gradient(xf.grad, xu.grad, torch.bfloat16)
    assert bool((xf.grad.reshape(b, rows // b, vocab)[:, -1] == 0).all()) and bool((xf.grad.float().abs().sum(-1) > 0).float().mean() > 0.4)
