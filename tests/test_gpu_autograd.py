"""The C++ host path: what autograd sees of its nodes, and what its operators refuse."""

import pytest
import torch

from rl_amd.algorithms.loss import ClippedPGLossConfig, ClippedPGLossFn, prepare_loss_input, wrap_loss_fn_with_input_preparation
from test_gpu_fused import _batch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _setup(vocab):
    logits, data, gs, gt = _batch(3, 9, vocab, torch.bfloat16, seed=vocab)
    return logits.to(DEV), {k: v.to(DEV) for k, v in data.items()}, gs.to(DEV), gt.to(DEV)


def _loss(route, logits, data, gs, gt):
    fn = ClippedPGLossFn(ClippedPGLossConfig())
    if route == "general":
        loss_input, data = prepare_loss_input(logits, dict(data), fn)
        return fn(data=data, global_valid_seqs=gs, global_valid_toks=gt, **loss_input)[0]
    return wrap_loss_fn_with_input_preparation(logits, data, gs, gt, fn, prepare_loss_input)[0]


ROUTES = [("general", 4096), ("single pass", 4096), ("single pass", 4099)]


@pytest.mark.parametrize("route,vocab", ROUTES)
@pytest.mark.parametrize("key", ["advantages", "prev_logprobs", "generation_logprobs", "reference_policy_logprobs"])
def test_loss_inputs_are_inputs_of_the_node(route, vocab, key):
    """Forward-mode differentiation through any of them is refused; one that requires a gradient is part of the graph and
    receives none."""
    import torch.autograd.forward_ad as fad

    logits, data, gs, gt = _setup(vocab)
    x = logits.clone().requires_grad_(True)
    with fad.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
        _loss(route, x, {**data, key: fad.make_dual(data[key], torch.ones_like(data[key]))}, gs, gt)
    leaf = data[key].clone().requires_grad_(True)
    want = _loss(route, x, data, gs, gt)
    (dx,) = torch.autograd.grad(want, x)
    got = _loss(route, x, {**data, key: leaf}, gs, gt)
    dx2, dleaf = torch.autograd.grad(got, (x, leaf), allow_unused=True)
    assert torch.equal(dx, dx2) and dleaf is None
    if route == "general":  # (the single pass is taken for logits that require a gradient)
        got = _loss(route, logits, {**data, key: leaf}, gs, gt)
        assert got.requires_grad and torch.autograd.grad(got, leaf, allow_unused=True) == (None,)


@pytest.mark.parametrize("op", ["logprobs", "filtered", "gather", "single pass"])
def test_a_second_derivative_is_not_taken_for_zero(op):
    """Under create_graph the gradient depends on the upstream one, and differentiating it warns."""
    from rl_amd.algorithms.logits_sampling_utils import TrainingSamplingParams
    from rl_amd.distributed import model_utils as MU

    logits, data, gs, gt = _setup(4099)
    x = logits.float().requires_grad_(True)
    if op == "gather":
        ids = data["input_ids"].unsqueeze(-1).contiguous()
        y = MU.get_distillation_topk_logprobs_from_logits(x, torch.zeros_like(ids, dtype=torch.float32), ids, True, True)[0].square().sum()
    elif op == "single pass":
        y = _loss(op, x, data, gs, gt).square()
    else:
        params = TrainingSamplingParams(top_k=4000, top_p=1.0, temperature=1.0) if op == "filtered" else None
        y = MU.from_parallel_logits_to_logprobs(x, data["input_ids"], 0, 4099, None, sampling_params=params).clamp(min=-50).square().sum()
    (d,) = torch.autograd.grad(y, x, create_graph=True)
    assert d.requires_grad
    with pytest.warns(UserWarning, match="autograd|no gradient of its own"):
        torch.autograd.grad(d.sum(), x, allow_unused=True)
    (d,) = torch.autograd.grad(_loss("general", x, data, gs, gt), x)
    assert not d.requires_grad


def test_logits_of_another_rank_are_a_value_error():
    from rl_amd.algorithms.logits_sampling_utils import TrainingSamplingParams
    from rl_amd.distributed import model_utils as MU

    logits, data, _, _ = _setup(4096)
    flat, ids = logits[0], data["input_ids"]
    params = TrainingSamplingParams(top_k=20, top_p=0.9, temperature=1.0)
    ops = torch.ops.rl_amd
    for call in (
        lambda: MU.from_parallel_logits_to_logprobs(flat, ids, 0, 4096, None, sampling_params=params),
        lambda: MU.from_parallel_logits_to_logprobs(flat, ids, 0, 4096, None),
        lambda: ops.topk_topp_logprob_fwd(flat, ids, 8, 20, 0.9, 1.0, 1, False),
        lambda: ops.gather_entropy_fwd(flat, ids.unsqueeze(-1), 8, True),
    ):
        with pytest.raises(ValueError, match="logits"):
            call()


@pytest.mark.parametrize("name", ["lp", "prev", "gen", "ref", "adv", "token_mask", "sample_mask", "global_valid"])
def test_loss_operators_take_fp32_on_the_gpu_only(name):
    ops = torch.ops.rl_amd
    logits, data, _, _ = _setup(4096)
    iflags, fparams = ClippedPGLossFn(ClippedPGLossConfig())._kernel_config(False)
    rows = lambda k: data[k][:, 1:].float().contiguous()  # noqa: E731
    good = dict(lp=-torch.rand(3, 8, device=DEV), prev=rows("prev_logprobs"), gen=rows("generation_logprobs"), ref=rows("reference_policy_logprobs"),
                adv=rows("advantages"), token_mask=rows("token_mask"), sample_mask=data["sample_mask"].float(),
                global_valid=torch.tensor([2.0, 9.0], device=DEV))

    def general(a):
        return ops.grpo_loss(a["lp"], None, a["prev"], a["gen"], a["ref"], a["adv"], a["token_mask"], a["sample_mask"], None,
                             a["global_valid"], iflags, fparams)

    def single_pass(a):
        return ops.fused_logits_grpo_loss(logits, data["input_ids"][:, 1:], 8, a["prev"], a["gen"], a["ref"], a["adv"], a["token_mask"],
                                          a["sample_mask"], a["global_valid"], iflags, fparams, 1.0, 1.0, 1)

    for call in (general, single_pass)[: 1 if name == "lp" else 2]:
        call(good)
        for bad in (good[name].double(), good[name].long(), good[name].cpu()):
            with pytest.raises((ValueError, RuntimeError), match="fp32|GPU only"):
                call({**good, name: bad})
