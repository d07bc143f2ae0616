"""The work a policy worker has this package do, as cases with inputs, one pass each and its necessary work.

A case is a dict of plain values.  Its ``kind`` says which call sequence it stands for:

  policy    one training microbatch through the DTensor worker's ``forward_with_post_processing_fn`` and its
            ``LossPostProcessor``: model output -> clipped policy-gradient loss -> gradient of the logits
  packed    one packed training microbatch through the Megatron worker's ``SequencePackingFusionLossWrapper``
  filtered  a training microbatch whose rollout sampled with temperature and top-k / top-p, through the same
            ``forward_with_post_processing_fn``
  logprobs  the forward-only pass for prev / reference logprobs, ``LogprobsPostProcessor``, right-padded sequences
  lm_head   hidden states -> logprobs -> loss -> (dH, dW) through the fused lm_head of the Megatron worker
  distill   top-k distillation: ``prepare_loss_input`` -> ``DistillationLossFn`` -> gradient of the student's logits

Logits are N(0, std) with a standard deviation of their own for every row (a language model's rows run from nearly
flat to nearly certain), target ids are drawn from the distribution the logits give, and the logprobs of earlier passes
are the current ones plus N(0, 0.05), as after a few optimizer steps.
"""

from __future__ import annotations

import math
from functools import partial
from types import SimpleNamespace

import torch

from rl_amd.algorithms.advantage_estimator import AdvEstimatorConfig, GRPOAdvantageEstimator
from rl_amd.algorithms.logits_sampling_utils import TrainingSamplingParams
from rl_amd.algorithms.loss import (
    ClippedPGLossConfig,
    ClippedPGLossFn,
    DistillationLossConfig,
    DistillationLossFn,
    SequencePackingFusionLossWrapper,
    prepare_loss_input,
    prepare_packed_loss_input,
)
from rl_amd.distributed.model_utils import from_parallel_hidden_states_to_logprobs
from rl_amd.models.automodel import train as worker

_DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
_BYTES = {"bf16": 2, "fp16": 2, "fp32": 4}

# the model side of the worker's forward function: here the "model" hands out resident logits
worker.MODEL_HELPERS = {"model_forward": lambda model, inputs, **kw: model(inputs), "extract_logits": lambda model, out: out}

# fraction of the positions that carry a loss (prompts are a sixteenth to a quarter of a sequence) and of the rows a
# right-padded batch really holds (lengths are uniform between half and the whole width)
_LIVE = 27 / 32
_PACKED_LIVE = 0.6   # packed sequences are shorter than the widest one, their prompts are not
_FILLED = 0.75


def listed():
    return [
        # a debugging-size GRPO step: group advantages, fp32 logits of a 32 000-word vocabulary; launch-bound
        dict(name="policy_small", kind="policy", batch=8, seq=64, vocab=32000, dtype="fp32", loss="grpo", advantages=True),
        # the ordinary training microbatch of a 150 k vocabulary in bf16, PPO clip and k3 KL
        dict(name="policy_mid", kind="policy", batch=4, seq=1024, vocab=151936, dtype="bf16", loss="grpo", advantages=False),
        # the microbatch that 288 GB allow: long sequences, 10 GB of logits
        dict(name="policy_large", kind="policy", batch=8, seq=4096, vocab=151936, dtype="bf16", loss="grpo", advantages=False),
        # a model wrapper that returns fp32 logits, DAPO (clip-higher, no KL)
        dict(name="policy_fp32", kind="policy", batch=2, seq=1024, vocab=151936, dtype="fp32", loss="dapo", advantages=False),
        # an unpadded odd vocabulary and a ragged sequence length: no row but the first starts on 16 bytes
        dict(name="policy_odd", kind="policy", batch=3, seq=701, vocab=50257, dtype="bf16", loss="grpo", advantages=False),
        # sequence-packed microbatch of the Megatron worker, ragged sequences padded to multiples of 16
        dict(name="packed", kind="packed", tokens=16384, seqs=7, vocab=131072, dtype="bf16"),
        # rollouts sampled with temperature 0.7, top-k 50 and top-p 0.95, DAPO
        dict(name="filtered", kind="filtered", batch=2, seq=2048, vocab=151936, dtype="bf16", top_k=50, top_p=0.95, temperature=0.7),
        # nucleus sampling alone: kept sets from a few tokens to tens of thousands
        dict(name="nucleus", kind="filtered", batch=1, seq=1500, vocab=151936, dtype="bf16", top_k=0, top_p=0.95, temperature=1.0),
        # prev / reference logprobs of a right-padded batch
        dict(name="logprobs", kind="logprobs", batch=8, seq=2048, vocab=151936, dtype="bf16"),
        # fused lm_head on a short microbatch (one 512-token sample) ...
        dict(name="lm_head_short", kind="lm_head", batch=1, seq=512, hidden=4096, vocab=151936),
        # ... and on a full one
        dict(name="lm_head_full", kind="lm_head", batch=2, seq=4096, hidden=4096, vocab=151936),
        # on-policy distillation from a teacher's top 64, mixed KL with the correction for the mass outside them
        dict(name="distill", kind="distill", batch=2, seq=1024, vocab=151936, dtype="bf16", topk=64, kl="mixed"),
    ]


_MOST_LOGITS = 8 * 4096 * 151936 * 2       # bytes of the largest listed logits
_MOST_PRODUCT = 2 * 4096 * 4096 * 151936   # tokens x hidden x vocab of the largest listed product


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_vocab(rng):
    v = _log_uniform(rng, 8192, 262144)
    return v if rng.random() < 0.3 else max(64, v // 64 * 64)   # most checkpoints pad it, some do not


def draw(rng):
    kind = rng.choice(["policy", "policy", "packed", "filtered", "logprobs", "lm_head", "distill"])
    vocab = _draw_vocab(rng)
    if kind == "lm_head":
        hidden = 64 * _log_uniform(rng, 16, 80)
        tokens = _log_uniform(rng, 128, min(16384, _MOST_PRODUCT // (hidden * vocab)))
        batch = rng.choice([1, 1, 2, 4])
        return dict(kind=kind, batch=batch, seq=max(32, tokens // batch), hidden=hidden, vocab=vocab)
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp32", "fp32", "fp16"])
    if kind in ("filtered", "distill"):
        most = _MOST_LOGITS // 8            # these make several passes over the logits
    else:
        most = _MOST_LOGITS
    rows = _log_uniform(rng, 128, min(32768, most // (vocab * _BYTES[dtype])))
    if kind == "packed":
        return dict(kind=kind, tokens=rows, seqs=rng.randint(1, max(1, min(12, rows // 64))), vocab=vocab, dtype=dtype)
    batch = min(rng.choice([1, 2, 3, 4, 8]), max(1, rows // 32))
    shape = dict(kind=kind, batch=batch, seq=rows // batch, vocab=vocab, dtype=dtype)
    if kind == "policy":
        shape.update(loss=rng.choice(["grpo", "grpo", "dapo", "gspo"]), advantages=rng.random() < 0.25)
    elif kind == "filtered":
        top_k = rng.choice([0, _log_uniform(rng, 4, 400), _log_uniform(rng, 20, 100)])
        shape.update(top_k=top_k, top_p=round(rng.uniform(0.8, 0.99), 3), temperature=rng.choice([1.0, round(rng.uniform(0.6, 1.2), 2)]))
    elif kind == "distill":
        shape.update(topk=_log_uniform(rng, 8, 256), kl=rng.choice(["forward", "reverse", "mixed"]))
    return shape


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _rows(x):
    """Views of at most about 1 GB of fp32 each over the rows of ``x`` ([rows, V])."""
    return x.split(max(1, (1 << 28) // x.shape[1]))


def _make_logits(g, rows, vocab, dtype, lo=2.0, hi=6.0):
    x = torch.empty((rows, vocab), dtype=dtype, device="cuda").normal_(0.0, 1.0, generator=g)
    return x.mul_(torch.empty((rows, 1), device="cuda").uniform_(lo, hi, generator=g).to(dtype))


def _sample_and_score(g, x, temperature=1.0, top_k=0, top_p=1.0):
    """Ids drawn from softmax(x / T) under the filter, and their log-probabilities (the nucleus counted as holding
    exactly ``top_p`` of the mass): what a rollout with these logits would have produced."""
    ids, logp = [], []
    for part in _rows(x):
        z = part.float() / temperature
        if top_k:
            top, at = z.topk(min(top_k, z.shape[1]), dim=-1)
            p = top.softmax(-1)
            keep = p.cumsum(-1) - p < top_p
            z = top.masked_fill(~keep, float("-inf"))
            shift = 0.0
        else:
            at, shift = None, math.log(top_p)
        norm = z.logsumexp(-1, keepdim=True)
        noise = torch.empty_like(z).exponential_(generator=g)
        pick = (z - noise.log_()).argmax(-1, keepdim=True)
        logp.append((z.gather(-1, pick) - norm - shift).squeeze(-1))
        ids.append((pick if at is None else at.gather(-1, pick)).squeeze(-1))
    return torch.cat(ids), torch.cat(logp)


def _shifted(scores, batch, seq):
    """Per-row scores -> [B, S] logprobs with the zero first column the workers carry."""
    s = scores.view(batch, seq)
    return torch.cat([torch.zeros_like(s[:, :1]), s[:, :-1]], dim=1)


def _batch_of(g, ids_next, logp_next, batch, seq, vocab):
    """The loss inputs of ``batch`` sequences whose row ``t`` predicts ``ids_next[b, t]``."""
    first = torch.randint(0, vocab, (batch, 1), generator=g, device="cuda")
    ids = torch.cat([first, ids_next.view(batch, seq)[:, :-1]], dim=1)
    cur = _shifted(logp_next, batch, seq)
    prompt = torch.randint(max(1, seq // 16), max(2, seq // 4 + 1), (batch, 1), generator=g, device="cuda")
    mask = (torch.arange(seq, device="cuda").unsqueeze(0) >= prompt).to(torch.int64)

    def moved():
        return cur + 0.05 * torch.randn((batch, seq), generator=g, device="cuda")

    return {"input_ids": ids, "token_mask": mask, "sample_mask": torch.ones(batch, device="cuda"),
            "advantages": torch.randn((batch, 1), generator=g, device="cuda").expand(batch, seq).contiguous(),
            "prev_logprobs": moved(), "generation_logprobs": moved(), "reference_policy_logprobs": moved()}


def _valid(data):
    toks = (data["token_mask"][:, 1:] * data["sample_mask"].unsqueeze(-1)).sum().float()
    return data["sample_mask"].sum(), toks


def _loss_fn(name, **kw):
    if name == "dapo":
        return ClippedPGLossFn(ClippedPGLossConfig(ratio_clip_min=0.2, ratio_clip_max=0.28, reference_policy_kl_penalty=0.0), **kw)
    if name == "gspo":
        return ClippedPGLossFn(ClippedPGLossConfig(token_level_loss=False, sequence_level_importance_ratios=True,
                                                   ratio_clip_min=3e-4, ratio_clip_max=4e-4), **kw)
    if name == "packed":
        return ClippedPGLossFn(ClippedPGLossConfig(token_level_loss=False, reference_policy_kl_penalty=0.001), **kw)
    return ClippedPGLossFn(ClippedPGLossConfig(), **kw)


def prepare(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    st = SimpleNamespace(kind=kind)
    if kind == "lm_head":
        b, s, h, v = case["batch"], case["seq"], case["hidden"], case["vocab"]
        st.hidden = torch.randn((s, b, h), generator=g, device="cuda").to(torch.bfloat16).requires_grad_(True)
        st.weight = (torch.randn((v, h), generator=g, device="cuda") * 0.02).to(torch.bfloat16).requires_grad_(True)
        ids = torch.randint(0, v, (b, s), generator=g, device="cuda")
        flat = st.hidden.detach().transpose(0, 1).reshape(b * s, h)
        w = st.weight.detach()
        scores = []
        for rows, tgt in zip(flat.split(1024), ids.reshape(-1).split(1024)):
            z = (rows @ w.t()).float()
            scores.append(z.gather(-1, tgt.unsqueeze(-1)).squeeze(-1) - z.logsumexp(-1))
        st.data = _batch_of(g, ids.reshape(-1), torch.cat(scores), b, s, v)
        st.seqs, st.toks = _valid(st.data)
        st.loss_fn = _loss_fn("grpo", use_fused_linear_logprobs=True)
        return st
    dtype = _DTYPES[case["dtype"]]
    v = case["vocab"]
    if kind == "packed":
        total, n = case["tokens"], case["seqs"]
        width = total // n
        cuts = [16 * max(1, int(width * u) // 16) for u in torch.empty(n, device="cuda").uniform_(0.5, 1.0, generator=g).tolist()]
        cuts[-1] = total - sum(cuts[:-1])
        pad = torch.randint(0, 16, (n,), generator=g, device="cuda").tolist()
        lens = [max(1, c - p) for c, p in zip(cuts, pad)]
        x = _make_logits(g, total, v, dtype)
        ids, logp = _sample_and_score(g, x)
        st.logits = x.unsqueeze(0).requires_grad_(True)
        seq = max(cuts)
        next_ids = torch.zeros((n, seq), dtype=torch.int64, device="cuda")
        next_lp = torch.zeros((n, seq), device="cuda")
        start = 0
        for i, (c, m) in enumerate(zip(cuts, lens)):
            next_ids[i, :m], next_lp[i, :m] = ids[start:start + m], logp[start:start + m]
            start += c
        st.data = _batch_of(g, next_ids, next_lp, n, seq, v)
        inside = torch.arange(seq, device="cuda").unsqueeze(0) < torch.tensor(lens, device="cuda").unsqueeze(-1)
        st.data["token_mask"] = st.data["token_mask"] * inside
        st.data["input_ids"] = st.data["input_ids"] * inside
        st.seqs, st.toks = _valid(st.data)
        cu = torch.tensor([0] + lens, device="cuda").cumsum(0).to(torch.int32)
        cup = torch.tensor([0] + cuts, device="cuda").cumsum(0).to(torch.int32)
        st.wrapped = SequencePackingFusionLossWrapper(
            _loss_fn("packed"), partial(prepare_packed_loss_input, sampling_params=None, chunk_size=None), cu, cup, 0, None, None)
        return st
    b, s = case["batch"], case["seq"]
    x = _make_logits(g, b * s, v, dtype)
    st.logits = x.view(b, s, v)
    if kind == "logprobs":
        ids, _ = _sample_and_score(g, x)
        st.ids = torch.cat([torch.zeros_like(ids[:b]).view(b, 1), ids.view(b, s)[:, :-1]], dim=1)
        st.lengths = torch.randint(s // 2, s + 1, (b,), generator=g, device="cuda")
        st.post = worker.LogprobsPostProcessor({"logprob_chunk_size": None}, None, None, None, 1)
        st.microbatch = SimpleNamespace(data_dict={"input_lengths": st.lengths}, processed_inputs=SimpleNamespace(seq_len=s, input_ids=st.ids),
                                        original_batch_size=b, original_seq_len=s)
        return st
    if kind == "distill":
        k = case["topk"]
        top, at = [], []
        for part in _rows(x):   # a teacher that agrees with the student up to noise
            z = part.float() + torch.randn(part.shape, generator=g, device="cuda")
            t, i = z.topk(k, dim=-1)
            top.append(t)
            at.append(i)
        ids = torch.randint(0, v, (b * s,), generator=g, device="cuda")
        st.data = _batch_of(g, ids, torch.zeros(b * s, device="cuda"), b, s, v)
        st.data["teacher_topk_logits"] = torch.cat(top).view(b, s, k)
        st.data["teacher_topk_indices"] = torch.cat(at).view(b, s, k)
        st.loss_fn = DistillationLossFn(DistillationLossConfig(kl_type=case["kl"], mixed_kl_weight=0.5, zero_outside_topk=True))
        st.logits.requires_grad_(True)
        st.seqs, st.toks = _valid(st.data)
        return st
    params = None
    if kind == "filtered":
        params = TrainingSamplingParams(top_k=case["top_k"] or None, top_p=case["top_p"], temperature=case["temperature"])
        ids, logp = _sample_and_score(g, x, case["temperature"], case["top_k"], case["top_p"])
        fn = _loss_fn("dapo")
    else:
        ids, logp = _sample_and_score(g, x)
        fn = _loss_fn(case["loss"])
    st.params = params
    st.data = _batch_of(g, ids, logp, b, s, v)
    st.estimator = None
    if kind == "policy" and case["advantages"]:
        # groups of four generations of one prompt (the last group may be shorter)
        prompts = torch.randint(0, v, ((b + 3) // 4, 16), generator=g, device="cuda")
        st.prompts = prompts.repeat_interleave(4, dim=0)[:b].contiguous()
        st.rewards = torch.rand(b, generator=g, device="cuda")
        st.estimator = GRPOAdvantageEstimator(AdvEstimatorConfig(), None)
    st.seqs, st.toks = _valid(st.data)
    st.post = worker.LossPostProcessor(fn, {}, None, None, None, 1, 1, False, params)
    st.shape = (b, s)
    st.logits.requires_grad_(True)
    return st


def run(st):
    if st.kind == "lm_head":
        vocab = st.weight.shape[0]
        lp = from_parallel_hidden_states_to_logprobs(st.hidden, st.weight, False, st.data["input_ids"], 0, vocab, None)
        loss, metrics = st.loss_fn(next_token_logprobs=lp, data=st.data, global_valid_seqs=st.seqs, global_valid_toks=st.toks)
        dh, dw = torch.autograd.grad(loss, (st.hidden, st.weight))
        return {"logprobs": lp.detach(), "loss": loss.detach(), "metrics": metrics, "dhidden": dh, "dweight": dw}
    if st.kind == "packed":
        loss, metrics = st.wrapped(st.logits, dict(st.data), st.seqs, st.toks)
        (d,) = torch.autograd.grad(loss, st.logits)
        return {"loss": loss.detach(), "metrics": metrics, "dlogits": d}
    if st.kind == "logprobs":
        out, _, _ = worker.forward_with_post_processing_fn(lambda inputs: st.logits, st.post, st.microbatch)
        return out
    if st.kind == "distill":
        kwargs, data = prepare_loss_input(st.logits, dict(st.data), st.loss_fn)
        loss, metrics = st.loss_fn(data=data, global_valid_seqs=st.seqs, global_valid_toks=st.toks, **kwargs)
        (d,) = torch.autograd.grad(loss, st.logits)
        return {"loss": loss.detach(), "metrics": metrics, "dlogits": d}
    data = dict(st.data)
    if st.estimator is not None:
        data["advantages"] = st.estimator.compute_advantage(st.prompts, st.rewards, data["token_mask"])
    mb = SimpleNamespace(data_dict=data, processed_inputs=None, original_batch_size=st.shape[0], original_seq_len=st.shape[1])
    loss, metrics, _ = worker.forward_with_post_processing_fn(lambda inputs: st.logits, st.post, mb, global_valid_seqs=st.seqs,
                                                              global_valid_toks=st.toks, sampling_params=st.params)
    (d,) = torch.autograd.grad(loss, st.logits)
    return {"loss": loss.detach(), "metrics": metrics, "dlogits": d}


def work(case):
    kind = case["kind"]
    if kind == "lm_head":
        n, h, v = case["batch"] * case["seq"], case["hidden"], case["vocab"]
        # the logits of every token; dH and dW of the tokens that carry a gradient
        return {"bytes": 2 * (2 * v * h + 2 * n * h), "flops": 2 * n * h * v * (1 + 2 * _LIVE)}
    elt = _BYTES[case["dtype"]]
    rows = case["tokens"] if kind == "packed" else case["batch"] * case["seq"]
    one = rows * case["vocab"] * elt
    flops = 4 * rows * case["vocab"]   # an exponential and a sum each for the normaliser and for the gradient
    if kind == "logprobs":
        return {"bytes": _FILLED * one, "flops": flops / 2}
    if kind == "packed":
        return {"bytes": _PACKED_LIVE * one + one, "flops": flops}
    if kind == "distill":
        return {"bytes": 2 * one + rows * case["topk"] * 12, "flops": 2 * flops}
    return {"bytes": _LIVE * one + one, "flops": flops}


def tolerance(case):
    """About four times what the outputs differ by from the same formulas in 64 bits (2-norm, and largest difference)."""
    kind, dtype = case["kind"], case.get("dtype", "bf16")
    if dtype == "fp32":
        if kind == "distill":    # 4.7e-6 and 1.3e-3: p (log p - H) cancels
            return {"rel": 2e-5, "max": 5e-3}
        if kind == "filtered":   # 4e-6 (a difference of logprobs) and 4.3e-3 (the mass at the nucleus boundary)
            return {"rel": 1.6e-5, "max": 2e-2}
        return {"rel": 5e-6, "max": 4e-4}            # 1.2e-6 and 8e-5
    if kind == "lm_head":        # 2.6e-3 and 1e-2: logits and their gradient are bf16 between the products
        return {"rel": 1e-2, "max": 4e-2}
    if kind == "distill":        # 2.6e-3 and 6e-2
        return {"rel": 1e-2, "max": 0.25}
    if dtype == "fp16":          # single elements of a large batch's gradient are subnormal numbers
        return {"rel": 7e-3, "max": 0.99}
    return {"rel": 7e-3, "max": 1.6e-2}              # 1.7e-3 and 3.9e-3: one rounding to bf16
