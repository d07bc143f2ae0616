"""Single-pass path: logits -> clipped-PG loss -> dlogits in one kernel.

``fused_logits_clipped_pg_loss`` does what ``prepare_loss_input`` + ``ClippedPGLossFn`` + the
backward of the logprob op do (``nemo_rl/algorithms/loss/wrapper.py:292-322``), but the logits are
read once and the gradient written once: the kernel keeps each row on chip between the
log-sum-exp and the gradient and evaluates the token's loss terms in between.  The gradient exists
as soon as the forward returns; ``backward`` hands it to autograd, rescaled in place on the device when
the upstream gradient is not the ``loss_scale`` it was computed with.
"""

from __future__ import annotations

from typing import Any, Optional

import torch

from ... import ops as _ops  # noqa: F401
from ..._deferred import pending_temperature
from ..._lib import NRL_TEMP_RCP
from ..._lib import host as _host
from .loss_functions import ClippedPGLossFn, _scalar, metrics_record_to_dict


def _why_not(loss_fn, logits, data, sampling_params) -> Optional[str]:
    """The reason, if any, why a single pass over the rows cannot compute this loss, wherever the rows lie."""
    from ..logits_sampling_utils import need_top_k_or_top_p_filtering

    if type(loss_fn) is not ClippedPGLossFn:
        return "not a ClippedPGLossFn"
    if getattr(loss_fn, "use_fused_linear_logprobs", False):
        return "the model already returned logprobs"
    if need_top_k_or_top_p_filtering(sampling_params):
        return "top-k/top-p filtering"
    if loss_fn.sequence_level_importance_ratios and not (loss_fn.disable_ppo_ratio or loss_fn.force_on_policy_ratio):
        return "sequence-level probability ratios"
    if loss_fn.force_on_policy_ratio and (
        loss_fn.sequence_level_importance_ratios or loss_fn.truncated_importance_sampling_type == "seq-mask-tis"
    ):
        return "sequence-level importance weights of the current policy"
    if loss_fn.positive_example_nll_weight > 0 and "rewards" in data:
        return "positive-example NLL term"
    if not isinstance(logits, torch.Tensor) or not logits.is_cuda or logits.dim() != 3:
        return "logits are not a [B, S, V] GPU tensor"
    if logits.dtype not in (torch.float32, torch.bfloat16, torch.float16) or logits.stride(2) != 1:
        return "unsupported logits dtype or layout"
    if logits.shape[1] < data["input_ids"].shape[1]:
        return "logits shorter than input_ids"
    return None


def why_not_fusable(loss_fn, logits, data, sampling_params=None) -> Optional[str]:
    """None if the fused kernel covers this call, else the reason it does not."""
    reason = _why_not(loss_fn, logits, data, sampling_params)
    if reason is not None:
        return reason
    elt, vocab = logits.element_size(), logits.shape[2]
    if (vocab * elt) % 16 or vocab * elt > 20480 * 16:
        return "vocabulary row does not fit the on-chip path"
    if logits.data_ptr() % 16 or (logits.stride(0) * elt) % 16 or (logits.stride(1) * elt) % 16:
        return "rows are not 16-byte aligned"
    return None


_ANY_ROW_BYTES = (1024, 1 << 20)  # NRL_FUSED_ANY_ROW_MIN, NRL_FUSED_ANY_ROW_MAX


def any_row_fusable(loss_fn, logits, data, sampling_params=None) -> bool:
    """Whether the single pass for rows off the 16-byte grid, or longer than the chip holds, covers this call: the gradient, a
    contiguous tensor, must sit on that grid as the logits do."""
    if _why_not(loss_fn, logits, data, sampling_params) is not None:
        return False
    elt, (_, s, v) = logits.element_size(), logits.shape
    return (_ANY_ROW_BYTES[0] <= v * elt <= _ANY_ROW_BYTES[1] and logits.data_ptr() % 16 == 0
            and (logits.stride(1) - v) * elt % 16 == 0 and (logits.stride(0) - s * v) * elt % 16 == 0)


def fused_logits_clipped_pg_loss(
    logits: torch.Tensor,
    data: Any,
    loss_fn: ClippedPGLossFn,
    global_valid_seqs,
    global_valid_toks,
    *,
    loss_scale: float = 1.0,
    in_place: bool = False,
):
    """``(loss, metrics)`` exactly as ``loss_fn(prepare_loss_input(logits, data, loss_fn))`` would return them.

    ``loss_scale`` is the gradient the caller will send into ``loss.backward()`` (1 for a plain
    ``backward()``, ``dp_size * cp_size`` when the worker scales the loss first); with it the stored
    gradient is final and ``backward`` moves no data.  ``in_place=True`` writes the gradient over the
    logits buffer instead of allocating a second ``[B, S, V]`` tensor (the logits are dead after the
    loss in the training step).  The metrics do not include values for masked positions, which are
    never evaluated."""
    reason = why_not_fusable(loss_fn, logits, data)
    if reason is not None:
        raise NotImplementedError(f"fused logits->loss path: {reason}")
    return _single_pass(logits, data, loss_fn, global_valid_seqs, global_valid_toks, loss_scale, in_place, False)


def _single_pass(logits, data, loss_fn, global_valid_seqs, global_valid_toks, loss_scale, in_place, any_row):
    dev = logits.device
    ids = data["input_ids"]
    sample_mask_in = data["sample_mask"]
    iflags, fparams = loss_fn._kernel_config(False)
    # (row (b, i) reads input_ids[b, i + 1] and column i + 1 of the loss inputs: offsets, not slices)
    loss, metrics = _host().fused_clipped_pg(
        logits, ids, 1, ids.shape[1] - 1, None, None if loss_fn.force_on_policy_ratio else data["prev_logprobs"],
        data["generation_logprobs"], data["reference_policy_logprobs"] if loss_fn.reference_policy_kl_penalty != 0 else None,
        data["advantages"], data["token_mask"], sample_mask_in, _scalar(global_valid_seqs, dev), _scalar(global_valid_toks, dev), iflags,
        fparams, float(loss_scale), pending_temperature(logits),  # a divide apply_temperature_scaling left to this kernel
        NRL_TEMP_RCP, bool(in_place), any_row,
    )
    return loss, metrics_record_to_dict(metrics, loss_fn, sample_mask_in)


def why_not_fusable_packed(loss_fn, logits, data, sampling_params=None) -> Optional[str]:
    """As ``why_not_fusable`` for a packed ``[1, T, V]`` microbatch."""
    if not isinstance(logits, torch.Tensor) or logits.dim() != 3 or logits.shape[0] != 1:
        return "logits are not a packed [1, T, V] tensor"
    return why_not_fusable(loss_fn, logits, _packed_probe(data), sampling_params)


def _packed_probe(data):
    probe = dict(data)
    probe["input_ids"] = data["input_ids"][:, :1]  # the shape test of the unpacked path does not apply
    return probe


def any_row_fusable_packed(loss_fn, logits, data, sampling_params=None) -> bool:
    return (isinstance(logits, torch.Tensor) and logits.dim() == 3 and logits.shape[0] == 1
            and any_row_fusable(loss_fn, logits, _packed_probe(data), sampling_params))


def fused_packed_logits_clipped_pg_loss(logits, data, loss_fn, cu_seqlens_q, cu_seqlens_q_padded, global_valid_seqs,
                                        global_valid_toks, *, loss_scale: float = 1.0):
    """``SequencePackingFusionLossWrapper.__call__`` (``loss/wrapper.py:169-228``) in one pass over the packed
    logits: ``prepare_packed_loss_input`` + ``ClippedPGLossFn`` + the backward of the packed logprob op."""
    reason = why_not_fusable_packed(loss_fn, logits, data)
    if reason is not None:
        raise NotImplementedError(f"fused packed logits->loss path: {reason}")
    return _single_pass_packed(logits, data, loss_fn, cu_seqlens_q, cu_seqlens_q_padded, global_valid_seqs, global_valid_toks, loss_scale, False)


def _single_pass_packed(logits, data, loss_fn, cu_seqlens_q, cu_seqlens_q_padded, global_valid_seqs, global_valid_toks, loss_scale, any_row):
    from ...distributed.model_utils import _checked_cu_seqlens
    from .utils import _packed_targets

    dev = logits.device
    input_ids = data["input_ids"]
    x = logits.squeeze(0)
    targets = _packed_targets(input_ids, cu_seqlens_q, cu_seqlens_q_padded, x.shape[0], dev).reshape(-1)
    cu = _checked_cu_seqlens(cu_seqlens_q_padded, x.shape[0], targets.shape[0], dev)
    sample_mask_in = data["sample_mask"]
    iflags, fparams = loss_fn._kernel_config(False)
    loss, metrics = _host().fused_clipped_pg(
        x, targets, 0, input_ids.shape[1] - 1, cu, None if loss_fn.force_on_policy_ratio else data["prev_logprobs"],
        data["generation_logprobs"], data["reference_policy_logprobs"] if loss_fn.reference_policy_kl_penalty != 0 else None,
        data["advantages"], data["token_mask"], sample_mask_in, _scalar(global_valid_seqs, dev), _scalar(global_valid_toks, dev), iflags,
        fparams, float(loss_scale), pending_temperature(logits), NRL_TEMP_RCP, False, any_row,
    )
    return loss, metrics_record_to_dict(metrics, loss_fn, sample_mask_in)
