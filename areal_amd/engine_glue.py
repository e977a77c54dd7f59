"""The engine-side call contract of the path, as a small harness.

Mirrors what FSDPEngine does around the functional ops for one packed
micro-batch (areal/engine/fsdp_engine.py:1908-1964, 1977-2046) and the part of
``grpo_loss_fn`` that feeds ``ppo_actor_loss_fn`` (areal/trainer/ppo/actor.py:408-480):
labels are the packed ``input_ids`` rolled by one over the WHOLE packed tensor,
the batch padding is trimmed after the log-prob op, entropy is detached, and the
loss is scaled by ``local_weight / total_loss_weight * loss_multiplier``.
"""
from __future__ import annotations

import ctypes
from typing import Any

import torch

from .advantages import advantage_rows, gae_advantages, kl_regularized_rewards, reward_scores, score_step
from .functional import (
    COUNT_ON_DEVICE_BYTES,
    _HostCounts,
    _PerValidToken,
    _lm_head_impl,
    _logprobs_impl,
    _ppo_actor_loss,
    fused_lm_head_ppo_loss,
    fused_logprobs_ppo_loss,
    gather_logprobs,
    gather_logprobs_entropy_stats,
    lm_head_chunk_tokens,
    lm_head_logprobs_entropy,
    lm_head_logprobs_entropy_stats,
    ppo_actor_loss_fn,
)


def rolled_labels(model_inputs: dict[str, Any]) -> torch.Tensor:
    """``rolled_input_ids`` if present, else ``roll(input_ids, -1)``; a leading batch dim of 1 is dropped
    (fsdp_engine.py:1915-1921).  The roll is over the packed tensor, not per sequence: the last token of a
    sequence is labelled with the first token of the next one and is expected to be masked out."""
    labels = model_inputs.get("rolled_input_ids")
    if labels is None:
        labels = torch.roll(model_inputs["input_ids"], shifts=-1, dims=-1)
    if labels.ndim == 2 and labels.shape[0] == 1:
        labels = labels.squeeze(0)
    return labels


def _weight_is_zero(local_weight):
    """(a function that tells whether the weight of the micro-batch is zero, whether it has to wait for the device, a
    function that gives the weight as the host read it, if it had to).  A device tensor starts on its way to the host now,
    behind what is queued already."""
    if isinstance(local_weight, torch.Tensor) and local_weight.is_cuda:
        pending, read = _HostCounts(local_weight.detach().reshape(())), []

        def value():
            if not read:
                read.append(pending.tolist())
            return read[0]

        return lambda: value() == 0, True, value
    zero = bool(local_weight == 0)
    return lambda: zero, False, None


def _times_weight(loss, local_weight, host_weight, total_loss_weight, multiplier):
    """``loss * (local_weight / total_loss_weight * multiplier)``.  A count that the host has read already is scaled there,
    in the float32 steps that torch takes on the device (a division by a number is a product with its reciprocal): the same
    bits, one launch behind the loss instead of three.  Only for a loss on the device of the weight: a Python number or a
    loss on the host takes type and device of the result from the weight tensor, or is refused with it."""
    if (host_weight is not None and local_weight.dim() == 0 and local_weight.dtype in (torch.int32, torch.int64)
            and isinstance(loss, torch.Tensor) and loss.device == local_weight.device
            and loss.dtype in (torch.float32, torch.float64) and type(total_loss_weight) in (int, float)
            and type(multiplier) in (int, float) and torch.get_default_dtype() is torch.float32
            and 1e-30 < abs(total_loss_weight) < 1e30 and abs(multiplier) < 1e30):
        f32 = lambda x: ctypes.c_float(x).value
        return loss * f32(f32(f32(host_weight()) * f32(1.0 / f32(total_loss_weight))) * f32(multiplier))
    return loss * (local_weight / total_loss_weight * multiplier)


def _no_tokens(scale: _PerValidToken, loss_mask: torch.Tensor):
    """The same for a step that counts the mask itself."""
    def is_zero():
        if scale.valid_tokens is None:
            scale.valid_tokens = int(loss_mask.count_nonzero())
        return scale.valid_tokens == 0

    return is_zero, loss_mask.numel() > 0


# A forward of at most this much work is queued before the host knows the weight of the micro-batch, so that the device
# has work while the host waits; what it computed is dropped when the weight is zero.  About 1 ms of forward at 6.4 TB/s
# and 1.2 PFLOP/s: asking first costs 10 to 50 us of a pass (us, forward and backward, first / ahead: 256 x 151 936 bf16
# logits PPO 158 / 131, 4 096 any loss 680 / 650, PPO 486 / 437, supervised 511 / 462; from hidden states of 1 024 entries
# 1 900 tokens any loss 1 700 / 1 660, PPO 1 550 / 1 498), 1 to 2 % of the passes past this line (16 384 x 151 936 PPO
# 1 672 / 1 625, 2 048 x 2 048 2 705 / 2 660, 4 096 x 4 096 9 520 / 9 480), and a micro-batch without a token never pays
# more than this for a result that nobody reads.
RUN_AHEAD_BYTES = 6_400_000_000
RUN_AHEAD_FLOPS = 1_200_000_000_000


def _unless_weightless(forward, weight, run_ahead: bool):
    """``forward()``, or None for a micro-batch of weight zero, whatever else it holds (an incomplete one may make
    ``forward`` raise).  ``weight``: what ``_weight_is_zero`` returned."""
    is_zero, waits = weight[:2]
    if not (run_ahead and waits) and is_zero():
        return None
    try:
        out = forward()
    except Exception:
        if is_zero():
            return None
        raise
    return None if is_zero() else out


def _float32_total(total_loss_weight) -> bool:
    """Whether ``local_weight / total_loss_weight * multiplier`` is a float32 expression, which the kernels can form
    themselves (a float64 total makes torch form it in float64)."""
    return not (isinstance(total_loss_weight, torch.Tensor) and total_loss_weight.dtype is torch.float64)


def compute_logprobs(logits: torch.Tensor, model_inputs: dict[str, Any], temperature: float = 1.0) -> torch.Tensor:
    """Forward-only log-probs of a micro-batch (fsdp_engine.py:1938-1964)."""
    return gather_logprobs(logits, rolled_labels(model_inputs), temperature=temperature)


def compute_logprobs_and_loss(
    logits: torch.Tensor,
    model_inputs: dict[str, Any],
    mb_input: dict[str, Any],
    pad_length: int,
    total_loss_weight: torch.Tensor | float,
    eps_clip: float,
    eps_clip_higher: float | None = None,
    c_clip: float | None = None,
    rejection_sampling: Any | None = None,
    importance_sampling_level: str = "token",
    temperature: float = 1.0,
    loss_multiplier: float = 1.0,
    fused: bool = True,
    inplace_backward: bool = False,
    use_sapo_loss: bool = False,
    sapo_tau_pos: float = 1.0,
    sapo_tau_neg: float = 1.05,
) -> tuple[torch.Tensor, dict]:
    """Scaled PPO loss of one micro-batch and its stat dict (fsdp_engine.py:1977-2046 with
    ``loss_fn = grpo_loss_fn`` and ``loss_weight_fn = loss_mask.count_nonzero``, actor.py:345-364).

    ``logits`` is ``[T_pad, V]``; ``mb_input`` holds the un-padded ``[T]`` tensors ``loss_mask``, ``logprobs``
    (behaviour policy), ``prox_logp``, ``advantages`` and ``cu_seqlens``.  An all-masked micro-batch returns
    ``logits.mean() * 0`` like the reference (fsdp_engine.py:1988-1989).  ``inplace_backward``: the gradient is
    written over the logits, see ``fused_logprobs_ppo_loss``.  ``use_sapo_loss`` (token level, fused): the SAPO gate in
    place of the clip, on the behaviour log-probs (actor.py:448-462: SAPO takes ``old_logp``, no proximal policy).
    The tensors of the stat dict share memory: one that is kept for longer keeps all of them, 45 bytes a token.
    """
    loss_mask = mb_input["loss_mask"].bool()
    old_logp = mb_input["logprobs"]
    prox_logp = mb_input.get("prox_logp")
    if (fused and not use_sapo_loss and importance_sampling_level == "token" and prox_logp is not None
            and not inplace_backward and torch.is_grad_enabled() and logits.requires_grad
            and _float32_total(total_loss_weight)):
        # one call that counts the tokens itself
        scale = _PerValidToken(total_loss_weight, loss_multiplier)
        out = _unless_weightless(
            lambda: fused_logprobs_ppo_loss(
                logits, rolled_labels(model_inputs), prox_logp, old_logp, mb_input["advantages"], eps_clip, loss_mask,
                eps_clip_higher, c_clip, rejection_sampling, importance_sampling_level, mb_input.get("cu_seqlens"),
                temperature, scale),
            _no_tokens(scale, loss_mask), 2 * logits.numel() * logits.element_size() <= RUN_AHEAD_BYTES)
        return (logits.mean() * 0.0, {}) if out is None else out
    local_weight = loss_mask.count_nonzero()
    if local_weight == 0:
        return logits.mean() * 0.0, {}
    labels = rolled_labels(model_inputs)
    if prox_logp is None and not use_sapo_loss:
        raise ValueError("prox_logp is None: only the recomputed proximal log-probs are supported here")
    scale = local_weight / total_loss_weight * loss_multiplier
    if use_sapo_loss and fused and importance_sampling_level == "token":
        from .sapo import fused_logprobs_sapo_loss

        return fused_logprobs_sapo_loss(logits, labels, old_logp, mb_input["advantages"], sapo_tau_pos, sapo_tau_neg,
                                        loss_mask, temperature=temperature, loss_scale=scale,
                                        inplace_backward=inplace_backward)
    if use_sapo_loss:
        raise ValueError("use_sapo_loss is built for the fused token-level call; use compute_loss_with(grpo_loss_fn) otherwise")
    kw = dict(
        eps_clip=eps_clip, eps_clip_higher=eps_clip_higher, c_clip=c_clip, rejection_sampling=rejection_sampling,
        importance_sampling_level=importance_sampling_level, cu_seqlens=mb_input.get("cu_seqlens"),
    )
    if fused:
        return fused_logprobs_ppo_loss(
            logits, labels, prox_logp, old_logp, mb_input["advantages"], loss_mask=loss_mask,
            temperature=temperature, loss_scale=scale, inplace_backward=inplace_backward, **kw,
        )
    logp, entropy, vmin, vmax = gather_logprobs_entropy_stats(logits, labels, temperature, inplace_backward)
    if pad_length > 0:
        logp, entropy, vmin, vmax = (t[:-pad_length] for t in (logp, entropy, vmin, vmax))
    loss, stat = ppo_actor_loss_fn(logp, prox_logp, old_logp, mb_input["advantages"], loss_mask=loss_mask, **kw)
    stat.update(logprobs=logp.detach(), entropy=entropy.detach(), vocab_min_logits=vmin, vocab_max_logits=vmax)
    return loss * scale, stat


def compute_lm_head_logprobs(hidden: torch.Tensor, weight: torch.Tensor, model_inputs: dict[str, Any],
                             temperature: float = 1.0, token_mask: torch.Tensor | None = None) -> torch.Tensor:
    """Forward-only log-probs of a micro-batch (fsdp_engine.py:1938-1964) from the final hidden states and the
    lm_head weight, without the ``[T_pad, V]`` logits.  ``token_mask`` (optional, beyond the reference's semantics):
    only these tokens go through the lm_head, the others get 0."""
    if hidden.ndim == 3 and hidden.shape[0] == 1:
        hidden = hidden.squeeze(0)
    return lm_head_logprobs_entropy(hidden, weight, rolled_labels(model_inputs), temperature, token_mask)[0]


def compute_lm_head_and_loss(
    hidden: torch.Tensor,
    weight: torch.Tensor,
    model_inputs: dict[str, Any],
    mb_input: dict[str, Any],
    pad_length: int,
    total_loss_weight: torch.Tensor | float,
    eps_clip: float,
    eps_clip_higher: float | None = None,
    c_clip: float | None = None,
    rejection_sampling: Any | None = None,
    importance_sampling_level: str = "token",
    temperature: float = 1.0,
    loss_multiplier: float = 1.0,
    host_loss_mask: torch.Tensor | None = None,
    backward: str = "carry",
) -> tuple[torch.Tensor, dict]:
    """``compute_logprobs_and_loss`` (fsdp_engine.py:1977-2046) one step earlier in the model: from the final hidden
    states ``[T_pad, H]`` (a leading batch dimension of 1 is dropped, as ``outputs.logits.squeeze(0)``,
    fsdp_engine.py:747) and the lm_head weight ``[V, H]``, so that the ``[T_pad, V]`` logits are never written.

    Same contract otherwise: labels are the packed ``input_ids`` rolled by one over the whole tensor
    (``rolled_labels``), the last ``pad_length`` rows are batch padding (they get no gradient and no outputs), the loss
    is scaled by ``local_weight / total_loss_weight * loss_multiplier`` with ``local_weight =
    loss_mask.count_nonzero()`` (actor.py:363), and a micro-batch without any unmasked token returns a zero that keeps
    the graph to ``hidden`` and ``weight`` alive (fsdp_engine.py:1987-1989).  The stat dict is that of
    ``fused_logprobs_ppo_loss`` (``logprobs``, ``entropy``, ``vocab_min_logits``, ``vocab_max_logits`` and the entries
    of ``ppo_actor_loss_fn``), i.e. what ``grpo_loss_fn`` is given and returns.

    ``host_loss_mask``: the host (CPU) copy of ``mb_input["loss_mask"]`` that the data loader still holds.  With it
    nothing is read back from the device: the weight of the micro-batch and the number of tokens with a gradient per
    chunk of ``lm_head_chunk_tokens()`` tokens, which size the gradient GEMMs, are counted on the host.  Rejection
    sampling can only shrink the mask on the device; the counts are then upper bounds, and the rows beyond the true
    count are cleared on the device.  Without it the call reads them from the device, as the reference's
    ``local_weight == 0`` does.
    """
    if hidden.ndim == 3 and hidden.shape[0] == 1:
        hidden = hidden.squeeze(0)
    if hidden.ndim != 2 or hidden.shape[0] - pad_length != mb_input["loss_mask"].shape[0]:
        raise ValueError(
            f"hidden {tuple(hidden.shape)} with pad_length {pad_length} does not fit loss_mask "
            f"{tuple(mb_input['loss_mask'].shape)}"
        )
    loss_mask = mb_input["loss_mask"].bool()
    kept = None
    if host_loss_mask is not None:
        host = host_loss_mask.reshape(-1).ne(0)
        if host.is_cuda or host.shape[0] != loss_mask.shape[0]:
            raise ValueError("host_loss_mask must be the CPU copy of mb_input['loss_mask']")
        local_weight: Any = int(host.sum())
        chunk = lm_head_chunk_tokens()
        kept = [int(host[i:i + chunk].sum()) for i in range(0, hidden.shape[0], chunk)]
    old_logp = mb_input["logprobs"]
    prox_logp = mb_input.get("prox_logp")
    scale: Any = None
    if host_loss_mask is None:
        if (prox_logp is not None and importance_sampling_level == "token" and torch.is_grad_enabled()
                and (hidden.requires_grad or weight.requires_grad) and _float32_total(total_loss_weight)):
            # the step counts the tokens itself
            scale = _PerValidToken(total_loss_weight, loss_multiplier)
        else:
            local_weight = loss_mask.count_nonzero()
    if scale is None and local_weight == 0:
        return hidden.mean() * 0.0 + weight.mean() * 0.0, {}
    if prox_logp is None:
        raise ValueError("prox_logp is None: only the recomputed proximal log-probs are supported here")

    def step(loss_scale):
        return fused_lm_head_ppo_loss(
            hidden, weight, rolled_labels(model_inputs), prox_logp, old_logp, mb_input["advantages"], eps_clip=eps_clip,
            loss_mask=loss_mask, eps_clip_higher=eps_clip_higher, c_clip=c_clip, rejection_sampling=rejection_sampling,
            importance_sampling_level=importance_sampling_level, cu_seqlens=mb_input.get("cu_seqlens"),
            temperature=temperature, loss_scale=loss_scale, kept_per_chunk=kept, backward=backward,
        )

    if scale is None:
        return step(local_weight / total_loss_weight * loss_multiplier)
    out = _unless_weightless(lambda: step(scale), _no_tokens(scale, loss_mask),
                             2 * hidden.numel() * weight.shape[0] <= RUN_AHEAD_FLOPS)
    return (hidden.mean() * 0.0 + weight.mean() * 0.0, {}) if out is None else out


def compute_advantages(
    data: dict[str, Any],
    *,
    kl_ctl: float = 0.0,
    kl_estimator: str = "k1",
    discount: float = 1.0,
    gae_lambda: float = 1.0,
    reward_bias: float = 0.0,
    reward_scaling: float = 1.0,
    reward_clip: float = 20.0,
    reward_norm: Any | None = None,
    adv_norm: Any | None = None,
    mask_no_eos_with_zero: bool = False,
    use_decoupled_loss: bool = False,
    recompute_logprob: bool = False,
    overlong_tokens: int | None = None,
    overlong_penalty_factor: float | None = None,
    max_new_tokens: int | None = None,
) -> dict[str, Any]:
    """``PPOActor._compute_advantages`` (areal/trainer/ppo/actor.py:145-250) on the GPU for one padded batch.

    ``data`` holds ``input_ids``, ``attention_mask``, ``loss_mask``, ``logprobs``, ``rewards`` as ``[bs, max_seqlen]``
    (``rewards`` is ``[bs]``) and optionally ``ref_logp``, ``values``, ``prox_logp``.  ``reward_norm`` / ``adv_norm``
    are ``Normalization`` objects or None.  Writes ``advantages``, ``returns``, ``kl_rewards``, ``tot_rewards``,
    the rolled ``loss_mask`` and ``logprobs`` back into ``data`` and returns it, as the reference does.  With
    ``overlong_tokens`` set (the reference's ``overlong_reward_penalty``), the length penalty of
    ``reward_overlong_penalty`` is applied to ``data["rewards"]`` first, in place (actor.py:152-164).
    """
    if overlong_tokens is not None:                                          # actor.py:152-164
        from .advantages import reward_overlong_penalty

        assert overlong_penalty_factor is not None and max_new_tokens is not None
        data = reward_overlong_penalty(data, overlong_tokens, overlong_penalty_factor, max_new_tokens)
    recomputed = not use_decoupled_loss and recompute_logprob

    def one_pass(reward_score, scores=None):
        return advantage_rows(data["loss_mask"], data["prox_logp"] if recomputed else data["logprobs"], not recomputed,
                              data.get("ref_logp"), data["attention_mask"], reward_score, data.get("values"), kl_ctl,
                              kl_estimator, discount, gae_lambda, mask_no_eos_with_zero, adv_norm, scores)

    scores = score_step(data["rewards"], reward_bias, reward_scaling, reward_clip, reward_norm)
    rows = None if scores is None else one_pass(data["rewards"], scores)
    if rows is None:
        reward_score = reward_scores(data["rewards"], reward_bias, reward_scaling, reward_clip, reward_norm)
        if reward_score is None:
            reward_score = (data["rewards"] + reward_bias) * reward_scaling      # actor.py:166-170
            reward_score = torch.clip(reward_score, max=reward_clip, min=-reward_clip)
            if reward_norm is not None:
                reward_score = reward_norm(reward_score)
        rows = one_pass(reward_score)
    if rows is not None:  # the whole of what follows in one pass per row
        loss_mask, old_logp, kl_rewards, rewards, advantages, returns = rows
        if not use_decoupled_loss and not recomputed:
            data["prox_logp"] = old_logp
        data.update(returns=returns, advantages=advantages, kl_rewards=kl_rewards, tot_rewards=rewards,
                    loss_mask=loss_mask, logprobs=old_logp)
        return data
    loss_mask = torch.roll(data["loss_mask"].float(), shifts=-1, dims=-1)    # :174-175
    if not use_decoupled_loss and recompute_logprob:                          # :177-186
        prox = data["prox_logp"]
        if prox is None:
            raise ValueError(
                "prox_logp is None but recompute_logprob=True. This indicates compute_logp() was skipped incorrectly."
            )
        old_logp = data["logprobs"] = prox
    else:
        old_logp = torch.roll(data["logprobs"], shifts=-1, dims=-1)          # :188
        if not use_decoupled_loss:
            data["prox_logp"] = old_logp
    # in place, as the reference does (:192-196): data["prox_logp"] (when it is this tensor) and data["ref_logp"]
    # come out masked as well
    old_logp.mul_(loss_mask)
    ref_logp = data.get("ref_logp")
    if ref_logp is not None:
        ref_logp.mul_(loss_mask)
    seqlens = data["attention_mask"].sum(-1).long()                           # :199-201
    rewards, kl_rewards = kl_regularized_rewards(old_logp, ref_logp, loss_mask, seqlens, reward_score, kl_ctl,
                                                 kl_estimator, mask_no_eos_with_zero)
    values = data.get("values")
    no_eos = seqlens == data["attention_mask"].shape[1]
    advantages, returns = gae_advantages(rewards, values, loss_mask, no_eos, discount, gae_lambda)   # :209-232
    data["returns"] = returns
    if adv_norm is not None:
        advantages = adv_norm(advantages, loss_mask)                          # :235-236
    data["advantages"] = advantages
    data["kl_rewards"] = kl_rewards
    data["tot_rewards"] = rewards
    data["loss_mask"] = loss_mask
    data["logprobs"] = old_logp
    return data


PROX_LOGP_METHOD_RECOMPUTE = "recompute"
PROX_LOGP_METHOD_LOGLINEAR = "loglinear"
PROX_LOGP_METHOD_METRICS = "metrics"


def infer_token_denominator(input_data: dict[str, Any], fallback: torch.Tensor) -> torch.Tensor:
    """All-true mask whose size is the number of logical tokens of the micro-batch, for the ``n_tokens``
    denominator of the logged statistics (areal/trainer/ppo/stats.py:10-40): the shape of ``attention_mask`` if
    that is a tensor, else ``cu_seqlens[-1]`` tokens, else the shape of ``input_ids`` when it matches ``fallback``,
    else the shape of ``fallback``."""
    common = dict(dtype=torch.bool, device=fallback.device)
    attention_mask = input_data.get("attention_mask")
    if isinstance(attention_mask, torch.Tensor):
        return torch.ones_like(attention_mask, **common)
    cu_seqlens = input_data.get("cu_seqlens")
    if isinstance(cu_seqlens, torch.Tensor) and cu_seqlens.numel() > 0:
        return torch.ones(int(cu_seqlens[-1].item()), **common)
    input_ids = input_data.get("input_ids")
    if isinstance(input_ids, torch.Tensor) and input_ids.shape == fallback.shape:
        return torch.ones_like(input_ids, **common)
    return torch.ones_like(fallback, **common)


def _ends_in_cu_seqlens(input_data: dict[str, Any]) -> bool:
    """Whether the number of logical tokens is the end of the last packed sequence (a number on the device)."""
    cu_seqlens = input_data.get("cu_seqlens")
    return (not isinstance(input_data.get("attention_mask"), torch.Tensor) and isinstance(cu_seqlens, torch.Tensor)
            and cu_seqlens.numel() > 0)


def _n_tokens(input_data: dict[str, Any], fallback: torch.Tensor, step=None) -> int:
    """``infer_token_denominator(input_data, fallback).numel()`` without the mask; ``step``: the step whose counts came to
    the host with the end of its ``cu_seqlens``, so that nothing else is read back."""
    attention_mask = input_data.get("attention_mask")
    if isinstance(attention_mask, torch.Tensor):
        return attention_mask.numel()
    if _ends_in_cu_seqlens(input_data):
        if step is not None and step.slot is not None and step.struct.cu_seqlens:
            return step.slot.read()[2]
        return int(input_data["cu_seqlens"][-1].item())
    input_ids = input_data.get("input_ids")
    if isinstance(input_ids, torch.Tensor) and input_ids.shape == fallback.shape:
        return input_ids.numel()
    return fallback.numel()


def resolve_proximal_logp(prox_logp_gt, prox_logp_method: str, old_logp, logprobs, versions, current_version):
    """``_resolve_proximal_logp`` (areal/trainer/ppo/actor.py:687-765): the recomputed proximal log-probs when
    they are there, the log-linear approximation from per-token versions when the forward pass was skipped."""
    from .actor_ops import compute_prox_logp_approximations

    if prox_logp_method not in (PROX_LOGP_METHOD_RECOMPUTE, PROX_LOGP_METHOD_LOGLINEAR, PROX_LOGP_METHOD_METRICS):
        raise ValueError(f"'{prox_logp_method}' is not a valid ProxLogpMethod")
    if prox_logp_gt is None:
        if prox_logp_method != PROX_LOGP_METHOD_LOGLINEAR:  # the only method that skips the forward pass
            raise ValueError(
                f"prox_logp is None but prox_logp_method='{prox_logp_method}'. "
                "This indicates compute_logp() was skipped incorrectly."
            )
        if versions is None:
            raise ValueError(
                f"prox_logp is None with prox_logp_method='{prox_logp_method}' but versions not available. "
                "Cannot proceed without either ground truth or approximation."
            )
    prox_logp = prox_logp_gt
    if prox_logp_method == PROX_LOGP_METHOD_LOGLINEAR:
        if prox_logp_gt is None and versions is not None and current_version is not None:
            prox_logp = compute_prox_logp_approximations(old_logp, logprobs, versions, current_version,
                                                         method="loglinear")["loglinear"]
    if prox_logp is None:
        raise RuntimeError(
            f"prox_logp is None after handling prox_logp_method='{prox_logp_method}'. "
            "This indicates configuration or computation error."
        )
    return prox_logp


def grpo_loss_fn(
    logprobs: torch.Tensor,
    entropy: torch.Tensor,
    input_data: dict,
    eps_clip: float,
    eps_clip_higher: float | None,
    c_clip: float | None,
    rejection_sampling: Any | None = None,
    m2_threshold: float | None = None,
    importance_sampling_level: str = "token",
    current_version: int | None = None,
    prox_logp_method: str = PROX_LOGP_METHOD_RECOMPUTE,
    use_sapo_loss: bool = False,
    sapo_tau_pos: float = 1.0,
    sapo_tau_neg: float = 1.05,
    use_decoupled_loss: bool = False,
    vocab_min_logits: torch.Tensor | None = None,
    vocab_max_logits: torch.Tensor | None = None,
) -> tuple[torch.Tensor, dict]:
    """The actor's loss function for one micro-batch (areal/trainer/ppo/actor.py:408-480) on the GPU ops: proximal
    log-probs resolved, optional M2PO masking, SAPO or clipped PPO loss, and the joint-distillation terms
    (``teacher_logp`` with ``rl_loss_weight`` / ``distill_loss_weight``, actor.py:482-511).

    Returns ``(loss, stat)``.  ``stat`` is the per-token dict of the loss function plus ``"reduced"``: what the
    reference hands to its statistics tracker tensor by tensor (actor.py:513-573) as sums / averages / extrema
    under the same denominators, computed in one launch per denominator, and under ``"compute_logp"`` and
    ``"version_stats"`` what it logs in those scopes (actor.py:573-594, 982-1110; ``proximal_logging_stats``).
    """
    from .actor_ops import apply_m2po_masking, distillation_terms, proximal_logging_stats
    from .advantages import moments_table
    from .functional import sapo_loss_fn

    old_logp = input_data["logprobs"]
    advantages = input_data["advantages"]
    loss_mask = input_data["loss_mask"].bool()
    entropy = entropy.detach()
    prox_logp = resolve_proximal_logp(input_data.get("prox_logp"), prox_logp_method, old_logp, logprobs.detach(),
                                      input_data.get("versions"), current_version)
    if m2_threshold is not None:
        loss_mask = apply_m2po_masking(old_logp, prox_logp, loss_mask, m2_threshold)
    step = None
    if use_sapo_loss:
        if use_decoupled_loss:
            raise ValueError(
                "SAPO is not compatible with `use_decoupled_loss=True`. "
                "Please set `actor.use_decoupled_loss=false` in your configuration."
            )
        loss, stat = sapo_loss_fn(logprobs, old_logp, advantages, sapo_tau_pos, sapo_tau_neg, loss_mask,
                                  importance_sampling_level, input_data.get("cu_seqlens"))
    else:
        loss, stat, step = _ppo_actor_loss(logprobs, prox_logp, old_logp, advantages, eps_clip, loss_mask, eps_clip_higher,
                                           c_clip, rejection_sampling, importance_sampling_level,
                                           input_data.get("cu_seqlens"),
                                           host_counts=_ends_in_cu_seqlens(input_data))
    rkl_stat = None
    teacher_logp = input_data.get("teacher_logp")
    if teacher_logp is not None:
        rl_loss_weight = input_data.get("rl_loss_weight", 1.0)
        distill_loss_weight = input_data.get("distill_loss_weight", 0.005)
        if rl_loss_weight == 0:  # pure distillation with the reverse KL as an importance-weighted reward
            mean, term = distillation_terms(logprobs, old_logp, teacher_logp, loss_mask, pure=True)
            loss = -distill_loss_weight * mean
            rkl_stat = -term
        else:                    # the RL loss plus a reverse-KL penalty
            mean, term = distillation_terms(logprobs, None, teacher_logp, loss_mask, pure=False)
            loss = rl_loss_weight * loss + distill_loss_weight * mean
            rkl_stat = term
    per_valid = dict(
        importance_weight=stat["importance_weight"], approx_kl=stat["approx_kl"], new_logp=logprobs, old_logp=old_logp,
        entropy=entropy, actor_loss=stat["loss"], clip_ratio=stat["clip_mask"], dual_clip_ratio=stat["dual_clip_mask"],
    )
    if use_sapo_loss:
        per_valid.update(sapo_soft_gate=stat["sapo_soft_gate"], sapo_scaled_gate_pos=stat["sapo_scaled_gate_pos"],
                         sapo_scaled_gate_neg=stat["sapo_scaled_gate_neg"])
    if rkl_stat is not None:
        per_valid.update(rkl_loss=rkl_stat)
    # every logged tensor under its own mask, one launch
    entries = [(name, t, loss_mask) for name, t in per_valid.items()]
    if not use_sapo_loss:
        clip_mask = stat["clip_mask"]
        entries += [("clipped_new_logp", logprobs, clip_mask), ("clipped_old_logp", old_logp, clip_mask)]
    if "behave_imp_weight" in stat:
        entries += [(k, stat[k], stat["behave_mask"]) for k in ("behave_imp_weight", "behave_approx_kl")]
    if vocab_min_logits is not None and vocab_max_logits is not None:
        entries += [("vocab_min_logits", vocab_min_logits, None), ("vocab_max_logits", vocab_max_logits, None)]
    reduced = moments_table(entries)
    # the compute_logp and version_stats scopes (actor.py:573-594) under the mask the loss kept
    reduced.update(proximal_logging_stats(old_logp, logprobs.detach(), input_data.get("prox_logp"),
                                          input_data.get("versions"), current_version,
                                          stat.get("behave_mask", loss_mask), prox_logp_method))
    # what the host has to wait for comes last, when everything is queued
    reduced["n_tokens"] = _n_tokens(input_data, loss_mask, step)
    if step is not None:
        step.finish(stat)
    if "filtered_fraction" in stat:
        reduced["rs_filtered_fraction"] = stat["filtered_fraction"]
    stat = dict(stat, loss_mask=loss_mask, reduced=reduced)
    return loss, stat


def critic_loss_fn(value: torch.Tensor, input_data: dict[str, Any], eps_clip: float) -> tuple[torch.Tensor, dict]:
    """The critic's loss function for one micro-batch (areal/trainer/ppo/critic.py:105-149) on the GPU ops.

    Returns ``(loss, stat)`` with ``stat["reduced"]`` holding what the reference logs tensor by tensor (sums,
    averages, extrema under ``n_valid_tokens`` and ``clipped_tokens``) and ``n_tokens``."""
    from .advantages import moments_table
    from .functional import ppo_critic_loss_fn

    value = value.squeeze(-1).float()
    old_value = input_data["values"].float()
    target_value = input_data["returns"].float()
    loss_mask = input_data["loss_mask"].bool()
    loss, stat = ppo_critic_loss_fn(value, old_value, target_value, eps_clip, loss_mask)
    clip_mask = stat["clip_mask"]
    reduced = moments_table(
        [("new_value", value, loss_mask), ("old_value", old_value, loss_mask), ("target_value", target_value, loss_mask),
         ("critic_loss", stat["loss"], loss_mask), ("clip_ratio", clip_mask, loss_mask),
         ("clipped_new_value", value, clip_mask), ("clipped_old_value", old_value, clip_mask)])
    reduced["n_tokens"] = _n_tokens(input_data, value)
    return loss, dict(stat, loss_mask=loss_mask, reduced=reduced)


def dpo_valid_pairs(x: dict[str, Any]) -> torch.Tensor:
    """Pairs whose chosen and rejected sequences are both non-empty (areal/trainer/dpo/dpo_engine.py:22-24)."""
    seqlens = x["cu_seqlens"][1:] - x["cu_seqlens"][:-1]
    return seqlens.view(-1, 2).ne(0).all(dim=1)


def dpo_loss_weight(x: dict[str, Any]) -> torch.Tensor:
    """Number of valid pairs as a float, the weight of a micro-batch (dpo_engine.py:27-28)."""
    return dpo_valid_pairs(x).count_nonzero().float()


def compute_dpo_loss(logprobs: torch.Tensor, entropy: torch.Tensor | None, input_: dict[str, Any], *, beta: float,
                     loss_type: str = "sigmoid", vocab_min_logits: torch.Tensor | None = None,
                     vocab_max_logits: torch.Tensor | None = None) -> tuple[torch.Tensor, dict]:
    """The DPO loss function of one packed micro-batch (dpo_engine.py:147-213) on the GPU ops.

    ``input_`` holds ``cu_seqlens``, ``loss_mask`` and ``ref_logprobs`` (``KeyError`` if one is missing), sequences
    interleaved chosen / rejected.  Returns ``(loss, stat)``: the mean over the valid pairs (0 when there are none,
    found on the device, without a read-back) and what the reference records per pair under its ``n_pairs``
    denominator: ``loss``, ``chosen_reward``, ``rejected_reward``, ``reward_accuracy``, ``reward_margin``, with
    ``valid_pairs`` selecting the pairs that count and ``n_pairs`` their number."""
    from .dpo import dpo_loss

    loss, stat = dpo_loss(logprobs, input_["ref_logprobs"], input_["cu_seqlens"], input_["loss_mask"], beta=beta,
                          loss_type=loss_type)
    with torch.no_grad():
        stat["reward_accuracy"] = (stat["chosen_reward"] > stat["rejected_reward"]).float()
        stat["reward_margin"] = stat["chosen_reward"] - stat["rejected_reward"]
    return loss, stat


def compute_packed_sft_loss(logprobs: torch.Tensor, entropy: torch.Tensor | None, input_: dict[str, Any],
                            vocab_min_logits: torch.Tensor | None = None,
                            vocab_max_logits: torch.Tensor | None = None) -> tuple[torch.Tensor, dict]:
    """The SFT loss function of one packed micro-batch (areal/trainer/sft/lm_engine.py:81-131) on the GPU ops.

    Returns ``(loss, stat)``; ``stat`` holds what the reference records: per token ``loss`` under ``n_valid_tokens``
    (= ``loss_mask``), per sequence ``ppl`` under ``n_seqs`` (the sequences with a selected token), and in
    ``stat["reduced"]`` the moments of ``loss`` and of the vocabulary extrema (under all tokens) when given."""
    from .advantages import moments_table
    from .sft import sft_loss_fn

    del entropy  # SFT does not use entropy
    loss_mask = input_["loss_mask"].bool()
    loss, stat = sft_loss_fn(logprobs, loss_mask, input_["cu_seqlens"])
    entries = [("loss", stat["loss"], loss_mask)]
    if vocab_min_logits is not None and vocab_max_logits is not None:
        entries += [("vocab_min_logits", vocab_min_logits, None), ("vocab_max_logits", vocab_max_logits, None)]
    reduced = moments_table(entries)
    reduced["n_tokens"] = logprobs.shape[0]
    return loss, dict(stat, loss_mask=loss_mask, reduced=reduced)


def rw_valid_pairs(x: dict[str, Any]) -> torch.Tensor:
    """Pairs whose chosen and rejected sequences are both non-empty (areal/trainer/rw/rw_engine.py:20-22)."""
    return dpo_valid_pairs(x)


def rw_loss_weight(x: dict[str, Any]) -> torch.Tensor:
    """Number of valid pairs as a float (rw_engine.py:25-26)."""
    return rw_valid_pairs(x).count_nonzero().float()


def compute_rw_loss(scores: torch.Tensor, input_: dict[str, Any]) -> tuple[torch.Tensor, dict]:
    """The reward-model loss function of one packed micro-batch (rw_engine.py:115-146) on the GPU ops.  Returns
    ``(loss, stat)`` with what the reference records per pair under ``n_pairs``: ``loss``, ``pos_score``,
    ``neg_score``, ``correct_ratio``, selected by ``valid_pairs``."""
    from .dpo import rw_pair_loss

    loss, stat = rw_pair_loss(scores, input_["cu_seqlens"])
    with torch.no_grad():
        stat["correct_ratio"] = (stat["pos_score"] > stat["neg_score"]).float()
    return loss, stat


def compute_loss_with(logits: torch.Tensor, model_inputs: dict[str, Any], mb_input: dict[str, Any], pad_length: int,
                      loss_fn, loss_weight_fn, total_loss_weight: torch.Tensor | float, temperature: float = 1.0,
                      loss_multiplier: float = 1.0, is_critic: bool = False, trie_node: Any = None):
    """``_compute_logprobs_and_loss`` for any loss function (areal/engine/fsdp_engine.py:1977-2046): log-probs,
    entropy and the vocabulary extrema of the micro-batch in one pass over the logits (packed trees: through the
    tree gather), the batch padding trimmed, ``loss_fn(logprobs, entropy, mb_input, vocab_min_logits=...,
    vocab_max_logits=...)`` (a critic: ``loss_fn(values, mb_input)``), scaled by ``local_weight / total_loss_weight *
    loss_multiplier``.  ``loss_fn`` may return the loss alone, like the reference's, or ``(loss, stat)`` like the
    loss functions of this module; the return value has the same form.  A micro-batch of weight 0 returns
    ``logits.mean() * 0``."""
    local_weight = loss_weight_fn(mb_input)
    zero_weight = _weight_is_zero(local_weight)
    if (is_critic or trie_node is not None) and zero_weight[0]():
        return logits.mean() * 0.0
    if is_critic:
        if trie_node is not None:
            raise NotImplementedError("Tree training with critic model is not supported yet.")
        values = logits.squeeze(-1)
        if pad_length > 0:
            values = values[:-pad_length]
        out = loss_fn(values, mb_input)
    else:
        if trie_node is not None:
            from .tree import gather_packed_tree_logprobs_entropy, gather_packed_tree_vocab_stats

            if not trie_node.all_sequence_ids:
                return logits.mean() * 0.0
            vmin, vmax = gather_packed_tree_vocab_stats(logits, trie_node)
            logp, entropy = gather_packed_tree_logprobs_entropy(logits, trie_node, mb_input["input_ids"],
                                                                temperature=temperature)
        else:
            def forward():
                labels = rolled_labels(model_inputs)
                if logits.dim() == 2 and logits.shape[0] > pad_length:
                    lp, ent, hi, lo = _logprobs_impl(logits, labels, temperature, None, True, True,
                                                     T_active=logits.shape[0] - pad_length if pad_length > 0 else None)
                    return lp, ent, lo, hi
                rows = gather_logprobs_entropy_stats(logits, labels, temperature)
                return tuple(t[:-pad_length] for t in rows) if pad_length > 0 else rows

            rows = _unless_weightless(forward, zero_weight, logits.numel() * logits.element_size() <= RUN_AHEAD_BYTES)
            if rows is None:
                return logits.mean() * 0.0
            logp, entropy, vmin, vmax = rows
        out = loss_fn(logp, entropy, mb_input, vocab_min_logits=vmin, vocab_max_logits=vmax)
    if isinstance(out, tuple):
        return _times_weight(out[0], local_weight, zero_weight[2], total_loss_weight, loss_multiplier), out[1]
    return _times_weight(out, local_weight, zero_weight[2], total_loss_weight, loss_multiplier)


def compute_lm_head_loss_with(hidden: torch.Tensor, weight: torch.Tensor, model_inputs: dict[str, Any],
                              mb_input: dict[str, Any], pad_length: int, loss_fn, loss_weight_fn,
                              total_loss_weight: torch.Tensor | float, temperature: float = 1.0,
                              loss_multiplier: float = 1.0, backward: str = "carry",
                              grad_token_mask: torch.Tensor | None = None, kept_per_chunk: list[int] | None = None):
    """``compute_loss_with`` one step earlier in the model: any loss function of the reference's form
    (``grpo_loss_fn`` with sequence-level ratios, SAPO, M2PO or distillation terms, ``compute_packed_sft_loss``, a custom
    one) on the final hidden states ``[T_pad, H]`` and the lm_head weight ``[V, H]``, without the ``[T_pad, V]`` logits:
    log-probs, entropy and the vocabulary extrema come from ``lm_head_logprobs_entropy_stats``, the batch padding is
    trimmed, ``loss_fn(logprobs, entropy, mb_input, vocab_min_logits=..., vocab_max_logits=...)`` is called as the
    engine calls it (fsdp_engine.py:2032-2040) and its result scaled by ``local_weight / total_loss_weight *
    loss_multiplier``.  A micro-batch of weight 0 returns a zero that keeps the graph to ``hidden`` and ``weight``.

    ``backward="carry"`` (default): the op keeps the bf16 probability ratios of the tokens named by ``grad_token_mask``
    (default: ``mb_input["loss_mask"]``; tokens outside it get no gradient) from its forward to its backward, which is
    then two GEMMs instead of three; ``kept_per_chunk``: their number per chunk of ``lm_head_chunk_tokens()`` tokens,
    if the host knows it.  Otherwise the device counts them, and the op keeps room for every token, up to
    ``COUNT_ON_DEVICE_BYTES`` (2 GiB) of rows; past that the counts are read back and the rows sized by them.
    ``"recompute"`` keeps nothing and forms the logits again."""
    if hidden.ndim == 3 and hidden.shape[0] == 1:
        hidden = hidden.squeeze(0)
    local_weight = loss_weight_fn(mb_input)

    def forward():
        # (a micro-batch of nothing but padding goes through the op with its padding rows, which are then cut off)
        trim = 0 < hidden.shape[0] <= pad_length
        n_rows = hidden.shape[0] - (pad_length if pad_length > 0 and not trim else 0)
        carry = backward == "carry"
        mask = grad_token_mask
        if mask is None and carry:
            mask = mb_input.get("loss_mask")
        if mask is not None:
            mask = mask.reshape(-1)
            if mask.dtype is not torch.bool:
                mask = mask.ne(0)
            if pad_length > 0:  # without padding the op refuses a mask of another length
                mask = torch.nn.functional.pad(mask, (0, n_rows - mask.shape[0])) if mask.shape[0] < n_rows else mask[:n_rows]
        rows = _lm_head_impl(
            hidden, weight, rolled_labels(model_inputs), temperature, None, True, backward, mask if carry else None,
            kept_per_chunk if carry else None, count_on_device=2 * n_rows * weight.shape[0] <= COUNT_ON_DEVICE_BYTES,
            T_active=n_rows)
        return tuple(t[:-pad_length] for t in rows) if trim else rows

    zero_weight = _weight_is_zero(local_weight)
    rows = _unless_weightless(forward, zero_weight,
                              2 * hidden.numel() * weight.shape[0] <= RUN_AHEAD_FLOPS)
    if rows is None:
        return hidden.mean() * 0.0 + weight.mean() * 0.0
    logp, entropy, vmin, vmax = rows
    out = loss_fn(logp, entropy, mb_input, vocab_min_logits=vmin, vocab_max_logits=vmax)
    if isinstance(out, tuple):
        return _times_weight(out[0], local_weight, zero_weight[2], total_loss_weight, loss_multiplier), out[1]
    return _times_weight(out, local_weight, zero_weight[2], total_loss_weight, loss_multiplier)


def compute_logprobs_and_sft_loss(logits: torch.Tensor, model_inputs: dict[str, Any], mb_input: dict[str, Any],
                                  total_loss_weight: torch.Tensor | float, temperature: float = 1.0,
                                  loss_multiplier: float = 1.0) -> tuple[torch.Tensor, dict]:
    """The supervised step of one micro-batch in one pass over the logits: what ``compute_loss_with`` does with
    ``loss_fn = compute_packed_sft_loss`` and ``loss_weight_fn = loss_mask.count_nonzero``
    (areal/trainer/sft/lm_engine.py:28-35), fused with the log-prob op and its backward.  ``mb_input`` holds the
    un-padded ``loss_mask`` and ``cu_seqlens``; the rows of ``logits`` past them are the batch padding."""
    from .sft import fused_logprobs_sft_loss

    loss_mask = mb_input["loss_mask"].bool()
    if torch.is_grad_enabled() and logits.requires_grad and _float32_total(total_loss_weight):
        # one call that counts the tokens itself
        per_token = _PerValidToken(total_loss_weight, loss_multiplier)
        out = _unless_weightless(
            lambda: fused_logprobs_sft_loss(logits, rolled_labels(model_inputs), loss_mask, mb_input["cu_seqlens"],
                                            temperature, loss_scale=per_token),
            _no_tokens(per_token, loss_mask), 2 * logits.numel() * logits.element_size() <= RUN_AHEAD_BYTES)
        return (logits.mean() * 0.0, {}) if out is None else out
    local_weight = loss_mask.count_nonzero()
    if local_weight == 0:
        return logits.mean() * 0.0, {}
    scale = local_weight / total_loss_weight * loss_multiplier
    return fused_logprobs_sft_loss(logits, rolled_labels(model_inputs), loss_mask, mb_input["cu_seqlens"], temperature,
                                   loss_scale=scale)
