"""Actor-side per-token helpers that sit next to the loss: proximal log-prob approximations and M2PO masking.

Host-side mirror of ``compute_prox_logp_approximations`` (areal/trainer/ppo/actor.py:604-684) and
``_apply_m2po_masking`` (areal/trainer/ppo/actor.py:769-850).
"""
from __future__ import annotations

from typing import Any

import torch

from . import _native as N
from .advantages import _MOMENT_KEYS
from .functional import _f32, _f32_values, _mask_bytes, _mask_u8, _on, _ptr, _require_gpu, _stream, _work_words

PROX_APPROX_METHOD_LOGLINEAR = "loglinear"
PROX_APPROX_METHOD_LINEAR = "linear"
PROX_APPROX_METHOD_ROLLOUT = "rollout"
PROX_APPROX_METHODS_ALL = [PROX_APPROX_METHOD_LOGLINEAR, PROX_APPROX_METHOD_LINEAR, PROX_APPROX_METHOD_ROLLOUT]
_METHOD_IDS = {PROX_APPROX_METHOD_LOGLINEAR: 0, PROX_APPROX_METHOD_LINEAR: 1, PROX_APPROX_METHOD_ROLLOUT: 2}


@torch.no_grad()
def compute_prox_logp_approximations(old_logp: torch.Tensor, logprobs: torch.Tensor, versions: torch.Tensor,
                                     current_version: int, method: str | None = None) -> dict[str, torch.Tensor]:
    """Version-aware interpolation between behaviour and current log-probs; actor.py:604-684.

    Returns ``{method: tensor}`` for the one method asked for, or for all three when ``method`` is None.  Unknown
    method names give an empty dict, as in the reference.
    """
    _require_gpu(old_logp, "old_logp")
    shape = old_logp.shape
    lo = _f32(old_logp.detach()).reshape(-1)
    ln = _f32(logprobs.detach()).reshape(-1)
    ver = versions.to(device=lo.device, dtype=torch.int32).contiguous().reshape(-1)
    if not (lo.numel() == ln.numel() == ver.numel()):
        raise ValueError("old_logp, logprobs and versions must have the same number of elements")
    lib = N.load()
    out = {}
    for m in ([method] if method else PROX_APPROX_METHODS_ALL):
        if m not in _METHOD_IDS:
            continue
        res = torch.empty_like(lo)
        with torch.cuda.device(lo.device):
            N.check(lib.aa_prox_logp_approx(_ptr(lo), _ptr(ln), _ptr(ver), lo.numel(), int(current_version),
                                            _METHOD_IDS[m], _ptr(res), _stream(lo.device)), "aa_prox_logp_approx")
        out[m] = res.view(shape)
    return out


@torch.no_grad()
def apply_m2po_masking(old_logp: torch.Tensor, prox_logp: torch.Tensor, loss_mask: torch.Tensor,
                       m2_threshold: float) -> torch.Tensor:
    """Loss mask with the highest second-momentum tokens removed; actor.py:769-850.

    Tokens are dropped from the largest ``(old_logp - prox_logp) ** 2`` down until the mean over the remaining valid
    tokens is below ``m2_threshold``; at least one valid token is always kept.  Returns a bool mask of the shape of
    ``loss_mask``.
    """
    _require_gpu(old_logp, "old_logp")
    shape = loss_mask.shape
    lo = _f32(old_logp.detach()).reshape(-1)
    lp = _f32(prox_logp.detach()).reshape(-1)
    m8 = _mask_u8(loss_mask).reshape(-1)
    n = m8.numel()
    if not (lo.numel() == lp.numel() == n):
        raise ValueError("old_logp, prox_logp and loss_mask must have the same number of elements")
    if n == 0:
        return loss_mask.bool()
    lib = N.load()
    dev = lo.device
    ws = torch.empty(lib.aa_m2po_workspace_bytes(n), dtype=torch.uint8, device=dev)
    out = torch.empty(n, dtype=torch.bool, device=dev)
    info = torch.empty(2, dtype=torch.int32, device=dev)
    with _on(dev):
        N.check(lib.aa_m2po_mask(_ptr(lo), _ptr(lp), _ptr(m8), n, float(m2_threshold), _ptr(out), _ptr(info), _ptr(ws),
                                 ws.numel(), _stream(dev)), "aa_m2po_mask")
    return out.view(shape)


class _KdTerms(torch.autograd.Function):
    """sum(term) / max(sum(mask), 1) of ``aa_kd_terms`` and the per-token terms; differentiable in ``logp``."""

    @staticmethod
    def forward(ctx, logp, old, teacher, mask_u8, pure):
        from .functional import _count_nonzero

        lib = N.load()
        dev = logp.device
        n = logp.numel()
        term = torch.empty(n, dtype=torch.float32, device=dev)
        dterm = torch.empty(n, dtype=torch.float32, device=dev)
        mean = torch.empty((), dtype=torch.float32, device=dev)
        n_valid = _count_nonzero(mask_u8)
        with _on(dev):
            st = _stream(dev)
            N.check(lib.aa_kd_terms(_ptr(logp), _ptr(old), _ptr(teacher), _ptr(mask_u8), n, 1 if pure else 0, _ptr(term),
                                    _ptr(dterm), st), "aa_kd_terms")
            N.check(lib.aa_masked_sum(_ptr(term), None, n, _ptr(n_valid), None, _ptr(mean), st), "aa_masked_sum")
        ctx.save_for_backward(dterm, n_valid)
        ctx.mark_non_differentiable(term)
        return mean, term

    @staticmethod
    def backward(ctx, g_mean, _g_term):
        dterm, n_valid = ctx.saved_tensors
        return dterm * (g_mean / n_valid.clamp(min=1).float()), None, None, None, None


def distillation_terms(logprobs: torch.Tensor, old_logp: torch.Tensor | None, teacher_logp: torch.Tensor,
                       loss_mask: torch.Tensor, pure: bool) -> tuple[torch.Tensor, torch.Tensor]:
    """The reverse-KL terms of the joint-distillation branch of the actor loss; actor.py:482-511.

    ``pure`` (``rl_loss_weight == 0``): per token ``exp(logp - old) * (teacher - logp.detach()) * mask``
    (actor.py:494-498); otherwise ``(logp - teacher) * mask`` (actor.py:505).  Returns
    ``(sum(term) / max(sum(mask), 1), term)``: the first is differentiable in ``logprobs``, the second is detached.
    """
    _require_gpu(logprobs, "logprobs")
    shape = logprobs.shape
    if teacher_logp.shape != shape or loss_mask.shape != shape or (pure and old_logp.shape != shape):
        raise ValueError("logprobs, old_logp, teacher_logp and loss_mask must have the same shape")
    lp = logprobs.reshape(-1)
    if lp.dtype != torch.float32 or not lp.is_contiguous():
        lp = lp.float().contiguous()
    old = _f32(old_logp.detach()).reshape(-1) if pure else None
    mean, term = _KdTerms.apply(lp, old, _f32(teacher_logp.detach()).reshape(-1), _mask_u8(loss_mask).reshape(-1),
                                bool(pure))
    return mean, term.view(shape)


_LOGSTAT_METHOD_KEYS = ("approx_logp", "behave_imp_weight", "importance_weight", "abs_error", "rel_error",
                        "squared_error", "behave_imp_weight_abs_error", "behave_imp_weight_rel_error",
                        "importance_weight_abs_error", "importance_weight_rel_error")


@torch.no_grad()
def proximal_logging_stats(old_logp: torch.Tensor, logprobs: torch.Tensor, prox_logp_gt: torch.Tensor | None,
                           versions: torch.Tensor | None, current_version: int | None, mask: torch.Tensor,
                           prox_logp_method: str = "recompute") -> dict[str, dict]:
    """What ``grpo_loss_fn`` logs under its ``compute_logp`` and ``version_stats`` scopes (actor.py:573-594,
    982-1110), already reduced over ``mask``: one pass over the tokens instead of one tensor and one reduction per
    logged quantity.

    Returns ``{"compute_logp": {name: moments}, "version_stats": {...}}`` with ``moments`` = ``{"sum", "avg", "min",
    "max", "count"}`` of 0-d device tensors.  The names and the conditions under which each appears are the
    reference's: ``prox_logp_gt`` whenever it is given; nothing more without ``versions`` / ``current_version``;
    ``loglinear/{approx_logp, behave_imp_weight, importance_weight}`` for the ``"loglinear"`` method; all three
    methods with their error metrics for ``"metrics"`` with ground truth; ``kl_div_direct / taylor / dual``.
    ``version_stats`` holds ``sample_staleness_proximal``, ``sample_staleness_theta`` (moments over the selected
    tokens with ``version >= 0``; ``count`` is ``n_valid_generated_tokens``), ``v_theta`` and ``v_proximal``; it
    is empty without versions.  Nothing is read back: whether any generated token is selected is the ``count``.
    """
    _require_gpu(old_logp, "old_logp")
    lo, ln = _f32_values(old_logp), _f32_values(logprobs)
    m8 = _mask_bytes(mask.to(lo.device))
    n = lo.numel()
    if ln.numel() != n or m8.numel() != n:
        raise ValueError("old_logp, logprobs and mask must have the same number of elements")
    gt = _f32_values(prox_logp_gt) if prox_logp_gt is not None else None
    have_versions = versions is not None and current_version is not None
    ver = versions.to(device=lo.device, dtype=torch.int32).contiguous() if have_versions else None
    methods, with_errors = 0, False
    if have_versions and prox_logp_method == "loglinear":
        methods = 1
    elif have_versions and prox_logp_method == "metrics" and gt is not None:
        methods, with_errors = 7, True
    lib = N.load()
    dev = lo.device
    out = torch.empty(36, 5, dtype=torch.float32, device=dev)
    scratch = torch.empty(lib.aa_logging_stats_scratch_bytes(n), dtype=torch.uint8, device=dev)
    with _on(dev):
        N.check(lib.aa_logging_stats_table(_ptr(lo), _ptr(ln), _ptr(gt), _ptr(ver), _ptr(m8), n,
                                           int(current_version) if have_versions else 0, methods, 1 if with_errors else 0,
                                           _ptr(out), _ptr(scratch), scratch.numel(), _ptr(_work_words(dev)), _stream(dev)),
                "aa_logging_stats_table")
    # the cells of the rows that are returned, as 0-d tensors
    want = {}  # row of the table -> where its moments go
    compute_logp: dict[str, dict] = {}
    version_stats: dict[str, Any] = {}
    if gt is not None:
        want[0] = (compute_logp, "prox_logp_gt")
    if have_versions:
        for m, name in enumerate(PROX_APPROX_METHODS_ALL):
            if not (methods >> m) & 1:
                continue
            for j, key in enumerate(_LOGSTAT_METHOD_KEYS[: 10 if with_errors else 3]):
                want[4 + 10 * m + j] = (compute_logp, f"{name}/{key}")
        for j, key in enumerate(("kl_div_direct", "kl_div_taylor", "kl_div_dual")):
            want[1 + j] = (compute_logp, key)
        want[34] = (version_stats, "sample_staleness_proximal")
        want[35] = (version_stats, "sample_staleness_theta")
    for first, last in ((0, 4), (4, 34), (34, 36)):  # one unbind for each part of the table that is in use
        if any(first <= r < last for r in want):
            cells = out[first:last].view(-1).unbind(0)
            for r, (where, key) in want.items():
                if first <= r < last:
                    where[key] = dict(zip(_MOMENT_KEYS, cells[5 * (r - first) : 5 * (r - first) + 5]))
    if have_versions:
        version_stats.update(v_theta=int(current_version), v_proximal=int(current_version) - 1)
    return dict(compute_logp=compute_logp, version_stats=version_stats)
