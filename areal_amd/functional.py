"""Drop-in functional API of the PPO/GRPO log-prob / entropy / actor-loss path.

Same names, argument meaning and error behaviour as the reference's
``areal.utils.functional`` (vocab_parallel.py:401-469, functional.py:185-559);
the arithmetic runs in hand-written gfx950 kernels reached through the C ABI of
``libareal_amd.so``.  PyTorch is used for device memory, streams and autograd
bookkeeping only.  Tensors must live on a ROCm device: there is no CPU path.
"""
from __future__ import annotations

import contextlib
import ctypes as C
import itertools
import time
from collections import deque
from dataclasses import dataclass
from typing import Any

import torch

from . import _native as N

__all__ = [
    "RejectionSamplingResult",
    "gather_logprobs",
    "gather_logprobs_entropy",
    "gather_logprobs_entropy_stats",
    "apply_rejection_sampling",
    "ppo_actor_loss_fn",
    "fused_logprobs_ppo_loss",
    "lm_head_logprobs_entropy",
    "lm_head_logprobs_entropy_stats",
]

_DTYPES = {torch.bfloat16: N.AA_BF16, torch.float16: N.AA_F16, torch.float32: N.AA_F32}


# ----------------------------------------------------------------------------
# helpers
# ----------------------------------------------------------------------------
def _ptr(t: torch.Tensor | None) -> int | None:
    return None if t is None else t.data_ptr()


def _stream(device: torch.device) -> int:
    return torch._C._cuda_getCurrentRawStream(device.index)


_SAME_DEVICE = contextlib.nullcontext()


def _on(device: torch.device):
    """Context in which ``device`` is the current one; nothing to enter when it is already."""
    return _SAME_DEVICE if torch._C._cuda_getDevice() == device.index else torch.cuda.device(device)


def _require_gpu(t: torch.Tensor, name: str) -> None:
    if not t.is_cuda:
        raise N.NativeLibraryError(
            f"{name} is on {t.device}: areal_amd ops run on a ROCm GPU only (no CPU fallback)"
        )


def _f32(t: torch.Tensor) -> torch.Tensor:
    return t.to(torch.float32).contiguous()


def _f32_values(t: torch.Tensor) -> torch.Tensor:
    """The values of ``t`` as contiguous float32 for a kernel that reads them (no autograd)."""
    if t.dtype is torch.float32 and t.is_contiguous():
        return t
    return t.detach().to(torch.float32).contiguous()


def _mask_u8(mask: torch.Tensor) -> torch.Tensor:
    """One byte per token, non-zero = valid, without a copy for bool masks."""
    m = mask.contiguous()
    if m.dtype == torch.bool:
        return m.view(torch.uint8)
    return (m != 0).view(torch.uint8)


def _mask_bytes(mask: torch.Tensor) -> torch.Tensor:
    """The same for a kernel that only needs the address: a contiguous bool mask as it is."""
    if mask.dtype is torch.bool and mask.is_contiguous():
        return mask
    return _mask_u8(mask)


def _labels_i64(labels: torch.Tensor, dev: torch.device) -> torch.Tensor:
    if labels.dtype is torch.int64 and labels.device == dev and labels.is_contiguous():
        return labels
    return labels.to(device=dev, dtype=torch.int64).contiguous()


def _rows(logits: torch.Tensor) -> tuple[torch.Tensor, int, int, int]:
    """View logits as [T, V] rows with unit inner stride; returns (2-D tensor, T, V, row stride)."""
    V = logits.shape[-1]
    x = logits if logits.dim() == 2 else logits.reshape(-1, V)
    if x.dtype not in _DTYPES:
        x = x.float()
    if x.stride(-1) != 1 or (x.shape[0] > 1 and x.stride(0) < V):
        x = x.contiguous()
    T = x.shape[0]
    stride = x.stride(0) if T > 1 else V
    return x, T, V, stride


def _empty_rows_like(logits2d: torch.Tensor, stride: int) -> torch.Tensor:
    """An uninitialised [T, V] array for the gradient of ``logits2d``, laid out like it (``csrc/host.cpp``)."""
    return N.host().empty_rows_like(logits2d, stride)


def _check_tp(tp_group: Any) -> None:
    if tp_group is not None:
        import torch.distributed as dist

        if dist.get_world_size(tp_group) > 1:
            raise NotImplementedError(
                "vocab-parallel log-probs (tp_group with more than one rank) are not part of the "
                "single-GPU build; pass tp_group=None"
            )


_WORK: dict = {}


def _work_words(dev: torch.device) -> torch.Tensor:
    """The work buffer of the steps on the current stream of ``dev`` (AA_STEP_WORK_BYTES, zero between launches; its
    first two words are the row hand-out of the fused kernel): one per (device, stream), kept.  A graph that is being
    captured gets one of its own, cleared by the graph: it may be replayed on any stream, beside eager steps."""
    if torch.cuda.is_current_stream_capturing():
        return torch.zeros(N.STEP_WORK_BYTES // 4, dtype=torch.int32, device=dev)
    key = (dev.index, _stream(dev))
    buf = _WORK.get(key)
    if buf is None:
        buf = _WORK[key] = torch.zeros(N.STEP_WORK_BYTES // 4, dtype=torch.int32, device=dev)
    return buf


def _ppo_params(eps_clip, eps_clip_higher, c_clip, has_w) -> N.PpoParams:
    if c_clip is not None:
        assert c_clip > 1.0, c_clip
    hi = eps_clip if eps_clip_higher is None else eps_clip_higher
    return N.PpoParams(
        clip_lo=1.0 - eps_clip,
        clip_hi=1.0 + hi,
        c_clip=0.0 if c_clip is None else float(c_clip),
        has_c_clip=0 if c_clip is None else 1,
        has_behave_weight=1 if has_w else 0,
    )


# ----------------------------------------------------------------------------
# log-probs / entropy
# ----------------------------------------------------------------------------
class _LogprobsEntropy(torch.autograd.Function):
    """logp, entropy, vocab max, vocab min of each row; differentiable in logits."""

    @staticmethod
    def forward(ctx, logits2d, labels1d, temperature, stride, want_entropy, want_minmax, inplace=False, T_active=None):
        ctx.set_materialize_grads(False)  # no zero-filled gradients for the outputs that have none
        lib = N.load()
        ctx.inplace = bool(inplace)
        T, V = logits2d.shape
        if T_active is not None:  # the rows past it are batch padding: no outputs, a zero gradient
            T = T_active
        dev = logits2d.device
        kw = dict(dtype=torch.float32, device=dev)
        logp = torch.empty(T, **kw)
        entropy = torch.empty(T, **kw) if want_entropy else None
        need_bwd = ctx.needs_input_grad[0]
        row_lse = torch.empty(T, **kw) if need_bwd else None
        row_ez = torch.empty(T, **kw) if (need_bwd and want_entropy) else None
        vmax = torch.empty(T, **kw) if want_minmax else None
        vmin = torch.empty(T, **kw) if want_minmax else None
        with _on(dev):
            N.check(
                lib.aa_logits_fwd(
                    _ptr(logits2d), _DTYPES[logits2d.dtype], T, V, stride, _ptr(labels1d),
                    1.0 / float(temperature), _ptr(logp), _ptr(entropy), _ptr(row_lse), _ptr(row_ez),
                    _ptr(vmax), _ptr(vmin), _stream(dev),
                ),
                "aa_logits_fwd",
            )
        ctx.save_for_backward(logits2d, labels1d, row_lse, row_ez)
        ctx.temperature = float(temperature)
        ctx.stride = stride
        outs = (logp, entropy, vmax, vmin)
        ctx.mark_non_differentiable(*[o for o in (vmax, vmin) if o is not None])
        return outs

    @staticmethod
    def backward(ctx, g_logp, g_entropy, _g_vmax, _g_vmin):
        lib = N.load()
        logits2d, labels1d, row_lse, row_ez = ctx.saved_tensors
        if g_logp is None and g_entropy is None:
            return (None,) * 8
        T, V = logits2d.shape
        dev = logits2d.device
        T_active = row_lse.shape[0]
        g_logp = torch.zeros(T_active, dtype=torch.float32, device=dev) if g_logp is None else _f32_values(g_logp)
        g_entropy = _f32_values(g_entropy) if (g_entropy is not None and row_ez is not None) else None
        if ctx.inplace:
            # the gradient takes the place of the logits (the kernel reads an element before it writes it); the version
            # bump below makes any other operation that kept the logits for its own backward fail loudly
            dlogits = logits2d.detach()
        else:  # the row stride of the input, so that both buffers are walked alike
            dlogits = _empty_rows_like(logits2d, ctx.stride)
        with _on(dev):
            N.check(
                lib.aa_logits_bwd(
                    _ptr(logits2d), _DTYPES[logits2d.dtype], T, V, ctx.stride, _ptr(labels1d),
                    1.0 / ctx.temperature, _ptr(row_lse), _ptr(row_ez), _ptr(g_logp), _ptr(g_entropy),
                    T_active, _ptr(dlogits), _stream(dev),
                ),
                "aa_logits_bwd",
            )
        if ctx.inplace:
            torch.autograd.graph.increment_version(logits2d)
        return (dlogits,) + (None,) * 7


def _device_or_read_back_counts(T: int, T_active: int, mask_u8: torch.Tensor, on_device: bool) -> list[int]:
    """``kept_per_chunk`` of the lm_head step when the caller gave none: left to the device (the kernels stop at the
    rows in use, nothing is read back), or read back from the device (exact counts: one small copy that waits for the
    mask)."""
    chunk = int(N.load().aa_lmhead_chunk_tokens())
    n_chunks = (T + chunk - 1) // chunk
    if on_device:
        return [N.AA_LMHEAD_COUNT_ON_DEVICE] * n_chunks
    on = mask_u8.ne(0)
    if n_chunks * chunk != T_active:
        on = torch.nn.functional.pad(on, (0, n_chunks * chunk - T_active))
    return _HostCounts(on.view(n_chunks, chunk).sum(1)).tolist()


def _logprobs_impl(logits, labels, temperature, tp_group, want_entropy, want_minmax, inplace_backward=False,
                   T_active=None):
    """``T_active`` (2-D logits): only the first rows have outputs (of that length) and a gradient."""
    _check_tp(tp_group)
    _require_gpu(logits, "logits")
    assert logits.shape[0] > 0, "Input logits must have at least one element"
    if tuple(labels.shape) != tuple(logits.shape[:-1]):
        raise ValueError(f"labels shape {tuple(labels.shape)} != logits shape[:-1] {tuple(logits.shape[:-1])}")
    x, T, V, stride = _rows(logits)
    y = _labels_i64(labels, x.device)
    outs = _LogprobsEntropy.apply(x, y if y.dim() == 1 else y.reshape(-1), float(temperature), stride, want_entropy,
                                  want_minmax, bool(inplace_backward), T_active)
    if T_active is not None or labels.dim() == 1:
        return outs
    return tuple(None if t is None else t.view(labels.shape) for t in outs)


def gather_logprobs(
    logits: torch.Tensor,
    labels: torch.Tensor,
    temperature: float = 1.0,
    tp_group: Any | None = None,
    chunk_size: int = 1024,
    inplace_backward: bool = False,
) -> torch.Tensor:
    """``log_softmax(logits.float() / temperature)[..., labels]`` as fp32, shaped like ``labels``.

    Same contract as vocab_parallel.py:401-431.  ``chunk_size`` is accepted and
    ignored: the kernel never materialises an fp32 copy of the logits, and the
    result does not depend on chunking.  ``inplace_backward=True`` (not in the
    reference): the backward pass writes the gradient over the logits instead
    of allocating a second ``[T, V]`` array; for callers that need the logits
    for nothing else after this op.
    """
    del chunk_size
    return _logprobs_impl(logits, labels, temperature, tp_group, False, False, inplace_backward)[0]


def gather_logprobs_entropy(
    logits: torch.Tensor,
    labels: torch.Tensor,
    temperature: float = 1.0,
    tp_group: Any | None = None,
    chunk_size: int = 1024,
    inplace_backward: bool = False,
) -> tuple[torch.Tensor, torch.Tensor]:
    """(log-probs at ``labels``, entropy of each row); vocab_parallel.py:434-469.  ``inplace_backward`` as in
    ``gather_logprobs``."""
    del chunk_size
    logp, entropy, _, _ = _logprobs_impl(logits, labels, temperature, tp_group, True, False, inplace_backward)
    return logp, entropy


def gather_logprobs_entropy_stats(
    logits: torch.Tensor, labels: torch.Tensor, temperature: float = 1.0, inplace_backward: bool = False
) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]:
    """(logp, entropy, vocab_min_logits, vocab_max_logits) from the same single pass.

    The last two are what FSDPEngine._get_vocab_min_max_logits
    (fsdp_engine.py:1893-1906) computes with two more passes over the logits.
    """
    logp, entropy, vmax, vmin = _logprobs_impl(logits, labels, temperature, None, True, True, inplace_backward)
    return logp, entropy, vmin, vmax


# ----------------------------------------------------------------------------
# rejection sampling
# ----------------------------------------------------------------------------
@dataclass
class RejectionSamplingResult:
    """functional.py:152-164"""

    loss_mask: torch.Tensor
    behave_imp_weight: torch.Tensor
    filtered_fraction: float


def _segments(shape, cu_seqlens, what: str):
    """(cu_seqlens int32 tensor or None, number of segments) for a 1-D packed or 2-D padded layout."""
    if len(shape) == 1:
        if cu_seqlens is None:
            raise ValueError(what)
        cu = cu_seqlens.to(dtype=torch.int32).contiguous()
        return cu, cu.shape[0] - 1
    return None, shape[0]


def _rejection_sampling_device(prox, old, mask_u8, shape, cu_seqlens, cfg):
    """Runs the kernel; returns (mask_out u8 [n], weight f32 [n], counts i32 [3]) without syncing."""
    lib = N.load()
    dev = prox.device
    n = prox.numel()
    cu, B = (None, 0)
    if cfg.level == "sequence":
        cu, B = _segments(
            shape, cu_seqlens, "cu_seqlens is required for 1D packed tensors in sequence-level filtering."
        )
        if cu is not None:
            cu = cu.to(dev)
    mask_out = torch.empty(n, dtype=torch.uint8, device=dev)
    w = torch.empty(n, dtype=torch.float32, device=dev)
    counts = torch.empty(3, dtype=torch.int32, device=dev)
    lower = cfg.lower
    with _on(dev):
        N.check(
            lib.aa_rejection_sampling(
                _ptr(prox), _ptr(old), _ptr(mask_u8), n, _ptr(cu), B,
                N.RS_LEVEL[cfg.level], N.RS_ACTION[cfg.action], N.RS_METRIC[cfg.metric], N.RS_AGG[cfg.agg],
                float(cfg.upper), 0.0 if lower is None else float(lower), 0 if lower is None else 1,
                _ptr(mask_out), _ptr(w), _ptr(counts), _stream(dev),
            ),
            "aa_rejection_sampling",
        )
    return mask_out, w, counts


class _HostCounts:
    """The counters of the rejection-sampling kernel on their way to the host.

    The copy into pinned memory is queued right behind the kernel and gets an event of its own, so reading the
    counters later (``filtered_fraction`` is a Python float, as in the reference) waits for that copy only and not
    for the long kernels queued after it: the host keeps running ahead of the GPU.  The wait polls the event: a
    blocking wait took 0.2 ms to wake up here, which a step of a few thousand tokens cannot hide.  After a bounded
    number of polls (some tens of milliseconds) it blocks after all."""

    _POLLS = 20000

    def __init__(self, counts: torch.Tensor):
        self._host = torch.empty(counts.shape, dtype=counts.dtype, pin_memory=True)
        with _on(counts.device):
            self._host.copy_(counts, non_blocking=True)
            self._event = torch.cuda.Event()
            self._event.record()

    def tolist(self):
        event = self._event
        for _ in range(self._POLLS):
            if event.query():
                break
        else:
            event.synchronize()
        return self._host.tolist()


def _validate_rs(cfg) -> None:
    for field, table in (("level", N.RS_LEVEL), ("action", N.RS_ACTION), ("agg", N.RS_AGG)):
        if getattr(cfg, field) not in table:
            raise ValueError(f"Unknown {field}: {getattr(cfg, field)}")
    if cfg.metric not in N.RS_METRIC:
        raise ValueError(f"Unknown metric: {cfg.metric}")


def apply_rejection_sampling(
    proximal_logprobs: torch.Tensor,
    old_logprobs: torch.Tensor,
    loss_mask: torch.Tensor,
    cu_seqlens: torch.Tensor | None,
    config: Any,
) -> RejectionSamplingResult:
    """Filter or clamp tokens / sequences by the divergence between the proximal
    and the behaviour policy; functional.py:185-426.

    ``config`` is any object with the attributes of ``RejectionSamplingConfig``.
    """
    if proximal_logprobs.shape != old_logprobs.shape:
        raise ValueError(
            f"proximal_logprobs shape {proximal_logprobs.shape} != old_logprobs shape {old_logprobs.shape}"
        )
    if proximal_logprobs.shape != loss_mask.shape:
        raise ValueError(
            f"proximal_logprobs shape {proximal_logprobs.shape} != loss_mask shape {loss_mask.shape}"
        )
    if proximal_logprobs.ndim not in (1, 2):
        raise ValueError(f"Expected 1D (packed) or 2D (padded) tensors, got ndim={proximal_logprobs.ndim}")
    _validate_rs(config)
    _require_gpu(proximal_logprobs, "proximal_logprobs")
    shape = proximal_logprobs.shape
    prox = _f32(proximal_logprobs.detach()).reshape(-1)
    old = _f32(old_logprobs.detach()).reshape(-1)
    m8 = _mask_u8(loss_mask).reshape(-1)
    mask_out, w, counts = _rejection_sampling_device(prox, old, m8, shape, cu_seqlens, config)
    total, hit, _ = counts.tolist()  # the reference returns a Python float here too
    if config.action == "mask":
        new_mask = mask_out.view(shape).to(loss_mask.dtype)
    else:
        new_mask = loss_mask
    return RejectionSamplingResult(
        loss_mask=new_mask,
        behave_imp_weight=w.view(shape),
        filtered_fraction=hit / max(total, 1),
    )


# ----------------------------------------------------------------------------
# what the steps share: per-token arrays, loss scale, counters on the host
# ----------------------------------------------------------------------------
class _HostSlot:
    """Four words of pinned host memory that the first kernel of a step writes the counts of the mask to, the tag last.

    Reading them (``filtered_fraction`` is a Python float, as in the reference, and a micro-batch without a token is
    found out on the host) waits for that kernel only, not for the long ones queued after it, and needs no copy and no
    event of its own.  Slots are taken from and given back to a bounded pool (any thread, any stream): the tag tells a
    use from the ones before it.  The memory of a slot that nobody read waits until its kernel has written to it."""

    __slots__ = ("_memory", "_words", "address", "tag", "_device", "_got")
    _pool: deque = deque(maxlen=64)
    _tags = itertools.count(1)
    _unread: deque = deque()  # memory that a kernel may still write to, with the tag that says that it has
    _SPINS = 20000  # about a millisecond, then short sleeps: other threads run

    def __init__(self, device: torch.device):
        if _HostSlot._unread:
            _HostSlot._take_back()
        try:
            self._memory, self._words = _HostSlot._pool.pop()
        except IndexError:
            self._memory = torch.empty(4, dtype=torch.int32, pin_memory=True)
            self._words = (C.c_int32 * 4).from_address(self._memory.data_ptr())
            self._words[3] = 0
        self.address = self._memory.data_ptr()
        self.tag = next(_HostSlot._tags) % 0x7FFFFFFF + 1  # 31 bits, never 0
        self._device = device
        self._got = None

    def read(self) -> tuple[int, int, int]:
        """(non-zero entries of the loss mask, tokens filtered or clamped, end of the last segment if there are any)"""
        if self._got is not None:
            return self._got
        words, tag = self._words, self.tag
        for _ in range(self._SPINS):
            if words[3] == tag:
                break
        else:
            done = None  # an event behind everything queued so far: the counts are there when it has passed
            while words[3] != tag:
                if done is None:
                    done = torch.cuda.Event()
                    done.record(torch.cuda.current_stream(self._device))
                if done.query() and words[3] != tag:
                    raise N.NativeLibraryError("the counts of a step never reached the host")
                time.sleep(2e-5)
        self._got = (words[0], words[1], words[2])
        memory, self._memory = self._memory, None
        _HostSlot._pool.append((memory, words))
        return self._got

    @staticmethod
    def _take_back() -> None:
        """Unread memory that has been written to goes back to the pool.  What a failed launch left behind is never
        written to: past a bound the device is waited for, after which nothing writes to any of it."""
        unread = _HostSlot._unread
        if len(unread) > _HostSlot._pool.maxlen and not torch.cuda.is_current_stream_capturing():
            old = []
            try:
                while len(old) <= 2 * _HostSlot._pool.maxlen:
                    old.append(unread.popleft())
            except IndexError:  # that was all, or another thread takes the rest
                pass
            try:
                for index in {device.index for *_, device in old}:
                    torch.cuda.synchronize(index)
            except RuntimeError:  # (not while another thread captures a graph): kernels may still write to any of it
                unread.extend(old)
            else:
                _HostSlot._pool.extend((memory, words) for memory, words, _, _ in old)
            return
        for _ in range(len(unread)):
            try:
                entry = unread.popleft()
            except IndexError:  # another thread was faster
                return
            memory, words, tag, _ = entry
            if words[3] == tag:
                _HostSlot._pool.append((memory, words))
            else:
                unread.append(entry)

    def __del__(self):
        if getattr(self, "_memory", None) is not None:
            _HostSlot._unread.append((self._memory, self._words, self.tag, self._device))


class _PerValidToken:
    """Loss scale ``loss_mask.count_nonzero() / total * multiplier`` (fsdp_engine.py:1983-1985, 2045), formed inside the
    kernels from the count they have anyway.  ``total`` is a number or a tensor with one element."""

    __slots__ = ("total", "multiplier", "valid_tokens")

    def __init__(self, total, multiplier: float):
        self.total, self.multiplier = total, multiplier
        self.valid_tokens = None  # the count, once a step that was given this scale has it on the host


def _note_valid_tokens(scale, step) -> None:
    if isinstance(scale, _PerValidToken):
        # the count on the host is that of the tokens inside the sequences; without any, the mask itself is asked
        scale.valid_tokens = step.slot.read()[0] or int(step.mask.count_nonzero())


def _scale_struct(scale, dev: torch.device):
    """(``aa_loss_scale``, tensors it points into)"""
    if scale is None:
        return N.LossScale(None, None, 1.0, 1.0, 0), None
    if isinstance(scale, _PerValidToken):
        total = scale.total
        if isinstance(total, torch.Tensor) and total.is_cuda:
            total = total.detach().to(device=dev, dtype=torch.float32).reshape(1)
            return N.LossScale(None, total.data_ptr(), float(scale.multiplier), 1.0, 1), total
        return N.LossScale(None, None, float(scale.multiplier), float(total), 1), None
    if isinstance(scale, torch.Tensor) and scale.is_cuda:
        factor = scale.detach().to(device=dev, dtype=torch.float32).reshape(1)
        return N.LossScale(factor.data_ptr(), None, 1.0, 1.0, 0), factor
    return N.LossScale(None, None, float(scale), 1.0, 0), None


_NO_RS = N.RsParams()


def _rs_struct(cfg) -> N.RsParams:
    if cfg is None:
        return _NO_RS
    _validate_rs(cfg)
    lower = cfg.lower
    return N.RsParams(1, N.RS_LEVEL[cfg.level], N.RS_ACTION[cfg.action], N.RS_METRIC[cfg.metric], N.RS_AGG[cfg.agg],
                      0 if lower is None else 1, float(cfg.upper), 0.0 if lower is None else float(lower))


class _Step:
    """One micro-batch's per-token arrays and the ``aa_ppo_step`` that describes them to the library.

    The outputs are rows of two arrays (float32 and bytes), so that a step allocates three times and not sixteen; an entry
    of the stat dict that is kept keeps all of them (45 bytes a token, a clone its own four)."""

    __slots__ = ("T", "T_active", "device", "floats", "bools", "loss", "mask", "slot", "struct", "rs", "_keep")

    def __init__(self, dev, T, T_active, mask, prox, old, adv, params, rs=None, cu=None, n_segments=0, scale=None,
                 derived=True, host_counts=False, behave_w=None, counts=None):
        self.T, self.T_active, self.device, self.rs, self.mask = T, T_active, dev, rs, mask
        work = _work_words(dev)
        scale_c, scale_t = _scale_struct(scale, dev)
        self.slot = _HostSlot(dev) if (rs is not None or host_counts or isinstance(scale, _PerValidToken)) else None
        c = self.struct = N.PpoStep()
        c.params, c.rs, c.scale = params, _rs_struct(rs), scale_c
        if self.slot is not None:
            c.host_counts, c.host_tag = self.slot.address, self.slot.tag
        self.floats, self.bools, self.loss = N.host().make_step(
            C.addressof(c), T, T_active, mask, prox, old, adv, cu, n_segments, derived, rs is not None, behave_w, counts, work, dev)
        self._keep = (prox, old, adv, mask, cu, scale_t, behave_w, counts, work)

    @property
    def counts_address(self) -> int:
        """Where the device has the number of tokens with a loss (an int32)."""
        return self.struct.counts

    def rows(self) -> list:
        """logp, entropy, vmax, vmin, stat_loss, ratio: ``[T_active]`` each."""
        return N.host().step_rows(self.floats, self.T_active)

    def stats(self, rows: bool, shape=None) -> dict:
        """The stat dict of ``ppo_actor_loss_fn`` (functional.py:505-558); ``rows``: with the per-row outputs as well."""
        stat = N.host().step_stats(self.floats, self.bools, self.T_active, rows, self.rs is not None)
        if shape is not None and len(shape) != 1:
            stat = {k: v.view(shape) for k, v in stat.items()}
        return stat

    def finish(self, stat: dict) -> dict:
        """Adds what has to be waited for: with rejection sampling the share of the tokens it hit."""
        if self.rs is not None:
            total, hit, _ = self.slot.read()
            stat["filtered_fraction"] = hit / max(total, 1)
        return stat


# ----------------------------------------------------------------------------
# PPO actor loss on log-probs
# ----------------------------------------------------------------------------
class _PpoLoss(torch.autograd.Function):
    @staticmethod
    def forward(ctx, logp, step, seq_level):
        dev = step.device
        g_logp = torch.empty_like(logp)
        with _on(dev):
            N.check(N.load().aa_ppo_loss_step(step.struct, _ptr(logp), 1 if seq_level else 0, 0, _ptr(g_logp), _stream(dev)),
                    "aa_ppo_loss_step")
        ctx.save_for_backward(g_logp)
        return step.loss

    @staticmethod
    def backward(ctx, g_loss):
        (g_logp,) = ctx.saved_tensors
        return g_logp * g_loss, None, None


def _count_nonzero(mask_u8: torch.Tensor) -> torch.Tensor:
    lib = N.load()
    dev = mask_u8.device
    out = torch.empty(1, dtype=torch.int32, device=dev)
    with _on(dev):
        N.check(lib.aa_count_nonzero_u8(_ptr(mask_u8), mask_u8.numel(), _ptr(out), _stream(dev)), "aa_count_nonzero_u8")
    return out


def _rs_stats(stat, behave_mask, behave_kl, w, counts, shape):
    total, hit, _ = counts.tolist()
    stat.update(
        behave_approx_kl=behave_kl.view(shape),
        behave_imp_weight=w.view(shape),
        behave_mask=behave_mask.view(shape),
        filtered_fraction=hit / max(total, 1),
    )


def ppo_actor_loss_fn(
    logprobs: torch.Tensor,
    proximal_logprobs: torch.Tensor,
    old_logprobs: torch.Tensor,
    advantages: torch.Tensor,
    eps_clip: float,
    loss_mask: torch.Tensor,
    eps_clip_higher: float | None = None,
    c_clip: float | None = None,
    rejection_sampling: Any | None = None,
    importance_sampling_level: str = "token",
    cu_seqlens: torch.Tensor | None = None,
) -> tuple[torch.Tensor, dict]:
    """Decoupled-proximal clipped PPO actor loss; functional.py:429-559.

    Returns ``(loss, stat)`` with the reference's stat keys: ``loss``,
    ``importance_weight``, ``approx_kl``, ``clip_mask``, ``dual_clip_mask`` and,
    with rejection sampling, ``behave_approx_kl``, ``behave_imp_weight``,
    ``behave_mask``, ``filtered_fraction``.  The loss is differentiable in
    ``logprobs`` (closed-form gradient computed with the forward).
    """
    loss, stat, step = _ppo_actor_loss(logprobs, proximal_logprobs, old_logprobs, advantages, eps_clip, loss_mask,
                                       eps_clip_higher, c_clip, rejection_sampling, importance_sampling_level, cu_seqlens)
    return loss, step.finish(stat)


def _ppo_actor_loss(logprobs, proximal_logprobs, old_logprobs, advantages, eps_clip, loss_mask, eps_clip_higher=None,
                    c_clip=None, rejection_sampling=None, importance_sampling_level="token", cu_seqlens=None,
                    host_counts=False):
    """``ppo_actor_loss_fn`` without its wait: the caller finishes the stat dict (``_Step.finish``) when it has queued
    what else it has.  ``host_counts``: the counts come to the host (``step.slot``) also without rejection sampling, and
    with them the end of the last sequence of a packed batch."""
    if importance_sampling_level not in ("token", "sequence"):
        raise ValueError(
            f"Invalid importance_sampling_level: {importance_sampling_level}. Must be 'token' or 'sequence'."
        )
    _require_gpu(logprobs, "logprobs")
    shape = logprobs.shape
    seq_level = importance_sampling_level == "sequence"
    rs = rejection_sampling
    cu, B = None, 0
    if seq_level:
        cu, B = _segments(
            shape,
            cu_seqlens,
            "cu_seqlens is required for 1D tensors (packed format). For a single sequence, use "
            "cu_seqlens=torch.tensor([0, seq_len], dtype=torch.int32).",
        )
    params = _ppo_params(eps_clip, eps_clip_higher, c_clip, rs is not None)
    if rs is not None:
        _validate_rs(rs)
        if rs.level == "sequence" and not seq_level:
            cu, B = _segments(shape, cu_seqlens,
                              "cu_seqlens is required for 1D packed tensors in sequence-level filtering.")
    dev = logprobs.device
    if cu is None and host_counts and cu_seqlens is not None and cu_seqlens.numel() > 0 and len(shape) == 1:
        cu, B = _segments(shape, cu_seqlens, "")
    if cu is not None:
        cu = cu.to(dev)
    lp = logprobs if logprobs.dtype is torch.float32 and logprobs.is_contiguous() else _f32(logprobs)
    if lp.dim() != 1:
        lp = lp.reshape(-1)
    n = lp.numel()
    step = _Step(dev, n, n, _mask_bytes(loss_mask), _f32_values(proximal_logprobs), _f32_values(old_logprobs),
                 _f32_values(advantages), params, rs, cu, B, host_counts=host_counts)
    loss = _PpoLoss.apply(lp, step, seq_level)
    return loss, step.stats(rows=False, shape=shape), step


# ----------------------------------------------------------------------------
# fused: logits -> logp/entropy -> token-level PPO loss -> d(logits), one pass
# ----------------------------------------------------------------------------
def _hand_out_once(ctx) -> None:
    """The fused steps keep their gradients in the buffers the forward pass wrote and scale them in place by the
    upstream factor, so those buffers can be handed out once: a second backward through a retained graph would scale
    them again."""
    if getattr(ctx, "handed_out", False):
        raise RuntimeError("the gradient of this fused step was already handed out; run the forward pass again "
                           "instead of a second backward through a retained graph")
    ctx.handed_out = True


def _fused_logits(logits2d, step, labels1d, stride, temperature, inplace):
    """The loss of the step on logits, differentiable in them; its per-token outputs are in ``step``."""
    return N.host().fused_logits(logits2d, C.addressof(step.struct), step.loss, labels1d, stride, 1.0 / temperature, inplace)


def _scaled(loss, scale, loss_mask):
    """``loss`` times a loss scale, for the paths that form the loss with torch."""
    if scale is None:
        return loss
    if isinstance(scale, _PerValidToken):
        return loss * (loss_mask.count_nonzero() / scale.total * scale.multiplier)
    return loss * torch.as_tensor(scale, dtype=torch.float32, device=loss.device).reshape(())


def _ppo_step(dev, T, T_active, loss_mask, prox, old, adv, eps_clip, eps_clip_higher, c_clip, rs, cu_seqlens, loss_scale):
    """The ``_Step`` of a token-level PPO loss on a packed micro-batch."""
    params = _ppo_params(eps_clip, eps_clip_higher, c_clip, rs is not None)
    cu, B = None, 0
    if rs is not None:
        _validate_rs(rs)
        if rs.level == "sequence":
            cu, B = _segments(loss_mask.shape, cu_seqlens,
                              "cu_seqlens is required for 1D packed tensors in sequence-level filtering.")
            cu = cu.to(dev)
    return _Step(dev, T, T_active, _mask_bytes(loss_mask), _f32_values(prox), _f32_values(old), _f32_values(adv), params,
                 rs, cu, B, loss_scale)


def fused_logprobs_ppo_loss(
    logits: torch.Tensor,
    labels: torch.Tensor,
    proximal_logprobs: torch.Tensor,
    old_logprobs: torch.Tensor,
    advantages: torch.Tensor,
    eps_clip: float,
    loss_mask: torch.Tensor,
    eps_clip_higher: float | None = None,
    c_clip: float | None = None,
    rejection_sampling: Any | None = None,
    importance_sampling_level: str = "token",
    cu_seqlens: torch.Tensor | None = None,
    temperature: float = 1.0,
    loss_scale: torch.Tensor | float | None = None,
    inplace_backward: bool = False,
) -> tuple[torch.Tensor, dict]:
    """``gather_logprobs_entropy`` + ``ppo_actor_loss_fn`` (+ backward) in one pass over the logits.

    ``logits`` is ``[T_pad, V]`` and ``labels`` ``[T_pad]`` (the batch-padded
    micro-batch, fsdp_engine.py:1908-1936); the per-token tensors are the
    un-padded ``[T]`` ones with ``T <= T_pad``: rows past ``T`` are the padding
    the engine trims after the log-prob op (fsdp_engine.py:2027-2031) and get a
    zero gradient.  ``loss_scale`` is the factor the engine multiplies the loss
    with (fsdp_engine.py:2045); the returned loss already includes it, and
    ``loss.backward()`` hands back a gradient that was written during the
    forward pass.

    The stat dict has the keys of ``ppo_actor_loss_fn`` plus ``logprobs``,
    ``entropy``, ``vocab_min_logits`` and ``vocab_max_logits`` (all ``[T]``).
    With ``importance_sampling_level="sequence"`` the loss of a token depends on
    its whole sequence, so the call runs the unfused kernels instead.

    ``inplace_backward=True`` (no counterpart in the reference, whose autograd
    allocates the gradient) writes the gradient over the logits instead of into
    a second ``[T_pad, V]`` array: half the memory of the step (37 GB instead of
    74 GB at 122 k tokens of a 152 k vocabulary) and the same bits.  After the
    call ``logits`` holds its own gradient (for an upstream factor of 1), so it
    is for callers that need the logits for nothing else; an operation that
    saved them for its backward raises autograd's modified-in-place error.
    On the sequence-level path the gradient lands there during
    ``loss.backward()``.  Ignored where no gradient is produced.

    fp32 logits of more than 114 688 entries per row (``V % 8 == 0``) are kept
    on the chip in 24 bits per value between their one read and the write of
    the gradient: log-probs, entropy and the extrema come from the fp32 values,
    the entries of the gradient row are within ``|x| / temperature * 2**-16``
    (relative) of the fp32 ones.
    """
    if importance_sampling_level not in ("token", "sequence"):
        raise ValueError(
            f"Invalid importance_sampling_level: {importance_sampling_level}. Must be 'token' or 'sequence'."
        )
    _require_gpu(logits, "logits")
    if logits.ndim != 2 or labels.ndim != 1 or labels.shape[0] != logits.shape[0]:
        raise ValueError(f"expected logits [T, V] and labels [T], got {tuple(logits.shape)} and {tuple(labels.shape)}")
    assert logits.shape[0] > 0, "Input logits must have at least one element"
    T_active = loss_mask.shape[0]
    if loss_mask.ndim != 1 or T_active > logits.shape[0]:
        raise ValueError(f"loss_mask shape {tuple(loss_mask.shape)} does not fit logits {tuple(logits.shape)}")
    for name, t in (("proximal_logprobs", proximal_logprobs), ("old_logprobs", old_logprobs), ("advantages", advantages)):
        if t.shape != loss_mask.shape:
            raise ValueError(f"{name} shape {tuple(t.shape)} != loss_mask shape {tuple(loss_mask.shape)}")
    dev = logits.device
    # Without a gradient to produce (evaluation, torch.no_grad) the step is the forward kernel (one read of the logits,
    # no [T, V] gradient buffer) followed by the loss on log-probs.
    forward_only = not (torch.is_grad_enabled() and logits.requires_grad)
    if importance_sampling_level == "sequence" or forward_only:
        logp, entropy, vmin, vmax = gather_logprobs_entropy_stats(logits, labels, temperature,
                                                                  inplace_backward and not forward_only)
        logp, entropy, vmin, vmax = (t[:T_active] for t in (logp, entropy, vmin, vmax))
        loss, stat = ppo_actor_loss_fn(
            logp, proximal_logprobs, old_logprobs, advantages, eps_clip, loss_mask, eps_clip_higher, c_clip,
            rejection_sampling, importance_sampling_level, cu_seqlens,
        )
        loss = _scaled(loss, loss_scale, loss_mask)
        stat.update(logprobs=logp.detach(), entropy=entropy.detach(), vocab_min_logits=vmin, vocab_max_logits=vmax)
        return loss, stat

    x, T, V, stride = _rows(logits)
    step = _ppo_step(dev, T, T_active, loss_mask, proximal_logprobs, old_logprobs, advantages, eps_clip, eps_clip_higher,
                     c_clip, rejection_sampling, cu_seqlens, loss_scale)
    loss = _fused_logits(x, step, _labels_i64(labels, dev), stride, float(temperature), bool(inplace_backward))
    stat = step.finish(step.stats(rows=True))
    _note_valid_tokens(loss_scale, step)
    return loss, stat


# ----------------------------------------------------------------------------
# fused lm_head: hidden @ weight.T -> logp / entropy without the [T, V] logits
# ----------------------------------------------------------------------------
_LMHEAD_BACKWARD = {"recompute": 0, "carry": 1}  # aa_lmhead_backward_mode


def lm_head_chunk_tokens() -> int:
    """Tokens per chunk of the lm_head entry points (what ``kept_per_chunk`` counts over)."""
    return int(N.load().aa_lmhead_chunk_tokens())


def _lmhead_workspace(T: int, H: int, V: int, dev, forward_only: bool = False, extrema: bool = False) -> torch.Tensor:
    lib = N.load()
    if forward_only:
        n = lib.aa_lmhead_fwd_stats_workspace_bytes(T, H, V) if extrema else lib.aa_lmhead_fwd_workspace_bytes(T, H, V)
    else:
        n = lib.aa_lmhead_workspace_bytes(T, H, V)
    if n < 0:
        raise N.NativeLibraryError(
            f"the lm_head path needs a hidden size that is a multiple of 8, and sizes below 2^22 (got H={H}, V={V})"
        )
    return torch.empty(n, dtype=torch.uint8, device=dev)


class _LmHeadLogprobsEntropy(torch.autograd.Function):
    @staticmethod
    def forward(ctx, hidden, weight, labels, temperature, want_minmax, T):
        ctx.set_materialize_grads(False)
        lib = N.load()
        H = hidden.shape[1]
        V = weight.shape[0]
        dev = hidden.device
        f32 = dict(dtype=torch.float32, device=dev)
        logp, entropy, row_lse, row_ez = (torch.empty(T, **f32) for _ in range(4))
        vmax = torch.empty(T, **f32) if want_minmax else None
        vmin = torch.empty(T, **f32) if want_minmax else None
        ws = _lmhead_workspace(T, H, V, dev, forward_only=True, extrema=want_minmax)  # partials only: nothing of size T x V
        with _on(dev):
            N.check(
                lib.aa_lmhead_fwd(
                    _ptr(hidden), _ptr(weight), T, H, V, _ptr(labels), 1.0 / float(temperature), _ptr(logp),
                    _ptr(entropy), _ptr(row_lse), _ptr(row_ez), _ptr(vmax), _ptr(vmin), _ptr(ws), ws.numel(),
                    _stream(dev),
                ),
                "aa_lmhead_fwd",
            )
        ctx.save_for_backward(hidden, weight, labels, row_lse, row_ez)
        ctx.temperature = float(temperature)
        if want_minmax:
            ctx.mark_non_differentiable(vmax, vmin)
        return logp, entropy, vmax, vmin

    @staticmethod
    def backward(ctx, g_logp, g_entropy, _g_vmax=None, _g_vmin=None):
        if g_logp is None and g_entropy is None:
            return (None,) * 6
        hidden, weight, labels, row_lse, row_ez = ctx.saved_tensors
        d_hidden, d_weight = _lmhead_recompute_backward(hidden, weight, labels, ctx.temperature, row_lse, row_ez,
                                                        g_logp, g_entropy)
        return (d_hidden, d_weight) + (None,) * 4


def _lmhead_recompute_backward(hidden, weight, labels, temperature, row_lse, row_ez, g_logp, g_entropy):
    """``aa_lmhead_bwd``: the logits tiles of the tokens with a gradient are formed again."""
    lib = N.load()
    T, H = row_lse.shape[0], hidden.shape[1]  # the rows past T are batch padding
    V = weight.shape[0]
    dev = hidden.device
    g_logp = torch.zeros(T, dtype=torch.float32, device=dev) if g_logp is None else _f32(g_logp)
    g_entropy = None if g_entropy is None else _f32(g_entropy)
    d_hidden = _empty_hidden_gradient(hidden, T)
    d_weight = torch.empty_like(weight)  # bf16: rounded once, after fp32 accumulation over the chunks
    ws = _lmhead_workspace(T, H, V, dev)
    # Rows whose upstream gradients are all zero (masked tokens) are left out of the gradient GEMMs; the device counts
    # them itself (no read-back: the host does not wait for the gradient to exist).
    has_grad = g_logp != 0 if g_entropy is None else (g_logp != 0) | (g_entropy != 0)
    chunk = int(lib.aa_lmhead_chunk_tokens())
    n_chunks = (T + chunk - 1) // chunk
    kept = (C.c_int64 * n_chunks)(*([N.AA_LMHEAD_COUNT_ON_DEVICE] * n_chunks))
    with _on(dev):
        N.check(
            lib.aa_lmhead_bwd(
                _ptr(hidden), _ptr(weight), T, H, V, _ptr(labels), 1.0 / temperature, _ptr(row_lse),
                _ptr(row_ez), _ptr(g_logp), _ptr(g_entropy), _ptr(has_grad.view(torch.uint8)), kept,
                _ptr(d_hidden), _ptr(d_weight), _DTYPES[d_weight.dtype], _ptr(ws), ws.numel(), _stream(dev),
            ),
            "aa_lmhead_bwd",
        )
    return d_hidden, d_weight


class _LmHeadCarry(torch.autograd.Function):
    """The lm_head op whose forward also keeps ``p_v / p_label`` of the tokens that may get a gradient (bf16 rows, in a
    tensor that lives until the backward), so that the backward is two plain GEMMs (``aa_lmhead_fwd_carry`` /
    ``aa_lmhead_bwd_carry``)."""

    @staticmethod
    def forward(ctx, hidden, weight, labels, temperature, grad_mask, kept_per_chunk, want_minmax, T):
        ctx.set_materialize_grads(False)
        lib = N.load()
        H = hidden.shape[1]
        V = weight.shape[0]
        dev = hidden.device
        f32 = dict(dtype=torch.float32, device=dev)
        logp, entropy, row_lse, row_ez = (torch.empty(T, **f32) for _ in range(4))
        vmax = torch.empty(T, **f32) if want_minmax else None
        vmin = torch.empty(T, **f32) if want_minmax else None
        kept = None if kept_per_chunk is None else (C.c_int64 * len(kept_per_chunk))(*kept_per_chunk)
        if kept_per_chunk is None:
            rows = T
        else:  # a chunk whose count stays on the device keeps room for every one of its tokens
            chunk = lm_head_chunk_tokens()
            rows = sum(min(chunk, T - i * chunk) if k == N.AA_LMHEAD_COUNT_ON_DEVICE else k
                       for i, k in enumerate(kept_per_chunk))
        panel = torch.empty(max(rows, 1), int(lib.aa_lmhead_panel_pitch(V)), dtype=torch.bfloat16, device=dev)
        n = lib.aa_lmhead_carry_workspace_bytes(T, H, V)
        if n < 0:
            raise N.NativeLibraryError(
                f"the lm_head path needs a hidden size that is a multiple of 8, and sizes below 2^22 (got H={H}, V={V})")
        ws = torch.empty(n, dtype=torch.uint8, device=dev)
        with _on(dev):
            N.check(
                lib.aa_lmhead_fwd_carry(
                    _ptr(hidden), _ptr(weight), T, H, V, _ptr(labels), 1.0 / float(temperature), _ptr(grad_mask), kept,
                    _ptr(logp), _ptr(entropy), _ptr(row_lse), _ptr(row_ez), _ptr(vmax), _ptr(vmin), _ptr(panel),
                    panel.shape[0], _ptr(ws), ws.numel(), _stream(dev),
                ),
                "aa_lmhead_fwd_carry",
            )
        ctx.save_for_backward(hidden, weight, labels, logp, row_lse, row_ez, panel, grad_mask)
        ctx.temperature = float(temperature)
        ctx.kept_per_chunk = kept_per_chunk
        if want_minmax:
            ctx.mark_non_differentiable(vmax, vmin)
        return logp, entropy, vmax, vmin

    @staticmethod
    def backward(ctx, g_logp, g_entropy, _g_vmax=None, _g_vmin=None):
        if g_logp is None and g_entropy is None:
            return (None,) * 8
        hidden, weight, labels, logp, row_lse, row_ez, panel, grad_mask = ctx.saved_tensors
        if g_entropy is not None:  # an entropy gradient is no multiple of the stored rows: form the logits again
            d_hidden, d_weight = _lmhead_recompute_backward(hidden, weight, labels, ctx.temperature, row_lse, row_ez,
                                                            g_logp, g_entropy)
            return (d_hidden, d_weight) + (None,) * 6
        # the backward patches the stored rows (and may overwrite a chunk of them): they serve one backward
        if getattr(ctx, "handed_out", False):
            raise RuntimeError("the stored rows of this lm_head forward were already used by a backward; run the forward "
                               "pass again instead of a second backward through a retained graph")
        ctx.handed_out = True
        lib = N.load()
        T, H = logp.shape[0], hidden.shape[1]
        V = weight.shape[0]
        dev = hidden.device
        g_logp = _f32(g_logp)
        kept_per_chunk = ctx.kept_per_chunk
        kept = None if kept_per_chunk is None else (C.c_int64 * len(kept_per_chunk))(*kept_per_chunk)
        d_hidden = _empty_hidden_gradient(hidden, T)
        d_weight = torch.empty_like(weight)
        ws = torch.empty(lib.aa_lmhead_carry_workspace_bytes(T, H, V), dtype=torch.uint8, device=dev)
        with _on(dev):
            N.check(
                lib.aa_lmhead_bwd_carry(
                    _ptr(hidden), _ptr(weight), T, H, V, _ptr(labels), 1.0 / ctx.temperature, _ptr(logp), _ptr(row_lse),
                    _ptr(g_logp), _ptr(grad_mask), kept, _ptr(panel), panel.shape[0], _ptr(d_hidden), _ptr(d_weight),
                    _DTYPES[d_weight.dtype], _ptr(ws), ws.numel(), _stream(dev),
                ),
                "aa_lmhead_bwd_carry",
            )
        return (d_hidden, d_weight) + (None,) * 6


def lm_head_logprobs_entropy(
    hidden: torch.Tensor, weight: torch.Tensor, labels: torch.Tensor, temperature: float = 1.0,
    token_mask: torch.Tensor | None = None, backward: str = "recompute", grad_token_mask: torch.Tensor | None = None,
    kept_per_chunk: list[int] | None = None, count_on_device: bool = False,
) -> tuple[torch.Tensor, torch.Tensor]:
    """``gather_logprobs_entropy(hidden @ weight.T, labels, temperature)`` without writing the ``[T, V]`` logits.
    Any vocabulary size; the hidden size has to be a multiple of 8.

    ``hidden`` is ``[T, H]`` and ``weight`` ``[V, H]`` (the lm_head), both bf16.  The forward forms 256 x 256 tiles of
    the logits in the accumulator registers of the library's bf16 MFMA tile GEMM (fp32 accumulation, not rounded to
    bf16 in between) and reduces each tile to softmax partials per token in the GEMM's epilogue; its only scratch
    memory is those partials (about ``24 * V / 256`` bytes per token of a chunk of at most 16384 tokens, 0.23 GB at
    ``V = 151936``).  Differentiable in ``hidden`` and ``weight``: the backward goes through the tokens in chunks of at
    most 16384, forms the chunk's logits tiles again, writes their gradient as bf16 rows (of the tokens whose upstream
    gradient is not zero) into a workspace panel ``[chunk, V]`` and contracts that panel with the weight and with the
    hidden states on the same tile GEMM (fp32 accumulation, the weight gradient is returned in the dtype of
    ``weight``).  The backward's workspace is that panel (``2 * chunk * V`` bytes), the hidden rows of the chunk's
    tokens with a gradient and a few fp32 planes of ``[chunk, H]``; the arrays are multiplied as they lie, nothing is
    transposed.
    The reference has no such op: it is the drop-in for its lm_head matmul followed by
    ``gather_logprobs_entropy`` (vocab_parallel.py:434-469).

    ``token_mask`` (``[T]``, optional, beyond the reference's semantics): only tokens whose entry is non-zero go
    through the lm_head; the others get log-prob 0 and entropy 0 (e.g. the forward-only ``compute_logp`` pass, whose
    results are multiplied by the loss mask anyway).

    ``backward="carry"`` (default ``"recompute"``): the forward also keeps ``p_v / p_label`` of the tokens that may get
    a gradient as bf16 rows until the backward, which is then two plain GEMMs instead of three (no second logits GEMM:
    about a fifth less time for forward + backward at the 8B shape).  For losses that need every log-prob before any
    gradient exists (sequence-level importance ratios, SAPO, anything custom).  The price is memory between the two
    passes: 2 bytes x V per such token.  ``grad_token_mask`` (``[T]``, e.g. the loss mask) names those tokens; tokens
    outside it get NO gradient, whatever the loss says; without it every token is kept.  The number of named tokens per
    chunk of ``lm_head_chunk_tokens()`` tokens sizes the stored rows: it is read back from the device unless the caller
    passes it as ``kept_per_chunk`` (counts that are too large are safe, too small ones drop tokens), or leaves it to
    the device with ``count_on_device=True``: nothing is read back then and the host does not wait, the stored rows
    take the room of every token (2 bytes x V x T) whatever the mask holds, and the kernels stop at the rows in use
    (same results, bit for bit).  A gradient
    with respect to the entropy cannot use the stored rows: such a backward forms the logits again, as ``"recompute"``
    does.  The stored rows serve one backward.
    """
    return _lm_head_impl(hidden, weight, labels, temperature, token_mask, False, backward, grad_token_mask,
                         kept_per_chunk, count_on_device)[:2]


def lm_head_logprobs_entropy_stats(
    hidden: torch.Tensor, weight: torch.Tensor, labels: torch.Tensor, temperature: float = 1.0,
    token_mask: torch.Tensor | None = None, backward: str = "recompute", grad_token_mask: torch.Tensor | None = None,
    kept_per_chunk: list[int] | None = None, count_on_device: bool = False,
) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor, torch.Tensor]:
    """``(logp, entropy, vocab_min_logits, vocab_max_logits)`` of ``hidden @ weight.T`` from the same tiles.

    The last two are what ``FSDPEngine._get_vocab_min_max_logits`` (areal/engine/fsdp_engine.py:1893-1906) reads from
    materialised logits and hands to the loss function; with no logits in memory the caller could not compute them.
    They come from the fp32 sums of the tiles, not from logits rounded to bf16 (the smallest exactly, the largest
    through the softmax exponent, i.e. to one rounding), and carry no gradient.  With ``token_mask`` the tokens left
    out of the lm_head get 0 for both.  The other arguments: see ``lm_head_logprobs_entropy``."""
    return _lm_head_impl(hidden, weight, labels, temperature, token_mask, True, backward, grad_token_mask,
                         kept_per_chunk, count_on_device)


def _lm_head_apply(hidden, weight, y, temperature, want_minmax, backward, grad_mask, kept_per_chunk,
                   count_on_device=False, T_active=None):
    """``T_active``: the rows past it are batch padding, without outputs and with a zero gradient (``grad_mask`` then has
    an entry for each of the others)."""
    needs_grad = torch.is_grad_enabled() and (hidden.requires_grad or weight.requires_grad)
    T = hidden.shape[0] if T_active is None else T_active
    if backward != "carry" or not needs_grad:
        return _LmHeadLogprobsEntropy.apply(hidden, weight, y, float(temperature), want_minmax, T)
    chunk = lm_head_chunk_tokens()
    n_chunks = (T + chunk - 1) // chunk
    m8 = kept = None
    if grad_mask is not None:
        m8 = _mask_bytes(grad_mask)
        if kept_per_chunk is not None:
            kept = [max(0, min(int(v), chunk)) for v in kept_per_chunk]
            if len(kept) != n_chunks:
                if len(kept) != (hidden.shape[0] + chunk - 1) // chunk:
                    raise ValueError(f"kept_per_chunk needs one count per chunk of {chunk} tokens")
                kept = kept[:n_chunks]  # chunks of nothing but padding
        elif count_on_device:
            kept = [N.AA_LMHEAD_COUNT_ON_DEVICE] * n_chunks
        else:
            on = m8.ne(0)
            if n_chunks * chunk != T:
                on = torch.nn.functional.pad(on, (0, n_chunks * chunk - T))
            kept = _HostCounts(on.view(n_chunks, chunk).sum(1)).tolist()
    return _LmHeadCarry.apply(hidden, weight, y, float(temperature), m8, kept, want_minmax, T)


def _empty_hidden_gradient(hidden, T):
    """An array for the gradient of ``hidden`` whose rows past ``T`` (batch padding) are zeros."""
    d_hidden = torch.empty_like(hidden)
    if T != hidden.shape[0]:
        d_hidden[T:].zero_()
    return d_hidden


# Rows that the carried op of compute_lm_head_loss_with may keep room for without knowing how many the mask holds
# (2 bytes x V per token).  Up to here the count stays on the device: reading it back makes the host wait for everything
# queued before, about 60 us in which nothing is queued behind it.  Beyond, the forward alone takes milliseconds and the
# exact size is worth more.
COUNT_ON_DEVICE_BYTES = 2 << 30


def _lm_head_impl(hidden, weight, labels, temperature, token_mask, want_minmax, backward="recompute",
                  grad_token_mask=None, kept_per_chunk=None, count_on_device=False, T_active=None):
    if backward not in _LMHEAD_BACKWARD:
        raise ValueError(f"backward must be one of {sorted(_LMHEAD_BACKWARD)}, got {backward!r}")
    _require_gpu(hidden, "hidden")
    if hidden.ndim != 2 or weight.ndim != 2 or hidden.shape[1] != weight.shape[1]:
        raise ValueError(f"expected hidden [T, H] and weight [V, H], got {tuple(hidden.shape)} and {tuple(weight.shape)}")
    if tuple(labels.shape) != (hidden.shape[0],):
        raise ValueError(f"labels shape {tuple(labels.shape)} != ({hidden.shape[0]},)")
    assert hidden.shape[0] > 0, "Input must have at least one token"
    if hidden.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16:
        raise TypeError("fused lm_head expects bf16 hidden states and weights")
    y = _labels_i64(labels, hidden.device)
    if token_mask is not None:
        if tuple(token_mask.shape) != (hidden.shape[0],):
            raise ValueError(f"token_mask shape {tuple(token_mask.shape)} != ({hidden.shape[0]},)")
        T, dev = hidden.shape[0], hidden.device
        idx = token_mask.to(dev).ne(0).nonzero().squeeze(-1)
        n_kept = idx.numel()
        if n_kept == 0:
            zero = (hidden[:1].float().sum() + weight[:1].float().sum()) * 0.0
            z = torch.zeros(T, dtype=torch.float32, device=dev) if want_minmax else None
            return zero.expand(T), zero.expand(T), z, z
        sub_mask = None if grad_token_mask is None else grad_token_mask.to(dev).reshape(-1).index_select(0, idx)
        lp, ent, vmax, vmin = _lm_head_apply(
            hidden.index_select(0, idx), weight.contiguous(), y.index_select(0, idx), temperature, want_minmax, backward,
            sub_mask, None, count_on_device)   # the caller's counts are per chunk of the whole batch, not of these tokens
        full = lambda v: torch.zeros(T, dtype=torch.float32, device=dev).index_copy(0, idx, v)
        return full(lp), full(ent), (full(vmin) if want_minmax else None), (full(vmax) if want_minmax else None)
    n_rows = hidden.shape[0] if T_active is None else T_active
    if grad_token_mask is not None and tuple(grad_token_mask.shape) != (n_rows,):
        raise ValueError(f"grad_token_mask shape {tuple(grad_token_mask.shape)} != ({n_rows},)")
    lp, ent, vmax, vmin = _lm_head_apply(hidden.contiguous(), weight.contiguous(), y, temperature, want_minmax, backward,
                                         None if grad_token_mask is None else grad_token_mask.to(hidden.device),
                                         kept_per_chunk, count_on_device, T_active)
    return lp, ent, vmin, vmax


def lm_head_logprobs_entropy_static(
    hidden: torch.Tensor, weight: torch.Tensor, labels: torch.Tensor, temperature: float = 1.0,
    out: tuple[torch.Tensor, torch.Tensor] | None = None,
) -> tuple[torch.Tensor, torch.Tensor]:
    """Forward of ``lm_head_logprobs_entropy`` through ``aa_lmhead_fwd_static``: no workspace, nothing allocated by
    the library (its softmax partials live in a 32 MiB device array of its own).  For callers that cannot allocate:
    with ``out = (logp, entropy)`` given (float32 ``[T]``) this function allocates nothing either.  No autograd.
    Calls that overlap on one GPU share that array and race; a vocabulary above ``aa_lmhead_fwd_static_max_vocab()``
    is refused.  The reference has no counterpart."""
    _require_gpu(hidden, "hidden")
    if hidden.ndim != 2 or weight.ndim != 2 or hidden.shape[1] != weight.shape[1]:
        raise ValueError(f"expected hidden [T, H] and weight [V, H], got {tuple(hidden.shape)} and {tuple(weight.shape)}")
    T, H = hidden.shape
    V = weight.shape[0]
    if tuple(labels.shape) != (T,) or labels.dtype != torch.int64 or not labels.is_contiguous():
        raise ValueError("labels must be a contiguous int64 tensor of shape [T]")
    assert T > 0, "Input must have at least one token"
    if hidden.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16:
        raise TypeError("fused lm_head expects bf16 hidden states and weights")
    if not hidden.is_contiguous() or not weight.is_contiguous():
        raise ValueError("hidden and weight must be contiguous")
    lib = N.load()
    if V > lib.aa_lmhead_fwd_static_max_vocab():
        raise ValueError(f"vocabulary {V} is beyond what aa_lmhead_fwd_static takes ({lib.aa_lmhead_fwd_static_max_vocab()})")
    dev = hidden.device
    if out is None:
        out = (torch.empty(T, dtype=torch.float32, device=dev), torch.empty(T, dtype=torch.float32, device=dev))
    logp, entropy = out
    for t in out:
        if t.dtype != torch.float32 or tuple(t.shape) != (T,) or not t.is_contiguous() or t.device != dev:
            raise ValueError("out must hold two contiguous float32 tensors of shape [T] on the device of hidden")
    with _on(dev):
        N.check(
            lib.aa_lmhead_fwd_static(_ptr(hidden), _ptr(weight), T, H, V, _ptr(labels), 1.0 / float(temperature), _ptr(logp),
                                     _ptr(entropy), None, None, _stream(dev)),
            "aa_lmhead_fwd_static",
        )
    return logp, entropy


class _FusedLmHeadPpo(torch.autograd.Function):
    """The step on hidden states; its per-token outputs are in ``step``."""

    @staticmethod
    def forward(ctx, hidden, weight, step, labels, temperature, kept_per_chunk, backward_mode):
        lib = N.load()
        T, H = hidden.shape
        V = weight.shape[0]
        dev = step.device
        # Batch padding has no outputs and a zero gradient: it stays out of the tiles where that makes them fewer (tiles
        # end at multiples of 128 tokens).  4 096 + 56 tokens x 1 536 x 151 936: 4 112 us a step with, 3 999 without the
        # padding; elsewhere clearing its gradient rows in a launch of their own would only cost, about 4 us.
        if 0 < step.T_active and (step.T_active + 127) // 128 < (T + 127) // 128:
            T = step.struct.T = step.T_active
            if kept_per_chunk is not None:
                chunk = lm_head_chunk_tokens()
                kept_per_chunk = kept_per_chunk[: (T + chunk - 1) // chunk]
        kept = None if kept_per_chunk is None else (C.c_int64 * len(kept_per_chunk))(*kept_per_chunk)
        d_hidden = _empty_hidden_gradient(hidden, T)
        d_weight = torch.empty_like(weight)  # bf16: rounded once, after fp32 accumulation over the chunks
        ws = _lmhead_workspace(T, H, V, dev)
        with _on(dev):
            N.check(
                lib.aa_lmhead_ppo_step(
                    step.struct, _ptr(hidden), _ptr(weight), H, V, _ptr(labels), 1.0 / temperature, kept,
                    int(backward_mode), _ptr(d_hidden), _ptr(d_weight), _DTYPES[d_weight.dtype], _ptr(ws), ws.numel(),
                    _stream(dev),
                ),
                "aa_lmhead_ppo_step",
            )
        ctx.save_for_backward(d_hidden, d_weight)
        return step.loss

    @staticmethod
    def backward(ctx, g_loss):
        _hand_out_once(ctx)
        lib = N.load()
        d_hidden, d_weight = ctx.saved_tensors
        dev = d_hidden.device
        g = _f32_values(g_loss)
        with _on(dev):  # both gradients were written with the loss; a factor of 1 is a no-op
            for t in (d_hidden, d_weight):
                N.check(lib.aa_scale_inplace(_ptr(t), _DTYPES[t.dtype], t.numel(), _ptr(g), _stream(dev)),
                        "aa_scale_inplace")
        return (d_hidden, d_weight) + (None,) * 5


def fused_lm_head_ppo_loss(
    hidden: torch.Tensor,
    weight: torch.Tensor,
    labels: torch.Tensor,
    proximal_logprobs: torch.Tensor,
    old_logprobs: torch.Tensor,
    advantages: torch.Tensor,
    eps_clip: float,
    loss_mask: torch.Tensor,
    eps_clip_higher: float | None = None,
    c_clip: float | None = None,
    rejection_sampling: Any | None = None,
    importance_sampling_level: str = "token",
    cu_seqlens: torch.Tensor | None = None,
    temperature: float = 1.0,
    loss_scale: torch.Tensor | float | None = None,
    skip_masked_tokens: bool = True,
    forward_masked_tokens: bool = True,
    kept_per_chunk: list[int] | None = None,
    backward: str = "carry",
    carry_rows_limit_bytes: int = 16 << 30,
    count_on_device: bool = True,
) -> tuple[torch.Tensor, dict]:
    """lm_head + ``gather_logprobs_entropy`` + ``ppo_actor_loss_fn`` (+ backward) for one micro-batch.

    ``hidden`` is ``[T_pad, H]`` (the final hidden states of the batch-padded micro-batch), ``weight`` the ``[V, H]``
    lm_head, both bf16; the other arguments are those of ``fused_logprobs_ppo_loss``.  The logits are formed as
    256 x 256 tiles in the accumulator registers of the library's bf16 MFMA tile GEMM and reduced to softmax partials
    in its epilogue; they are never written to memory.  Tokens are processed in chunks of at most 16384;
    ``loss.backward()`` hands back ``d(hidden)`` and ``d(weight)`` written during the forward pass (the loss is
    known by then).  With ``importance_sampling_level="sequence"`` (GSPO) every log-prob of a sequence is needed before
    any gradient exists, so the call runs ``lm_head_logprobs_entropy`` and the unfused loss; with ``backward="carry"``
    that op keeps the bf16 rows of the tokens with a mask from its forward to its backward (two GEMMs instead of
    three), as long as they take no more than ``carry_rows_limit_bytes`` (2 bytes x V per such token; default 16 GiB),
    and forms the logits again otherwise.

    ``backward`` chooses how the bf16 ``d(loss)/d(logits)`` rows of a chunk (``[tokens with gradient, V]`` in the
    workspace, which the two gradient GEMMs contract) are obtained.  ``"recompute"``: the logits tiles of those tokens
    are formed a second time once the loss is known, as ``lm_head_logprobs_entropy``'s backward does (a third more
    matrix work).  ``"carry"`` (default, the faster of the two by measurement): the forward tiles also write
    ``p_v / p_label`` of those tokens in bf16 into the rows (the label's logit is known before the tiles run); once
    the loss is known the gradient row is that row times one factor per token, which the two gradient GEMMs apply
    themselves, so there is neither a second logits GEMM nor a pass over the rows.  A chunk that holds a token whose
    label has a log-prob below -80, or whose factor is below 2^-100 in magnitude (outside the stored range), is redone
    by recompute, decided on the device.  Both
    modes use the same workspace (``2 * chunk * V`` bytes for the rows).

    ``skip_masked_tokens``: a token whose (effective) loss mask is zero has a zero gradient row, so the two gradient
    GEMMs run on the other tokens only; the results are those of the dense computation.  ``False`` multiplies the
    zero rows through, as the reference's autograd does.  How many tokens of a chunk take part is counted on the
    device (``count_on_device=True``, the default): the kernels are queued for every token that could and stop at
    the rows in use, so the host neither needs the mask nor waits for the device; the results are, bit for bit, those
    of the same counts given by the host, in the same time.  With ``count_on_device=False`` the
    host reads the per-chunk counts back (one small device-to-host copy that waits for the mask only) and sizes the
    GEMMs itself.  A caller that already knows the counts on the host (the number of tokens with a
    non-zero effective mask in each chunk of ``aa_lmhead_chunk_tokens()`` tokens, e.g. from the CPU copy of
    ``loss_mask`` when there is no rejection sampling) can pass them as ``kept_per_chunk``; nothing is read back then
    either.  A count that is too small drops the tokens beyond it from the gradient; a count that is too large (e.g.
    counts of ``loss_mask`` while rejection sampling shrinks the mask on the device) is safe: the surplus rows are
    cleared on the device and add nothing.

    ``stat`` also holds ``vocab_min_logits`` / ``vocab_max_logits`` (what the engine would read from materialised
    logits, areal/engine/fsdp_engine.py:1893-1906), from the fp32 sums of the tiles.

    ``forward_masked_tokens=False`` (token level only) goes one step further than the reference's semantics: tokens
    whose effective mask is zero are not run through the lm_head at all, so their entries of ``stat["logprobs"]``,
    ``stat["entropy"]``, ``stat["loss"]``, ``stat["importance_weight"]`` and ``stat["approx_kl"]`` are zero instead
    of the values the reference computes there (and every consumer masks out).  Loss, gradients and the entries of
    the other tokens are unchanged.
    """
    if importance_sampling_level not in ("token", "sequence"):
        raise ValueError(
            f"Invalid importance_sampling_level: {importance_sampling_level}. Must be 'token' or 'sequence'."
        )
    if backward not in _LMHEAD_BACKWARD:
        raise ValueError(f"backward must be one of {sorted(_LMHEAD_BACKWARD)}, got {backward!r}")
    _require_gpu(hidden, "hidden")
    if hidden.ndim != 2 or weight.ndim != 2 or hidden.shape[1] != weight.shape[1]:
        raise ValueError(f"expected hidden [T, H] and weight [V, H], got {tuple(hidden.shape)} and {tuple(weight.shape)}")
    if tuple(labels.shape) != (hidden.shape[0],):
        raise ValueError(f"labels shape {tuple(labels.shape)} != ({hidden.shape[0]},)")
    assert hidden.shape[0] > 0, "Input must have at least one token"
    if hidden.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16:
        raise TypeError("fused lm_head expects bf16 hidden states and weights")
    T_active = loss_mask.shape[0]
    if loss_mask.ndim != 1 or T_active > hidden.shape[0]:
        raise ValueError(f"loss_mask shape {tuple(loss_mask.shape)} does not fit hidden {tuple(hidden.shape)}")
    for name, t in (("proximal_logprobs", proximal_logprobs), ("old_logprobs", old_logprobs), ("advantages", advantages)):
        if t.shape != loss_mask.shape:
            raise ValueError(f"{name} shape {tuple(t.shape)} != loss_mask shape {tuple(loss_mask.shape)}")
    dev = hidden.device
    y = _labels_i64(labels, dev)

    forward_only = not (torch.is_grad_enabled() and (hidden.requires_grad or weight.requires_grad))
    if importance_sampling_level == "sequence" or forward_only:
        # forward-only: forward GEMM + loss.  Sequence level: every log-prob of a sequence is needed before any gradient
        # exists, so the op and the loss run one after the other; in carry mode the op keeps the rows of the tokens with
        # a mask for its backward (2 bytes x V per such token until then) unless that is more than the caller allows
        grad_mask = kept_seq = None
        op_backward = "recompute"
        if not forward_only and backward == "carry":
            pad = hidden.shape[0] - T_active
            grad_mask = loss_mask.to(dev).reshape(-1).ne(0)
            if pad:
                grad_mask = torch.nn.functional.pad(grad_mask, (0, pad))
            if kept_per_chunk is not None:
                kept_seq = [int(v) for v in kept_per_chunk]
            rows_bound = sum(kept_seq) if kept_seq is not None else hidden.shape[0]
            if 2 * rows_bound * weight.shape[0] <= carry_rows_limit_bytes:
                op_backward = "carry"
        logp, entropy, vmin, vmax = lm_head_logprobs_entropy_stats(
            hidden, weight, y, temperature, backward=op_backward,
            grad_token_mask=grad_mask if op_backward == "carry" else None,
            kept_per_chunk=kept_seq if op_backward == "carry" else None,
            count_on_device=count_on_device)
        logp, entropy = logp[:T_active], entropy[:T_active]
        loss, stat = ppo_actor_loss_fn(
            logp, proximal_logprobs, old_logprobs, advantages, eps_clip, loss_mask, eps_clip_higher, c_clip,
            rejection_sampling, importance_sampling_level, cu_seqlens,
        )
        loss = _scaled(loss, loss_scale, loss_mask)
        stat.update(logprobs=logp.detach(), entropy=entropy.detach(), vocab_min_logits=vmin[:T_active],
                    vocab_max_logits=vmax[:T_active])
        return loss, stat

    rs = rejection_sampling
    if not forward_masked_tokens:
        prox, old, adv = (_f32(t.detach()) for t in (proximal_logprobs, old_logprobs, advantages))
        m8 = _mask_u8(loss_mask)
        params = _ppo_params(eps_clip, eps_clip_higher, c_clip, rs is not None)
        w, mask_eff = None, m8
        if rs is not None:
            _validate_rs(rs)
            mask_eff, w, n_valid = _rejection_sampling_device(prox, old, m8, loss_mask.shape, cu_seqlens, rs)
            host_counts = _HostCounts(n_valid)
            if rs.action != "mask":
                mask_eff = m8
        else:
            n_valid = _count_nonzero(m8)
        # only the tokens with a mask go through the lm_head: gather them (autograd scatters d(hidden) back), run the
        # step on the closed-up batch with an all-true mask, and put the per-token results back at their tokens
        idx = mask_eff.nonzero().squeeze(-1)
        n_kept = idx.numel()
        full = lambda v, dtype=torch.float32: torch.zeros(T_active, dtype=dtype, device=dev).index_copy_(0, idx, v)
        if n_kept == 0:
            loss = (hidden[:1].float().sum() + weight[:1].float().sum()) * 0.0
            z = torch.zeros(T_active, dtype=torch.float32, device=dev)
            zb = torch.zeros(T_active, dtype=torch.bool, device=dev)
            stat = dict(loss=z, importance_weight=z.clone(), approx_kl=z.clone(), clip_mask=zb, dual_clip_mask=zb.clone(),
                        logprobs=z.clone(), entropy=z.clone(), vocab_min_logits=z.clone(), vocab_max_logits=z.clone())
        else:
            ones = torch.ones(n_kept, dtype=torch.uint8, device=dev)
            chunk = int(N.load().aa_lmhead_chunk_tokens())
            kept = [max(0, min(chunk, n_kept - c)) for c in range(0, n_kept, chunk)]
            step = _Step(dev, n_kept, n_kept, ones, prox.index_select(0, idx), None, adv.index_select(0, idx), params,
                         scale=loss_scale, behave_w=None if w is None else w.index_select(0, idx), counts=n_valid)
            loss = _FusedLmHeadPpo.apply(hidden.index_select(0, idx), weight.contiguous(), step, y.index_select(0, idx),
                                         float(temperature), kept, _LMHEAD_BACKWARD[backward])
            kept_stat = step.stats(rows=True)
            stat = {k: full(v, v.dtype) for k, v in kept_stat.items()}
        if rejection_sampling is not None:
            behave_mask = (w > 0) & mask_eff.bool()
            _rs_stats(stat, behave_mask, torch.where(behave_mask, prox - old, 0.0), w, host_counts, loss_mask.shape)
        return loss, stat
    T = hidden.shape[0]
    step = _ppo_step(dev, T, T_active, loss_mask, proximal_logprobs, old_logprobs, advantages, eps_clip, eps_clip_higher,
                     c_clip, rs, cu_seqlens, loss_scale)
    kept = None
    if skip_masked_tokens and kept_per_chunk is not None:
        chunk = lm_head_chunk_tokens()
        kept = [int(v) for v in kept_per_chunk]
        if len(kept) != (T + chunk - 1) // chunk:
            raise ValueError(f"kept_per_chunk needs one count per chunk of {chunk} tokens")
    elif skip_masked_tokens and count_on_device:
        kept = [N.AA_LMHEAD_COUNT_ON_DEVICE] * ((T + lm_head_chunk_tokens() - 1) // lm_head_chunk_tokens())
    elif skip_masked_tokens:  # the exact counts are read back: the mask after rejection sampling first
        mask_eff = _mask_u8(loss_mask)
        if rs is not None and rs.action == "mask":
            mask_eff = _rejection_sampling_device(_f32(proximal_logprobs.detach()), _f32(old_logprobs.detach()), mask_eff,
                                                  loss_mask.shape, cu_seqlens, rs)[0]
        kept = _device_or_read_back_counts(T, T_active, mask_eff, False)
    loss = _FusedLmHeadPpo.apply(hidden.contiguous(), weight.contiguous(), step, y, float(temperature), kept,
                                 _LMHEAD_BACKWARD[backward])
    stat = step.finish(step.stats(rows=True))
    _note_valid_tokens(loss_scale, step)
    return loss, stat


# ----------------------------------------------------------------------------
# sibling losses: SAPO, clipped value loss of the critic
# ----------------------------------------------------------------------------
class _SapoLoss(torch.autograd.Function):
    @staticmethod
    def forward(ctx, logp, old, adv, mask, cu, B, seq_level, tau_pos, tau_neg, n_valid):
        lib = N.load()
        dev = logp.device
        n = logp.numel()
        f32 = dict(dtype=torch.float32, device=dev)
        stat_loss, ratio, g_logp = (torch.empty(n, **f32) for _ in range(3))
        gates = torch.empty(3, n, **f32)
        loss = torch.empty((), **f32)
        with _on(dev):
            st = _stream(dev)
            N.check(
                lib.aa_sapo_loss(_ptr(logp), _ptr(old), _ptr(adv), _ptr(mask), n, _ptr(cu), B, 1 if seq_level else 0,
                                 float(tau_pos), float(tau_neg), _ptr(n_valid), _ptr(stat_loss), _ptr(ratio),
                                 _ptr(gates), _ptr(g_logp), st),
                "aa_sapo_loss",
            )
            N.check(lib.aa_masked_sum(_ptr(stat_loss), _ptr(mask), n, _ptr(n_valid), None, _ptr(loss), st),
                    "aa_masked_sum")
        ctx.save_for_backward(g_logp)
        ctx.mark_non_differentiable(stat_loss, ratio, gates)
        return loss, stat_loss, ratio, gates

    @staticmethod
    def backward(ctx, g_loss, *_unused):
        if g_loss is None:  # the loss was not used (gradients are not materialised, see forward)
            return (None,) * 10
        (g_logp,) = ctx.saved_tensors
        return (g_logp * g_loss,) + (None,) * 9


def sapo_loss_fn(
    logprobs: torch.Tensor,
    old_logprobs: torch.Tensor,
    advantages: torch.Tensor,
    tau_pos: float,
    tau_neg: float,
    loss_mask: torch.Tensor,
    importance_sampling_level: str = "token",
    cu_seqlens: torch.Tensor | None = None,
) -> tuple[torch.Tensor, dict]:
    """SAPO loss with asymmetric sigmoid gates; functional.py:562-638, same stat keys."""
    if tau_pos <= 0 or tau_neg <= 0:
        raise ValueError("SAPO temperatures (tau_pos, tau_neg) must be positive.")
    if importance_sampling_level not in ("token", "sequence"):
        raise ValueError(
            f"Invalid importance_sampling_level: {importance_sampling_level}. Must be 'token' or 'sequence'."
        )
    _require_gpu(logprobs, "logprobs")
    shape = logprobs.shape
    seq_level = importance_sampling_level == "sequence"
    cu, B = None, 0
    if seq_level:
        cu, B = _segments(
            shape,
            cu_seqlens,
            "cu_seqlens is required for 1D tensors (packed format). For a single sequence, use "
            "cu_seqlens=torch.tensor([0, seq_len], dtype=torch.int32).",
        )
        if cu is not None:
            cu = cu.to(logprobs.device)
    lp = _f32(logprobs).reshape(-1)
    old = _f32(old_logprobs.detach()).reshape(-1)
    adv = _f32(advantages.detach()).reshape(-1)
    m8 = _mask_u8(loss_mask).reshape(-1)
    n_valid = _count_nonzero(m8)
    loss, stat_loss, ratio, gates = _SapoLoss.apply(lp, old, adv, m8, cu, B, seq_level, tau_pos, tau_neg, n_valid)
    zeros = torch.zeros(shape, dtype=torch.bool, device=lp.device)
    stat = dict(
        loss=stat_loss.view(shape),
        importance_weight=ratio.view(shape),
        approx_kl=(lp.detach() - old).view(shape),
        clip_mask=zeros,
        dual_clip_mask=zeros.clone(),
        sapo_soft_gate=gates[0].view(shape),
        sapo_scaled_gate_pos=gates[1].view(shape),
        sapo_scaled_gate_neg=gates[2].view(shape),
    )
    return loss, stat


class _CriticLoss(torch.autograd.Function):
    @staticmethod
    def forward(ctx, value, old, target, mask, eps, loss_type, n_valid):
        lib = N.load()
        dev = value.device
        n = value.numel()
        f32 = dict(dtype=torch.float32, device=dev)
        stat_loss, g_value = torch.empty(n, **f32), torch.empty(n, **f32)
        clip = torch.empty(n, dtype=torch.uint8, device=dev)
        total = torch.empty((), **f32)
        with _on(dev):
            st = _stream(dev)
            N.check(
                lib.aa_critic_loss(_ptr(value), _ptr(old), _ptr(target), _ptr(mask), n, float(eps), loss_type,
                                   _ptr(n_valid), _ptr(stat_loss), _ptr(clip), _ptr(g_value), st),
                "aa_critic_loss",
            )
            N.check(lib.aa_masked_sum(_ptr(stat_loss), _ptr(mask), n, None, None, _ptr(total), st), "aa_masked_sum")
        loss = total / n_valid[0].to(torch.float32)  # no floor: an empty mask gives NaN, as in the reference
        ctx.save_for_backward(g_value)
        ctx.mark_non_differentiable(stat_loss, clip)
        return loss, stat_loss, clip

    @staticmethod
    def backward(ctx, g_loss, *_unused):
        (g_value,) = ctx.saved_tensors
        return (g_value * g_loss,) + (None,) * 6


def ppo_critic_loss_fn(
    value: torch.Tensor,
    old_value: torch.Tensor,
    target_value: torch.Tensor,
    value_eps_clip: float,
    loss_mask: torch.Tensor | None = None,
    loss_fn_type: str = "mse",
) -> tuple[torch.Tensor, dict]:
    """Clipped value loss of the PPO critic; functional.py:704-778 (stat keys ``clip_mask``, ``loss``)."""
    assert value.dtype == torch.float32
    assert old_value.dtype == torch.float32
    assert target_value.dtype == torch.float32
    if loss_fn_type not in ("mse", "huber"):
        raise NotImplementedError(f"Unknown loss fn type: {loss_fn_type}")
    _require_gpu(value, "value")
    shape = value.shape
    v = value.contiguous().reshape(-1)
    o = old_value.detach().contiguous().reshape(-1)
    t = target_value.detach().contiguous().reshape(-1)
    if loss_mask is not None:
        m8 = _mask_u8(loss_mask).reshape(-1)
        n_valid = _count_nonzero(m8)
    else:
        m8 = None
        n_valid = torch.full((1,), v.numel(), dtype=torch.int32, device=v.device)
    loss, stat_loss, clip = _CriticLoss.apply(v, o, t, m8, value_eps_clip, 0 if loss_fn_type == "mse" else 1, n_valid)
    return loss, dict(clip_mask=clip.bool().view(shape), loss=stat_loss.view(shape))
