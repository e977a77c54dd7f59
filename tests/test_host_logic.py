"""Host-side behaviour that needs no GPU: config validation, argument errors, the no-fallback rule."""
import pytest
import torch

import areal_amd
from areal_amd import RejectionSamplingConfig, synth
from helpers import lets_other_threads_run


# config validation: the cases of tests/test_rejection_sampling.py:8-41 and :806-839 of the reference
def test_config_validation_messages():
    with pytest.raises(ValueError, match="upper must be > 1.0"):
        RejectionSamplingConfig(metric="ratio", upper=1.0)
    with pytest.raises(ValueError, match="lower must be positive"):
        RejectionSamplingConfig(metric="ratio", lower=-0.1, upper=5.0)
    with pytest.raises(ValueError, match="upper must be positive"):
        RejectionSamplingConfig(metric="kl_k2", upper=0.0)
    with pytest.warns(UserWarning, match="agg=.*is ignored"):
        RejectionSamplingConfig(level="token", agg="max", metric="ratio", upper=5.0)
    with pytest.raises(ValueError, match="action='clamp' only supports metric='ratio'"):
        RejectionSamplingConfig(action="clamp", metric="kl_k2", upper=1.0)
    assert RejectionSamplingConfig(action="clamp", metric="ratio", upper=5.0).lower == 0.0
    with pytest.raises(ValueError, match="lower.*cannot be greater than upper"):
        RejectionSamplingConfig(metric="ratio", lower=3.0, upper=2.0)
    for field in ("level", "action", "metric", "agg"):
        with pytest.raises(ValueError, match=f"{field} must be one of"):
            RejectionSamplingConfig(**{field: "invalid"})
    RejectionSamplingConfig(metric="kl_k1", upper=-0.1)  # k1 may be negative: no positivity rule


def test_argument_errors_come_before_device_work():
    x = torch.randn(2, 4)
    m = torch.ones(2, 4, dtype=torch.bool)
    with pytest.raises(ValueError, match="Invalid importance_sampling_level"):
        areal_amd.ppo_actor_loss_fn(x, x, x, x, 0.2, m, importance_sampling_level="invalid")
    cfg = RejectionSamplingConfig(level="token", metric="ratio", upper=5.0)
    with pytest.raises(ValueError, match="shape"):
        areal_amd.apply_rejection_sampling(torch.zeros(1, 2), torch.zeros(1, 3), torch.ones(1, 2), None, cfg)
    with pytest.raises(ValueError, match="ndim"):
        areal_amd.apply_rejection_sampling(torch.zeros(1, 2, 2), torch.zeros(1, 2, 2), torch.ones(1, 2, 2), None, cfg)


def test_cpu_tensors_are_refused_not_emulated():
    x = torch.randn(4, 16)
    y = torch.zeros(4, dtype=torch.int64)
    with pytest.raises(areal_amd.NativeLibraryError, match="no CPU fallback"):
        areal_amd.gather_logprobs(x, y)
    with pytest.raises(areal_amd.NativeLibraryError, match="no CPU fallback"):
        areal_amd.ppo_actor_loss_fn(x, x, x, x, 0.2, torch.ones(4, 16, dtype=torch.bool))


def test_product_package_does_not_import_the_oracle():
    import pathlib

    pkg = pathlib.Path(areal_amd.__file__).parent
    for py in pkg.rglob("*.py"):
        text = py.read_text()
        assert "import oracle" not in text and "from oracle" not in text, py


def test_synthetic_layouts():
    lengths = synth.lengths_uniform(16, 64, 512, seed=0)
    assert len(lengths) == 16 and all(64 <= n <= 512 for n in lengths)
    cu = synth.cu_from_lengths(lengths)
    assert cu.dtype == torch.int32 and cu[0] == 0 and int(cu[-1]) == sum(lengths)
    mask = synth.prefix_mask(lengths, 0.3)
    for i, n in enumerate(lengths):
        seg = mask[int(cu[i]) : int(cu[i + 1])]
        assert int((~seg).sum()) == int(0.3 * n) and not seg[: int(0.3 * n)].any()
    ln = synth.lengths_lognormal(64, 7.5, 0.6, 128, 4096, seed=0)
    assert all(128 <= n <= 4096 for n in ln)
    assert sum(synth.truncate_to_total(ln, 32768)) == 32768
    adv = synth.grpo_advantages([3] * 32, 16, 0.4, seed=1)
    per_seq = adv[::3]
    for g0 in (0, 16):
        grp = per_seq[g0 : g0 + 16]
        assert abs(float(grp.mean())) < 1e-5  # normalised by the group mean
    alt = synth.alternating_mask([2048], 512)
    assert not alt[:512].any() and alt[512:1024].all() and not alt[1024:1536].any()
    case = synth.config0("cpu", seed=0, V=64, n_seqs=3, lo=4, hi=9)
    assert case.logits.shape == (case.n_tokens, 64) and case.logits.dtype == torch.bfloat16
    assert case.labels.dtype == torch.int64 and case.loss_mask.dtype == torch.bool


def test_synthetic_hidden_state_configurations():
    lengths = synth.lengths_until_total(4, 9, 50, seed=1)
    assert sum(lengths) == 50 and all(1 <= n <= 9 for n in lengths)
    c2 = synth.config2("cpu", seed=0, T=300, H=64, V=640)
    assert c2.hidden.shape == (300, 64) and c2.weight.shape == (640, 64) and c2.logits is None
    assert c2.hidden.dtype == torch.bfloat16 and int(c2.cu_seqlens[-1]) == 300
    assert 0.015 < float(c2.weight.float().std()) < 0.025 and 0.9 < float(c2.hidden.float().std()) < 1.1
    c3 = synth.config3("cpu", seed=0, n_seqs=2, seq_len=2048, H=64, V=128)
    assert c3.ppo["c_clip"] == 3.0 and c3.ppo["eps_clip_higher"] == 0.28
    assert c3.ppo["rejection_sampling"]["upper"] == 5.0
    assert not c3.loss_mask[:512].any() and c3.loss_mask[512:1024].all() and not c3.loss_mask[2048 : 2048 + 512].any()
    c4 = synth.config4("cpu", seed=0, T=400, H=64, V=256, lo=8, hi=32)
    assert c4.temperature == 0.7
    best = (c4.hidden.float() @ c4.weight.float().t()).argmax(-1)
    frac = float((best == c4.labels).float().mean())
    assert 0.12 < frac < 0.30  # 20 % argmax labels (+ chance hits)


def test_infer_token_denominator_cases_of_the_reference():
    """The four cases of tests/test_ppo_stats.py:11-51, inputs and expected shapes transcribed."""
    from areal_amd.engine_glue import infer_token_denominator

    cases = [
        (dict(attention_mask=torch.tensor([[1, 1, 0], [1, 1, 1]]), input_ids=torch.tensor([[11, 12], [13, 14]])),
         torch.zeros(5), (2, 3)),                                               # attention_mask wins
        (dict(input_ids=torch.tensor([[11, 12, 13], [14, 15, 16]])), torch.zeros(2, 3), (2, 3)),   # input_ids
        (dict(input_ids=torch.tensor([11, 12, 13, 0])), torch.zeros(3), (3,)),  # padded tree input_ids: fallback
        (dict(logprobs=torch.zeros(2)), torch.zeros(4), (4,)),                  # no metadata: fallback
        (dict(input_ids=torch.tensor([11, 12]), cu_seqlens=torch.tensor([0, 4], dtype=torch.int32)), torch.zeros(2),
         (4,)),                                                                 # tests/test_ppo_stats.py:54-87
    ]
    for data, fallback, shape in cases:
        n_tokens = infer_token_denominator(data, fallback)
        assert tuple(n_tokens.shape) == shape and n_tokens.dtype == torch.bool and bool(n_tokens.all())


@pytest.mark.parametrize("V,stride,lead", [(50257, 50257, 0), (151936, 151936, 1), (32001, 32004, 5), (64, 64, 0),
                                           (64, 72, 0)])
def test_gradient_array_is_laid_out_like_the_logits(V, stride, lead):
    """The array the fused step writes the gradient into has the row stride of the logits and starts at the same
    offset inside a 16-byte piece of memory (the register kernel's condition for rows that are not on 16-byte
    boundaries); rows do not overlap and nothing is shared with the logits."""
    from areal_amd import functional as F

    T = 5
    flat = torch.zeros(lead + T * stride + 8, dtype=torch.bfloat16)
    while flat.data_ptr() % 16:                      # a base on a 16-byte boundary, whatever the allocator gave
        flat = flat[1:]
    logits = flat.as_strided((T, V), (stride, 1), lead)
    out = F._empty_rows_like(logits, stride)
    assert out.shape == logits.shape and out.dtype == logits.dtype
    assert out.stride(1) == 1 and (out.stride(0) == stride or T == 1)
    assert out.data_ptr() % 16 == logits.data_ptr() % 16 == (2 * lead) % 16
    out.fill_(1.0)
    assert float(flat.abs().sum()) == 0.0
    assert float(out.float().sum()) == T * V


def test_arrays_that_the_advantage_rows_take_as_they_are():
    """The native check against the rule in words: float32, contiguous, of the shape and on the device of the mask, without a
    gradient, not made in inference mode; what is masked in place shares no memory with another input."""
    from areal_amd import _native as N

    bs, L = 4, 6
    flat = torch.zeros(4 * bs * L)
    good = lambda i=0: flat[i * bs * L : (i + 1) * bs * L].view(bs, L)
    with torch.inference_mode():
        inferred = torch.zeros(bs, L)
    mask, score = torch.ones(bs, L, dtype=torch.bool), torch.zeros(bs)

    def takes(logp=good(0), roll=True, ref=good(1), attention=mask, score=score, values=good(2), scored=False):
        return N.host().advantages_plain(mask, logp, roll, ref, attention, score, values, scored)

    assert takes() and takes(ref=None, values=None) and takes(roll=False) and takes(scored=True)
    others = [good().double(), good().half(), torch.zeros(L, bs).t(), torch.zeros(bs, 2 * L)[:, ::2], torch.zeros(bs, L + 1)[:, :L],
              torch.zeros(bs + 1, L), torch.zeros(bs * L), torch.zeros(bs, L, requires_grad=True), inferred,
              torch.zeros(bs, L, device="meta")]
    for x in others:
        assert not takes(logp=x) and not takes(ref=x) and not takes(values=x)
    with torch.inference_mode():
        assert takes(logp=inferred) and takes(ref=inferred)
    for x in (torch.zeros(bs + 1), torch.zeros(bs, 1), torch.zeros(2 * bs)[::2], torch.zeros(bs).double()):
        assert not takes(score=x)
    assert not takes(attention=mask[:, 1:]) and takes(attention=mask.long())
    shifted = flat[bs * L - 1 : 2 * bs * L - 1].view(bs, L)  # its first element is the last one of good(0)
    for x in (good(0), shifted):
        assert not takes(ref=x) and not takes(values=x, roll=False) and takes(values=x, ref=None)
    assert not takes(ref=good(1), values=good(1))
    inside = flat[bs * L : bs * L + bs]
    assert takes(score=inside) and not takes(score=inside, scored=True)
    inside = flat[:bs]
    assert takes(score=inside, scored=True) and not takes(score=inside, scored=True, roll=False)


def test_temperature_zero_is_refused_before_the_native_step():
    """A temperature of zero is a division by zero, as on every other path, not an infinite factor for the kernels."""
    from types import SimpleNamespace

    from areal_amd import _native as N
    from areal_amd import functional as F

    x = torch.zeros(2, 8, requires_grad=True)
    step = SimpleNamespace(struct=N.PpoStep(), loss=torch.zeros(()))
    with pytest.raises(ZeroDivisionError):
        F._fused_logits(x, step, torch.zeros(2, dtype=torch.int64), 8, 0.0, False)


def test_native_calls_that_allocate_let_other_threads_run():
    """An allocation can wait for the device: the native host side makes it without the GIL."""
    import ctypes as C

    from areal_amd import _native as N

    host, step, T = N.host(), N.PpoStep(), 400
    mask, rows = torch.ones(T, dtype=torch.bool), torch.zeros(10, 448)
    assert not lets_other_threads_run(lambda: host.step_rows(rows, T))  # (views only: the measure itself)
    assert lets_other_threads_run(lambda: host.make_step(C.addressof(step), T, T, mask, None, None, None, None, 0, True, False,
                                                         None, None, mask, torch.device("cpu")))
    assert lets_other_threads_run(lambda: host.empty_rows_like(rows, 448))


def test_moments_of_a_mask_in_host_memory_are_refused(monkeypatch):
    """Every mask is asked for its device before its address goes to a kernel: the supervised loss function takes a mask
    from anywhere, and its statistics used to refuse one in host memory."""
    from areal_amd import advantages as A

    def stands_for_a_device(t, name):
        if "mask" in name:
            raise areal_amd.NativeLibraryError(f"{name}: no CPU fallback")

    def launched():
        raise AssertionError("the address of the mask went to the library")

    monkeypatch.setattr(A, "_require_gpu", stands_for_a_device)
    monkeypatch.setattr(A.N, "load", launched)
    with pytest.raises(areal_amd.NativeLibraryError, match="the mask of x"):
        A.moments_table([("x", torch.zeros(4), torch.ones(4, dtype=torch.bool))])


@pytest.mark.parametrize("waiting_fails", [False, True])
def test_host_memory_of_abandoned_steps_under_threads(monkeypatch, waiting_fails):
    """Past the bound the memory that nobody read goes back once the device has been waited for.  Another thread may take
    entries after their number was read, and the wait may fail: nothing is raised into the caller's step, and memory that
    a kernel may still write to is not let go."""
    from collections import deque

    from areal_amd.functional import _HostSlot

    class AnotherThreadTakesSome(deque):
        def __len__(self):
            return super().__len__() + 3

    def wait(index):
        waited.append(index)
        if waiting_fails:
            raise RuntimeError("operation not permitted when stream is capturing")

    entries = [([tag], [0, 0, 0, -1], tag, torch.device("cuda:0")) for tag in range(1, 71)]
    unread, pool, waited = AnotherThreadTakesSome(entries), deque(maxlen=64), []
    monkeypatch.setattr(_HostSlot, "_unread", unread)
    monkeypatch.setattr(_HostSlot, "_pool", pool)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "synchronize", wait)
    _HostSlot._take_back()
    assert waited == [0]
    if waiting_fails:
        assert list(unread) == entries and not pool
    else:
        assert not list(unread) and [m for m, _ in pool] == [[tag] for tag in range(7, 71)]


def test_tags_of_steps_fit_the_word_they_come_back_in(monkeypatch):
    """A tag is compared with an int32 in host memory, also after 2^31 steps."""
    import ctypes
    import itertools
    from collections import deque

    from areal_amd.functional import _HostSlot

    for first in (1, 0x7FFFFFFE, 0x80000000, 0xFFFFFFFF, 2 ** 40):
        monkeypatch.setattr(_HostSlot, "_tags", itertools.count(first))
        monkeypatch.setattr(_HostSlot, "_unread", deque())
        monkeypatch.setattr(_HostSlot, "_pool", deque((torch.empty(4), None) for _ in range(3)))
        slots = [_HostSlot(torch.device("cuda:0")) for _ in range(3)]
        tags = [slot.tag for slot in slots]
        for slot in slots:
            slot._memory = None  # nothing is given back
        assert all(t > 0 and ctypes.c_int32(t).value == t for t in tags) and len(set(tags)) == 3


def test_weight_zero_that_the_host_knows_runs_no_forward(monkeypatch):
    from areal_amd import engine_glue as G

    ran = []
    monkeypatch.setattr(G, "_logprobs_impl", lambda *a, **kw: ran.append("logits"))
    monkeypatch.setattr(G, "_lm_head_impl", lambda *a, **kw: ran.append("lm_head"))
    x = torch.ones(4, 8, requires_grad=True)
    for zero in (0, 0.0, torch.tensor(0)):
        assert float(G.compute_loss_with(x, {}, {}, 0, None, lambda mb: zero, 1.0).detach()) == 0.0
        assert float(G.compute_lm_head_loss_with(x, x, {}, {}, 0, None, lambda mb: zero, 1.0).detach()) == 0.0
    assert not ran


@pytest.mark.parametrize("length,pad,want", [(10, 0, [1] * 10), (12, 0, [1] * 12), (8, 0, [1] * 8), (7, 3, [1] * 7),
                                             (10, 3, [1] * 7), (5, 3, [1] * 5 + [0] * 2), (0, 10, [0] * 10)])
def test_gradient_mask_of_a_padded_micro_batch(monkeypatch, length, pad, want):
    """Ten rows: with batch padding the mask is cut or continued with zeros to the rows without padding, without any it
    goes to the op as it is (which refuses other lengths)."""
    from areal_amd import engine_glue as G

    class Reached(Exception):
        pass

    def op(hidden, weight, labels, temperature, token_mask, want_minmax, backward, grad_token_mask, kept_per_chunk, **kw):
        seen.append(grad_token_mask.tolist())
        raise Reached

    seen = []
    monkeypatch.setattr(G, "_lm_head_impl", op)
    with pytest.raises(Reached):
        G.compute_lm_head_loss_with(torch.zeros(10, 8), torch.zeros(16, 8), dict(rolled_input_ids=torch.zeros(10)), {}, pad,
                                    None, lambda mb: 1.0, 1.0, grad_token_mask=torch.ones(length, dtype=torch.bool))
    assert seen == [[bool(v) for v in want]]


def test_arrays_that_the_advantage_kernel_may_write():
    """A tensor made in inference mode may not be written outside it: torch refuses the in-place product, and so the
    one-pass kernel, which masks in place through an address, does not take it."""
    from areal_amd.advantages import _plain

    cpu, made = torch.device("cpu"), torch.zeros(2, 3)
    with torch.inference_mode():
        made_there = torch.zeros(2, 3)
        assert _plain(made_there, (2, 3), cpu) and _plain(made, (2, 3), cpu)
    assert _plain(made, (2, 3), cpu) and not _plain(made_there, (2, 3), cpu)
    assert not _plain(made.double(), (2, 3), cpu) and not _plain(torch.zeros(3, 2).t(), (2, 3), cpu)
    assert not _plain(torch.zeros(2, 3, requires_grad=True), (2, 3), cpu) and _plain(None, (2, 3), cpu)
