"""The work that a trainer has this library do, as measurable cases.

One optimizer step of a PPO / GRPO trainer runs, in this order: log-probs of the rollout under the proximal and reference
policies (forward only), the advantage pipeline over the padded batch, and one loss per packed micro-batch with its
backward; a supervised trainer runs the last part with its own loss.  A model that hands over its logits takes the
logits entry points, one that hands over its final hidden states takes the lm_head ones.  Sizes are those of the
benchmark configurations (``areal_amd/synth.py``) and of the tests, or generic (hidden sizes of small and large models,
vocabularies that are and are not multiples of 8, micro-batches from a few hundred to some ten thousand tokens).

``op`` of a case:

  fused          ``fused_logprobs_ppo_loss`` on [T, V] logits and its backward
  sft            ``engine_glue.compute_logprobs_and_sft_loss``: the supervised step on [T, V] logits
  any_loss       ``engine_glue.compute_loss_with(grpo_loss_fn)``: log-prob op, loss with its logged statistics, backward
  logp           ``engine_glue.compute_logprobs``: forward-only log-probs of [T, V] logits
  lm_head        ``fused_lm_head_ppo_loss`` on [T, H] hidden states and the [V, H] weight, and its backward
  lm_head_any    ``engine_glue.compute_lm_head_loss_with(grpo_loss_fn)``: the same for sequence-level ratios
  lm_head_logp   ``engine_glue.compute_lm_head_logprobs``: forward-only log-probs from hidden states
  advantages     ``engine_glue.compute_advantages`` on padded [bs, L] tensors
"""
import math

import torch

from areal_amd import NormConfig, Normalization, RejectionSamplingConfig
from areal_amd import engine_glue, fused_lm_head_ppo_loss, fused_logprobs_ppo_loss, synth

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
MASKED = 0.3  # the prompt: this share of every sequence has no loss
ROWS_PER_PIECE = 1024  # rows whose fp32 values are held at a time while inputs are made


def listed():
    return [
        # the last micro-batch of a step, or one short sequence: latency and launches
        dict(name="fused_last_micro_batch", op="fused", T=200, V=151936, dtype="bf16", rs="token", pad=0),
        # configuration 0: 16 sequences of 64 to 512 tokens, no importance-weight cap
        dict(name="fused_cfg0", op="fused", T=4718, V=151936, dtype="bf16", rs="none", pad=0),
        # configuration 1 cut to one micro-batch of 32768 tokens: importance-weight cap, dual clip
        dict(name="fused_cfg1_32k", op="fused", T=32768, V=151936, dtype="bf16", rs="token", pad=0),
        # rows that start at any even address (vocabulary not a multiple of 8), fp16, batch padding
        dict(name="fused_odd_vocab_f16", op="fused", T=6007, V=50257, dtype="f16", rs="sequence", pad=41),
        # supervised fine-tuning on a 32k vocabulary
        dict(name="sft_32k_vocab", op="sft", T=8192, V=32768, dtype="bf16", pad=128),
        # the loss function as the engine calls it, on fp32 logits, with everything it logs
        dict(name="any_loss_f32", op="any_loss", T=4096, V=128256, dtype="f32", rs="token", level="token", pad=64),
        # proximal / reference log-probs of a rollout
        dict(name="logp_16k", op="logp", T=16384, V=151936, dtype="bf16"),
        # configuration 2: the 8B shape from hidden states
        dict(name="lm_head_cfg2", op="lm_head", T=16384, H=4096, V=151936, rs="none", pad=0),
        # the same step of a small model
        dict(name="lm_head_small_model", op="lm_head", T=4096, H=1536, V=151936, rs="token", pad=56),
        # sequence-level importance ratios of a small model on a vocabulary that is not a multiple of 8
        dict(name="lm_head_sequence_level", op="lm_head_any", T=1900, H=1024, V=50257, rs="none", level="sequence", pad=20),
        # forward-only log-probs from hidden states
        dict(name="lm_head_logp_2k", op="lm_head_logp", T=8000, H=2048, V=151936),
        # advantages of a batch of 512 responses: reward and advantage normalisation, KL penalty, GAE with a critic
        dict(name="advantages_512x4096", op="advantages", bs=512, L=4096, group=16, critic=True),
    ]


def _spread(rng, lo, hi):
    """A whole number from lo to hi, uniform in its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _vocab(rng, lo=16000, hi=262144):
    v = _spread(rng, lo, hi)
    kind = rng.randrange(3)  # as drawn (odd ones among them), a multiple of 8, a multiple of 128
    return v if kind == 0 else (max(lo, v // 8 * 8) if kind == 1 else max(lo, v // 128 * 128))


def draw(rng):
    op = rng.choice(["fused", "fused", "sft", "any_loss", "logp", "lm_head", "lm_head", "lm_head_any", "lm_head_logp", "advantages"])
    if op == "advantages":
        group = rng.choice([4, 8, 16])
        bs = max(group, _spread(rng, 32, 1024) // group * group)
        return dict(op=op, bs=bs, L=_spread(rng, 300, 4096), group=group, critic=rng.random() < 0.5)
    c = dict(op=op, V=_vocab(rng))
    if op in ("fused", "sft", "any_loss", "logp"):
        c["dtype"] = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
        width = 2 if c["dtype"] == "f32" else 1
        c["T"] = _spread(rng, 128, min(32768, 32768 * 151936 // (c["V"] * width)))
    else:
        c["H"] = _spread(rng, 512, 5376) // 8 * 8
        most = 16384 * 4096 * 151936 // (c["V"] * c["H"])
        c["T"] = _spread(rng, 256, min(16384, most))
    if op in ("fused", "any_loss", "lm_head", "lm_head_any"):
        c["rs"] = rng.choice(["none", "token", "sequence"])
    if op in ("any_loss", "lm_head_any"):
        c["level"] = "sequence" if op == "lm_head_any" else rng.choice(["token", "sequence"])
    if op in ("fused", "sft", "any_loss", "lm_head", "lm_head_any"):
        c["pad"] = rng.choice([0, rng.randrange(1, 128)])
    return c


def _rs_config(case):
    if case["rs"] == "none":
        return None
    if case["rs"] == "token":
        return RejectionSamplingConfig(level="token", action="mask", metric="ratio", upper=5.0)
    return RejectionSamplingConfig(level="sequence", action="mask", metric="ratio", agg="mean", upper=1.006)


def _loss_scale(case):
    return 256.0 if case.get("dtype") == "f16" else 0.25  # fp16 gradients are kept in range by a scaled loss


def _lengths(T, seed):
    """Sequence lengths that add up to T: T / 500 sequences (two at least), lognormal around their mean."""
    n = max(2, T // 500)
    weights = synth.lengths_lognormal(n, 6.2, 0.6, 32, 4096, seed)
    lengths = [max(1, T * w // sum(weights)) for w in weights]
    lengths[0] += T - sum(lengths)
    return lengths


def _label_logp(rows, labels):
    z = rows.float()
    return z.gather(1, labels[:, None]).squeeze(1) - torch.logsumexp(z, 1)


def _packed(case, seed, dev):
    """What surrounds the [T + pad] rows of a packed micro-batch, and the generator for the rest."""
    T, pad = case["T"], case.get("pad", 0)
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    lengths = _lengths(T, seed)
    s = dict(case=case, g=g, lengths=lengths, cu=synth.cu_from_lengths(lengths).to(dev),
             mask=synth.prefix_mask(lengths, MASKED).to(dev), labels=torch.randint(0, case["V"], (T + pad,), generator=g, device=dev))
    s["adv"] = synth.per_sequence_normal_advantages(lengths, seed + 3).float().to(dev)
    return s


def _with_policies(s, ref):
    """Behaviour and proximal log-probs around the model's own, and the policy version that wrote each token."""
    T, g, dev = s["case"]["T"], s["g"], ref.device
    noise = lambda: 0.05 * torch.randn(T, generator=g, device=dev)
    s["old"], s["prox"] = ref[:T] + noise(), ref[:T] + noise()
    s["versions"] = torch.randint(3, 7, (T,), generator=g, device=dev, dtype=torch.int32)
    return s


def _prepare_logits(case, seed, dev):
    s = _packed(case, seed, dev)
    n, V, dtype = case["T"] + case.get("pad", 0), case["V"], DTYPES[case["dtype"]]
    x = torch.empty(n, V, dtype=dtype, device=dev)
    # most tokens were sampled from a policy near this one: their logit stands out of the N(0, 3^2) of the others
    sampled = torch.rand(n, generator=s["g"], device=dev) < 0.8
    peak = 15.0 + 1.5 * torch.randn(n, generator=s["g"], device=dev)
    ref = torch.empty(n, device=dev)
    for a in range(0, n, ROWS_PER_PIECE):
        b = min(a + ROWS_PER_PIECE, n)
        z = 3.0 * torch.randn(b - a, V, generator=s["g"], device=dev)
        y = s["labels"][a:b, None]
        z.scatter_(1, y, torch.where(sampled[a:b, None], peak[a:b, None], z.gather(1, y)))
        x[a:b] = z.to(dtype)
        if case["op"] != "logp":
            ref[a:b] = _label_logp(x[a:b], s["labels"][a:b])
    if case["op"] == "logp":
        s["logits"] = x
        return s
    s["logits"] = x.requires_grad_()
    return _with_policies(s, ref)


def _prepare_hidden(case, seed, dev):
    s = _packed(case, seed, dev)
    n = case["T"] + case.get("pad", 0)
    s["hidden"] = torch.randn(n, case["H"], generator=s["g"], device=dev).to(torch.bfloat16)
    s["weight"] = (0.02 * torch.randn(case["V"], case["H"], generator=s["g"], device=dev)).to(torch.bfloat16)
    if case["op"] == "lm_head_logp":
        return s
    ref = torch.empty(n, device=dev)
    for a in range(0, n, ROWS_PER_PIECE):
        b = min(a + ROWS_PER_PIECE, n)
        ref[a:b] = _label_logp(torch.nn.functional.linear(s["hidden"][a:b], s["weight"]), s["labels"][a:b])
    s["hidden"].requires_grad_()
    s["weight"].requires_grad_()
    return _with_policies(s, ref)


def _prepare_advantages(case, seed, dev):
    bs, L, group = case["bs"], case["L"], case["group"]
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    at = torch.arange(L, device=dev)[None]
    lens = torch.randint(L // 4, L + 1, (bs, 1), generator=g, device=dev)
    attention = at < lens
    loss_mask = attention & (at >= (MASKED * lens).long())
    logp = -2.0 * torch.rand(bs, L, generator=g, device=dev)
    data = dict(
        input_ids=torch.randint(0, 32000, (bs, L), generator=g, device=dev), attention_mask=attention, loss_mask=loss_mask,
        logprobs=logp * loss_mask, rewards=(torch.rand(bs, generator=g, device=dev) < 0.4).float(),
        ref_logp=logp + 0.05 * torch.randn(bs, L, generator=g, device=dev),
        prox_logp=logp + 0.05 * torch.randn(bs, L, generator=g, device=dev),
    )
    if case["critic"]:
        data["values"] = torch.randn(bs, L, generator=g, device=dev)
    return dict(
        case=case, data=data,
        reward_norm=Normalization(NormConfig(mean_level="group", std_level="group", group_size=group)),
        adv_norm=Normalization(NormConfig(mean_level="batch", std_level="batch")),
    )


def prepare(case, seed):
    dev = torch.device("cuda")
    if case["op"] == "advantages":
        return _prepare_advantages(case, seed, dev)
    return (_prepare_hidden if "H" in case else _prepare_logits)(case, seed, dev)


def _micro_batch(s):
    return dict(loss_mask=s["mask"], logprobs=s["old"], prox_logp=s["prox"], advantages=s["adv"], cu_seqlens=s["cu"],
                versions=s["versions"])


def _grpo(s, eps_clip=0.2):
    case = s["case"]

    def loss_fn(logprobs, entropy, mb, vocab_min_logits=None, vocab_max_logits=None):
        return engine_glue.grpo_loss_fn(
            logprobs, entropy, mb, eps_clip, 0.28, 3.0, rejection_sampling=_rs_config(case),
            importance_sampling_level=case["level"], current_version=7, vocab_min_logits=vocab_min_logits,
            vocab_max_logits=vocab_max_logits)

    return loss_fn


def _weight(mb):
    return mb["loss_mask"].count_nonzero()


def _logged(stat):
    """The per-token statistics and, of every reduced one, the mean and the largest value (what a trainer exports)."""
    out = {k: v for k, v in stat.items() if k not in ("reduced", "loss_mask")}
    reduced = stat["reduced"]
    rows = {k: v for k, v in reduced.items() if isinstance(v, dict) and "avg" in v}
    rows.update(reduced["compute_logp"])
    rows.update({k: v for k, v in reduced["version_stats"].items() if isinstance(v, dict)})
    for k, v in rows.items():
        out["avg/" + k], out["max/" + k] = v["avg"], v["max"]
    return out


def run(s):
    case = s["case"]
    op = case["op"]
    if op == "fused":
        x = s["logits"]
        loss, stat = fused_logprobs_ppo_loss(
            x, s["labels"], s["prox"], s["old"], s["adv"], 0.2, s["mask"], eps_clip_higher=0.28, c_clip=3.0,
            rejection_sampling=_rs_config(case), cu_seqlens=s["cu"], loss_scale=_loss_scale(case))
        return dict(stat, loss_sum=loss, d_logits=torch.autograd.grad(loss, x)[0])
    if op == "sft":
        x = s["logits"]
        loss, stat = engine_glue.compute_logprobs_and_sft_loss(
            x, dict(rolled_input_ids=s["labels"]), dict(loss_mask=s["mask"], cu_seqlens=s["cu"]), 40000.0,
            loss_multiplier=_loss_scale(case))
        return dict(stat, loss_sum=loss, d_logits=torch.autograd.grad(loss, x)[0])
    if op == "any_loss":
        x = s["logits"]
        loss, stat = engine_glue.compute_loss_with(x, dict(rolled_input_ids=s["labels"]), _micro_batch(s), case["pad"],
                                                   _grpo(s), _weight, 40000.0, loss_multiplier=_loss_scale(case))
        return dict(_logged(stat), loss_sum=loss, d_logits=torch.autograd.grad(loss, x)[0])
    if op == "logp":
        return engine_glue.compute_logprobs(s["logits"], dict(rolled_input_ids=s["labels"]))
    if op == "lm_head":
        h, w = s["hidden"], s["weight"]
        loss, stat = fused_lm_head_ppo_loss(
            h, w, s["labels"], s["prox"], s["old"], s["adv"], 0.2, s["mask"], eps_clip_higher=0.28, c_clip=3.0,
            rejection_sampling=_rs_config(case), cu_seqlens=s["cu"], loss_scale=0.25)
        d_hidden, d_weight = torch.autograd.grad(loss, [h, w])
        return dict(stat, loss_sum=loss, d_hidden=d_hidden, d_weight=d_weight)
    if op == "lm_head_any":
        h, w = s["hidden"], s["weight"]
        loss, stat = engine_glue.compute_lm_head_loss_with(h, w, dict(rolled_input_ids=s["labels"]), _micro_batch(s),
                                                           case["pad"], _grpo(s, 3e-4), _weight, 40000.0)
        d_hidden, d_weight = torch.autograd.grad(loss, [h, w])
        return dict(_logged(stat), loss_sum=loss, d_hidden=d_hidden, d_weight=d_weight)
    if op == "lm_head_logp":
        return engine_glue.compute_lm_head_logprobs(s["hidden"], s["weight"], dict(rolled_input_ids=s["labels"]))
    data = engine_glue.compute_advantages(
        dict(s["data"]), kl_ctl=0.05, kl_estimator="k1", discount=1.0, gae_lambda=0.95 if case["critic"] else 1.0,
        reward_bias=-0.5, reward_scaling=10.0, reward_norm=s["reward_norm"], adv_norm=s["adv_norm"], use_decoupled_loss=True)
    return {k: data[k] for k in ("advantages", "returns", "kl_rewards", "tot_rewards", "loss_mask", "logprobs")}


def work(case):
    op = case["op"]
    if op == "advantages":
        n = case["bs"] * case["L"]
        # two byte masks, log-probs and reference log-probs (and values) in, six float tensors out
        return dict(bytes=n * (2 + 8 + (4 if case["critic"] else 0) + 24), flops=60 * n)
    T, V = case["T"] + case.get("pad", 0), case["V"]
    if "H" in case:
        H = case["H"]
        operands = 2 * H * (T + V)
        if op == "lm_head_logp":
            return dict(bytes=operands + 12 * T, flops=2 * T * V * H)
        kept = int((1 - MASKED) * case["T"])  # only tokens with a loss have a gradient
        return dict(bytes=2 * operands + 60 * T, flops=(2 * T + 4 * kept) * V * H)
    width = 4 if case["dtype"] == "f32" else 2
    if op == "logp":
        return dict(bytes=width * T * V + 12 * T, flops=5 * T * V)
    return dict(bytes=2 * width * T * V + 60 * T, flops=9 * T * V)


def tolerance(case):
    """About four times what the path differs by from the same computation in 64 bits (largest output first)."""
    op = case["op"]
    if op == "advantages":
        return dict(rel=1e-6, max=6e-6)  # 1.8e-7, 1.5e-6
    if op in ("logp", "lm_head_logp"):  # 5e-8, 2e-7; the sums of an lm_head in another order add as much again
        return dict(rel=5e-7, max=2e-6)
    if "H" in case:  # d(weight): 2.9e-3, its smallest entries 0.1 of the root mean square; bf16 rows and bf16 results
        return dict(rel=1.2e-2, max=0.4, differ=1e-3)
    if case["dtype"] == "bf16":  # d(logits): 1.6e-3, 4e-3
        return dict(rel=6e-3, max=2e-2, differ=1e-3)
    if case["dtype"] == "f16":  # d(logits): 2.2e-4, 5e-4
        return dict(rel=1e-3, max=2e-3, differ=1e-3)
    # fp32, long rows (held in 24 bits for the gradient): 4.8e-5, 5e-3; shorter rows: differences of log-probs, 8e-6, 4e-5
    return dict(rel=2e-4, max=2e-2, differ=1e-3) if case["V"] > 114688 else dict(rel=4e-5, max=2e-4, differ=1e-3)
