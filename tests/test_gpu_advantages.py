"""GPU parity of the advantage pipeline (GAE scan, Normalization, masked moments) against the CPU oracle and the
reference's own known-answer cases."""
import itertools
import math
import json
from pathlib import Path

import pytest
import torch

import areal_amd
from areal_amd import NormConfig, Normalization
from oracle import advantages as O

pytestmark = pytest.mark.gpu

GOLD = json.loads((Path(__file__).parent / "golden" / "reference_norm_known_answers.json").read_text())


@pytest.mark.parametrize("c", GOLD["cases"], ids=[c["name"] for c in GOLD["cases"]])
def test_normalization_reference_known_answers(device, c):
    x = torch.tensor(c["x"], dtype=torch.float32)
    mask = torch.ones_like(x) if c["mask"] == "ones" else torch.tensor(c["mask"], dtype=torch.float32)
    out = Normalization(NormConfig(**c["cfg"]))(x.to(device), mask.to(device)).cpu()
    assert out.dtype == torch.float32 and out.shape == x.shape
    atol = c.get("atol", 1e-6)
    if "expected" in c:
        assert torch.allclose(out, torch.tensor(c["expected"], dtype=torch.float32), atol=atol)
    for key, val in c.get("expected_at", {}).items():
        i, j = (int(t) for t in key.split(","))
        assert abs(float(out[i, j]) - val) <= atol
    p = c.get("properties", {})
    if "mean_abs_below" in p:
        assert abs(float(out.mean())) < p["mean_abs_below"]
    if "nonmasked_mean_abs_below" in p:
        nm = out[mask.bool()]
        assert abs(float(nm.mean())) < p["nonmasked_mean_abs_below"]
        assert abs(float(nm.std()) - 1.0) < p["nonmasked_unbiased_std_minus_one_abs_below"]


LEVELS = [None, "batch", "group"]


@pytest.mark.parametrize("mean_level,std_level", list(itertools.product(LEVELS, LEVELS)))
@pytest.mark.parametrize("loo,unbiased", [(False, True), (True, False), (True, True)])
def test_normalization_matches_oracle(device, mean_level, std_level, loo, unbiased):
    g = torch.Generator().manual_seed(hash((str(mean_level), str(std_level), loo, unbiased)) % 1000)
    for shape, gs, with_mask in [((14, 37), 4, True), ((12, 5), 3, False), ((9,), 2, False), ((6, 3, 4), 1, True),
                                 ((5, 8), 8, True)]:
        x = torch.randn(*shape, generator=g) * 2.0 + 0.5
        mask = (torch.rand(*shape, generator=g) < 0.6).float() if with_mask else None
        cfg = dict(mean_level=mean_level, mean_leave1out=loo, std_level=std_level, std_unbiased=unbiased, eps=1e-5,
                   group_size=gs)
        want = O.normalization(x, mask, **cfg)
        got = Normalization(NormConfig(**cfg))(x.to(device), None if mask is None else mask.to(device)).cpu()
        assert got.shape == want.shape and got.dtype == torch.float32
        scale = float(want.abs().max()) + 1.0
        assert float((got - want).abs().max()) <= 2e-6 * scale, (shape, gs, cfg)


def test_normalization_edge_cases(device):
    x = torch.randn(4, 6)
    zero = torch.zeros_like(x)
    out = Normalization(NormConfig())(x.to(device), zero.to(device))
    assert torch.equal(out.cpu(), x)  # nothing active: the input comes back
    with pytest.raises(ValueError, match="group_size must be a positive integer"):
        NormConfig(mean_level="group", std_level="batch", group_size=0)
    with pytest.raises(ValueError, match="mean_level must be"):
        NormConfig(mean_level="bad")
    with pytest.raises(areal_amd.NativeLibraryError):
        Normalization(NormConfig())(x)  # CPU tensors are refused
    # bf16 input is accepted and comes back float32
    out = Normalization(NormConfig())(x.bfloat16().to(device))
    assert out.dtype == torch.float32
    assert torch.allclose(out.cpu(), O.normalization(x.bfloat16().float()), atol=1e-5)


def test_normalization_full_size(device):
    bs, L = 512, 4096
    g = torch.Generator().manual_seed(0)
    x = torch.randn(bs, L, generator=g)
    mask = (torch.rand(bs, L, generator=g) < 0.7).float()
    for cfg in (dict(), dict(mean_level="group", std_level="group", group_size=16),
                dict(mean_level="batch", std_level="group", group_size=8, mean_leave1out=True)):
        want = O.normalization(x, mask, **cfg)
        norm = Normalization(NormConfig(**cfg))
        got = norm(x.to(device), mask.to(device))
        assert float((got.cpu() - want).abs().max()) < 1e-5
        assert torch.equal(got, norm(x.to(device), mask.to(device)))  # fixed summation order


@pytest.mark.parametrize("bs,L", [(1, 1), (3, 2), (5, 63), (4, 64), (7, 65), (6, 66), (9, 129), (2, 1000), (3, 4096),
                                   (2, 4097), (2, 4098), (2, 9001), (1, 20000)])
@pytest.mark.parametrize("gamma,lam", [(1.0, 1.0), (0.99, 0.95)])
def test_gae_matches_oracle(device, bs, L, gamma, lam):
    g = torch.Generator().manual_seed(bs * 1000 + L)
    r = torch.randn(bs, L, generator=g)
    v = torch.randn(bs, L, generator=g)
    m = (torch.rand(bs, L, generator=g) < 0.6).float()
    ne = torch.rand(bs, generator=g) < 0.5
    want_a, want_r = O.gae(r.double(), v.double(), m.double(), ne.double(), gamma, lam)
    adv, ret = areal_amd.gae_advantages(r.to(device), v.to(device), m.to(device), ne.to(device), gamma, lam)
    scale = float(want_a.abs().max()) + 1.0
    assert float((adv.cpu().double() - want_a).abs().max()) < 2e-5 * scale
    assert float((ret.cpu().double() - want_r).abs().max()) < 2e-5 * scale
    # the fp32 loop of the reference agrees to the same bar
    ref_a, _ = O.gae(r, v, m, ne.float(), gamma, lam)
    assert float((adv.cpu() - ref_a).abs().max()) < 4e-5 * scale
    # no critic: values = None stands for zeros
    adv0, ret0 = areal_amd.gae_advantages(r.to(device), None, m.to(device), None, gamma, lam)
    want0, _ = O.gae(r.double(), torch.zeros(bs, L).double(), m.double(), torch.zeros(bs).double(), gamma, lam)
    assert float((adv0.cpu().double() - want0).abs().max()) < 2e-5 * (float(want0.abs().max()) + 1.0)
    assert torch.equal(adv0, ret0)


def test_gae_full_size_and_grpo_shape(device):
    bs, L = 512, 4096
    g = torch.Generator().manual_seed(1)
    lens = torch.randint(L // 4, L + 1, (bs,), generator=g)
    pos = torch.arange(L)[None, :]
    m = ((pos >= (lens[:, None] * 0.3).long()) & (pos < lens[:, None] - 1)).float()
    r = torch.zeros(bs, L)
    r[torch.arange(bs), (lens - 2).clamp(min=0)] = torch.randn(bs, generator=g)   # one terminal reward per sequence
    r = r - 0.01 * torch.rand(bs, L, generator=g) * m                             # plus KL penalties
    v = torch.randn(bs, L, generator=g) * 0.1
    ne = lens == L
    want_a, want_r = O.gae(r, v, m, ne.float(), 1.0, 1.0)
    adv, ret = areal_amd.gae_advantages(r.to(device), v.to(device), m.to(device), ne.to(device), 1.0, 1.0)
    assert float((adv.cpu() - want_a).abs().max()) < 1e-4 and float((ret.cpu() - want_r).abs().max()) < 1e-4
    adv2, _ = areal_amd.gae_advantages(r.to(device), v.to(device), m.to(device), ne.to(device), 1.0, 1.0)
    assert torch.equal(adv, adv2)


def test_masked_moments(device):
    g = torch.Generator().manual_seed(2)
    n = 10007
    vals = {f"s{k}": torch.randn(n, generator=g) * (k + 1) for k in range(5)}
    vals["flag"] = (torch.rand(n, generator=g) < 0.3).float()
    mask = torch.rand(n, generator=g) < 0.4
    got = areal_amd.masked_moments({k: v.to(device) for k, v in vals.items()}, mask.to(device))
    want = O.masked_moments(list(vals.values()), mask)
    for i, k in enumerate(vals):
        assert float(got[k]["sum"]) == pytest.approx(float(want[i, 0]), rel=1e-5, abs=1e-4)
        assert float(got[k]["min"]) == float(want[i, 1]) and float(got[k]["max"]) == float(want[i, 2])
        assert float(got[k]["count"]) == float(want[i, 3])
        assert float(got[k]["avg"]) == pytest.approx(float(want[i, 0] / want[i, 3]), rel=1e-5, abs=1e-6)
    empty = areal_amd.masked_moments({"a": vals["s0"].to(device)}, torch.zeros(n, dtype=torch.bool, device=device))
    assert float(empty["a"]["count"]) == 0.0 and float(empty["a"]["min"]) == float("inf")
    with pytest.raises(ValueError):
        areal_amd.masked_moments({"a": vals["s0"][:5].to(device)}, mask.to(device))


@pytest.mark.parametrize("est", ["k1", "k2", "k3"])
@pytest.mark.parametrize("no_eos_zero", [False, True])
def test_kl_rewards_match_oracle(device, est, no_eos_zero):
    g = torch.Generator().manual_seed(11)
    bs, L = 9, 40
    seqlens = torch.tensor([40, 1, 2, 17, 40, 5, 39, 3, 40])
    old, ref = -torch.rand(bs, L, generator=g) * 12, -torch.rand(bs, L, generator=g) * 3
    mask = (torch.rand(bs, L, generator=g) < 0.6).float()
    score = torch.randn(bs, generator=g)
    want_r, want_k = O.kl_rewards(old * mask, ref * mask, mask, seqlens, score, 0.2, est, no_eos_zero)
    r, k = areal_amd.kl_regularized_rewards((old * mask).to(device), (ref * mask).to(device), mask.to(device),
                                            seqlens.to(device), score.to(device), 0.2, est, no_eos_zero)
    assert torch.allclose(k.cpu(), want_k, rtol=1e-5, atol=1e-6) and torch.allclose(r.cpu(), want_r, rtol=1e-5, atol=1e-6)
    r0, _ = areal_amd.kl_regularized_rewards((old * mask).to(device), None, mask.to(device), seqlens.to(device),
                                             score.to(device), 0.2, est, no_eos_zero)
    w0, _ = O.kl_rewards(old * mask, torch.zeros(bs, L), mask, seqlens, score, 0.2, est, no_eos_zero)
    assert torch.allclose(r0.cpu(), w0, rtol=1e-5, atol=1e-6)
    with pytest.raises(ValueError, match="Invalid KL estimator"):
        areal_amd.kl_regularized_rewards(old.to(device), None, mask.to(device), seqlens.to(device), score.to(device), 0.1, "k9")


@pytest.mark.parametrize("case", ["grpo", "critic_kl", "recompute", "overlong"])
def test_compute_advantages_matches_oracle(device, case):
    from areal_amd.engine_glue import compute_advantages

    g = torch.Generator().manual_seed(21)
    bs, L = 16, 96
    lens = torch.randint(4, L + 1, (bs,), generator=g)
    lens[0] = L
    pos = torch.arange(L)[None, :]
    am = (pos < lens[:, None]).long()
    lm = ((pos >= (lens[:, None] * 0.4).long()) & (pos < lens[:, None])).long()
    data = dict(input_ids=torch.randint(0, 100, (bs, L), generator=g), attention_mask=am, loss_mask=lm,
                logprobs=-torch.rand(bs, L, generator=g) * 2, rewards=torch.randn(bs, generator=g) * 3)
    if case == "grpo":
        kw = dict(reward_scaling=2.0, reward_bias=-0.5, reward_clip=4.0,
                  reward_norm=dict(mean_level="group", std_level="group", group_size=4),
                  adv_norm=dict(mean_level="batch", std_level="batch"))
    elif case == "critic_kl":
        data["values"] = torch.randn(bs, L, generator=g) * 0.3
        data["ref_logp"] = -torch.rand(bs, L, generator=g) * 2
        kw = dict(kl_ctl=0.1, kl_estimator="k3", discount=0.99, gae_lambda=0.95, mask_no_eos_with_zero=True,
                  use_decoupled_loss=True, adv_norm=dict(mean_level="batch", std_level=None, mean_leave1out=True))
    elif case == "overlong":
        kw = dict(overlong_tokens=16, overlong_penalty_factor=0.7, max_new_tokens=48,
                  adv_norm=dict(mean_level="batch", std_level="batch"))
    else:
        data["prox_logp"] = -torch.rand(bs, L, generator=g) * 2
        kw = dict(recompute_logprob=True, use_decoupled_loss=False)
    want = O.compute_advantages({k: (v.clone() if torch.is_tensor(v) else v) for k, v in data.items()}, **kw)
    gkw = dict(kw)
    for name in ("reward_norm", "adv_norm"):
        if gkw.get(name) is not None:
            gkw[name] = Normalization(NormConfig(**gkw[name]))
    got = compute_advantages({k: (v.to(device) if torch.is_tensor(v) else v) for k, v in data.items()}, **gkw)
    for key in ("advantages", "returns", "kl_rewards", "tot_rewards", "loss_mask", "logprobs"):
        scale = float(want[key].abs().max()) + 1.0
        assert float((got[key].cpu() - want[key]).abs().max()) < 2e-5 * scale, key
    rolled_mask = torch.roll(lm.float(), shifts=-1, dims=-1)
    if case != "critic_kl":
        # the reference masks old_logp in place (actor.py:195), and data["prox_logp"] is that very tensor
        assert torch.allclose(got["prox_logp"].cpu(), want["prox_logp"])
        assert got["prox_logp"] is got["logprobs"]
        assert float((got["prox_logp"].cpu() * (1 - rolled_mask)).abs().max()) == 0.0
    else:
        # ... and data["ref_logp"] likewise (actor.py:194)
        assert torch.equal(want["ref_logp"], data["ref_logp"] * rolled_mask)
        assert torch.equal(got["ref_logp"].cpu(), want["ref_logp"])


def test_overlong_penalty_matches_oracle_and_updates_in_place(device):
    g = torch.Generator().manual_seed(8)
    bs, L = 37, 300
    lens = torch.randint(1, L + 1, (bs,), generator=g)
    mask = (torch.arange(L)[None, :] < lens[:, None]).float()
    rewards = torch.randn(bs, generator=g)
    want = O.overlong_penalty(dict(rewards=rewards.clone(), loss_mask=mask, input_ids=torch.zeros(bs, L)), 40, 1.3, 200)
    r_dev = rewards.to(device)
    data = dict(rewards=r_dev, loss_mask=mask.to(device), input_ids=torch.zeros(bs, L, device=device))
    got = areal_amd.reward_overlong_penalty(data, 40, 1.3, 200)
    assert got["rewards"] is r_dev and torch.equal(r_dev.cpu(), want["rewards"])
    assert bool((want["rewards"] <= rewards).all()) and bool((want["rewards"] < rewards).any())


@pytest.mark.parametrize("shape,dim", [((2_000_003,), None), ((64, 4096), None), ((64, 4096), 1), ((64, 4096), 0),
                                       ((5, 7, 33), (0, 2)), ((3, 1), None), ((1,), None)])
@pytest.mark.parametrize("masked,unbiased", [(False, False), (True, True), (True, False)])
def test_masked_normalization_matches_oracle(device, shape, dim, masked, unbiased):
    g = torch.Generator().manual_seed(13)
    x = torch.randn(shape, generator=g) * 3 + 1.5
    mask = (torch.rand(shape, generator=g) < 0.7) if masked else None
    want = O.masked_normalization(x, mask, dim, unbiased, 1e-5)
    got = areal_amd.masked_normalization(x.to(device), None if mask is None else mask.to(device), dim, unbiased, 1e-5)
    assert got.dtype == torch.float32 and got.shape == x.shape
    # a single value (or a single selected value with Bessel's correction) divides by zero in both
    assert torch.allclose(got.cpu(), want, rtol=1e-5, atol=1e-6, equal_nan=True)


def test_masked_normalization_weights_and_broadcast_mask(device):
    g = torch.Generator().manual_seed(14)
    x = torch.randn(16, 300, generator=g)
    w = torch.rand(16, 1, generator=g)                      # a float mask that broadcasts over the row
    want = O.masked_normalization(x, w.expand_as(x), 1, False, 1e-3)
    got = areal_amd.masked_normalization(x.to(device), w.to(device), dim=1, eps=1e-3)
    assert torch.allclose(got.cpu(), want, rtol=1e-5, atol=1e-6)
    got16 = areal_amd.masked_normalization(x.to(device).bfloat16(), None, dim=-1)
    assert torch.allclose(got16.cpu(), O.masked_normalization(x.bfloat16(), None, 1), rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("estimator", ["k1", "k2", "k3"])
@pytest.mark.parametrize("clamp", [True, False])
def test_kl_estimator_matches_oracle(device, estimator, clamp):
    from oracle import kl_estimate

    g = torch.Generator().manual_seed(2)
    a = -torch.rand(4, 333, generator=g) * 5
    b = a + torch.randn(4, 333, generator=g) * 3          # differences large enough for the clamp to bind
    b[0, 0] = a[0, 0] - 40.0                              # k3 overflows the clamp by far
    want = kl_estimate(a, b, estimator)
    if clamp:
        want = want.clamp(min=-10, max=10)                # data.py:1654-1655
    got = areal_amd.KLEstimator(estimator, clamp)(a.to(device), b.to(device))
    assert got.shape == a.shape and torch.allclose(got.cpu(), want, rtol=2e-6, atol=1e-6)
    # the numbers the reference's tests quote (tests/test_rejection_sampling.py:507-546): log-ratios 0.5, -0.5, 2.0
    d = torch.tensor([0.5, -0.5, 2.0], device=device)
    val = areal_amd.KLEstimator(estimator, clamp)(d, torch.zeros(3, device=device)).tolist()
    quoted = {"k1": [0.5, -0.5, 2.0], "k2": [0.125, 0.125, 2.0], "k3": [0.1065, 0.1487, 1.1353]}[estimator]
    assert val == pytest.approx(quoted, abs=1e-4)
    with pytest.raises(ValueError, match="Invalid KL estimator"):
        areal_amd.KLEstimator("k4")


@pytest.mark.parametrize("n", [1, 63, 2048, 2049, 131072, 300001])
def test_moments_under_masks_of_their_own(device, n):
    """One workgroup per tensor, several slices, and more slices than one round of them; float and byte tensors, a mask
    each or none, an empty mask; twice on one work buffer, bit-equal; and the 16-tensor entry point of the C ABI.  Sums
    are fp64 sums rounded once to float32: 2^-23 of the sum of magnitudes."""
    import ctypes

    from areal_amd import _native as N
    from areal_amd.advantages import moments_table

    g = torch.Generator().manual_seed(n)
    x, y = torch.randn(n, generator=g), 3.0 + torch.randn(n, generator=g)
    flag = torch.rand(n, generator=g) < 0.2
    m1, m2, none = torch.rand(n, generator=g) < 0.6, torch.rand(n, generator=g) < 0.1, torch.zeros(n, dtype=torch.bool)
    cpu = [("x", x, m1), ("y", y, m2), ("all", y, None), ("flag", flag, m1), ("flag_all", flag, None), ("empty", x, none)]
    entries = [(k, t.to(device), None if m is None else m.to(device)) for k, t, m in cpu]
    got, again = moments_table(entries), moments_table(entries)
    for name, t, m in cpu:
        v = t.double() if m is None else t.double()[m]
        r = {k: float(c) for k, c in got[name].items()}
        assert r["count"] == v.numel()
        assert abs(r["sum"] - float(v.sum())) <= 2.0 ** -23 * float(v.abs().sum()) + 1e-30
        assert r["min"] == (float(v.min()) if v.numel() else float("inf"))
        assert r["max"] == (float(v.max()) if v.numel() else float("-inf"))
        assert (r["avg"] != r["avg"]) if v.numel() == 0 else abs(r["avg"] - r["sum"] / r["count"]) <= 2.0 ** -23 * abs(r["avg"])
        for k in r:
            assert torch.equal(got[name][k], again[name][k]) or v.numel() == 0
    lib, dev_x, dev_y, dev_m = N.load(), x.to(device), y.to(device), m1.to(device)
    out = torch.empty(2, 4, device=device)
    ptrs = (ctypes.c_void_p * 2)(dev_x.data_ptr(), dev_y.data_ptr())
    N.check(lib.aa_masked_moments(ptrs, 2, dev_m.data_ptr(), n, out.data_ptr(), torch.cuda.current_stream().cuda_stream), "aa_masked_moments")
    want = O.masked_moments([x, y], m1)
    assert torch.equal(out[:, 1:].cpu(), want[:, 1:])
    bound = 2.0 ** -23 * torch.stack([v.double()[m1].abs().sum() for v in (x, y)])
    assert bool(((out[:, 0].cpu().double() - want[:, 0].double()).abs() <= bound + 1e-30).all())


@pytest.mark.parametrize("bs,L", [(1, 1), (3, 2), (7, 17), (4, 4096), (5, 4097), (4, 4098), (6, 9000), (300, 33)])
@pytest.mark.parametrize("variant", ["batch", "group", "group mean, batch deviation", "no normalisation", "recomputed"])
def test_advantage_rows_agree_with_the_separate_kernels(device, bs, L, variant):
    """The one-pass kernel (one block of positions, edges, several; rows past the last full group) against the
    separate rolls, products, KL, GAE and two-pass normalisation, which an adv_norm that is no ``Normalization`` takes.
    What moves and multiplies is bit-equal; so are advantages and returns (the same scan); normalised advantages differ
    by the rounding of float64 sums in another order, then once to float32: 4 ulps of the largest."""
    from areal_amd import engine_glue

    g = torch.Generator().manual_seed(bs * 10007 + L)
    lens = torch.randint(1, L + 1, (bs, 1), generator=g)
    at = torch.arange(L)[None]
    attention = at < lens
    mask = attention & (torch.rand(bs, L, generator=g) < 0.7)
    logp = -2.0 * torch.rand(bs, L, generator=g)
    base = dict(attention_mask=attention, loss_mask=mask if L % 2 else mask.float(), logprobs=logp,
                rewards=torch.randn(bs, generator=g), prox_logp=logp + 0.05 * torch.randn(bs, L, generator=g))
    if variant != "no normalisation":
        base["ref_logp"] = logp + 0.05 * torch.randn(bs, L, generator=g)
    if variant in ("batch", "recomputed"):
        base["values"] = torch.randn(bs, L, generator=g) + 3.0
    cfg = {"group": dict(mean_level="group", std_level="group", group_size=4),
           "group mean, batch deviation": dict(mean_level="group", std_level="batch", group_size=4),
           "no normalisation": None}.get(variant, dict(mean_level="batch", std_level="batch"))
    norm = None if cfg is None else Normalization(NormConfig(**cfg))
    reward = Normalization(NormConfig(mean_level="group", mean_leave1out=True, std_level="batch", group_size=4))
    kw = dict(kl_ctl=0.1, kl_estimator="k3", discount=0.99, gae_lambda=0.95, reward_bias=0.1, reward_scaling=2.0,
              use_decoupled_loss=variant != "recomputed", recompute_logprob=variant == "recomputed")

    def run(adv_norm, reward_norm):
        data = {k: v.clone().to(device) for k, v in base.items()}
        return engine_glue.compute_advantages(data, adv_norm=adv_norm, reward_norm=reward_norm, **kw)

    got, again = run(norm, reward), run(norm, reward)
    want = run(lambda x, m: x.clone() if norm is None else norm(x, m), lambda x: reward(x))
    for k in ("loss_mask", "logprobs", "prox_logp", "ref_logp", "kl_rewards", "tot_rewards", "returns", "advantages"):
        if k not in want:
            continue
        a, b = got[k], want[k]
        assert torch.equal(got[k], again[k]) and a.dtype == b.dtype and a.shape == b.shape, k
        if k == "advantages" and norm is not None:
            assert float((a - b).abs().max()) <= 4 * 2.0 ** -23 * max(float(b.abs().max()), 1.0), k
        elif k in ("tot_rewards", "returns", "advantages"):  # the reward scores go through float64 sums of another order
            assert float((a - b).abs().max()) <= 4 * 2.0 ** -23 * max(float(b.abs().max()), 1.0), k
        else:
            assert torch.equal(a, b), k


@pytest.mark.parametrize("bs,group", [(1, 1), (7, 3), (12, 1), (32, 16), (130, 64), (64, 65), (5, 8)])
@pytest.mark.parametrize("levels", [None, ("group", False, "group", False), ("group", True, "group", True), ("group", False, None, False),
                                    (None, False, "group", True), (None, False, None, False)])
@pytest.mark.parametrize("lengths", [False, True])
def test_scores_formed_by_the_advantage_rows(device, bs, group, levels, lengths):
    """The reward scores of the one-pass kernel against those of a launch of their own (``reward_scores``): the same sums in
    the same order, so the same bits; rows past the last full group, groups up to a wave and one row more (which takes the
    other way); lengths from an attention mask of bytes or as numbers."""
    from areal_amd import engine_glue
    from areal_amd.advantages import advantage_rows, reward_scores, score_step

    g = torch.Generator().manual_seed(bs * 100 + group)
    L = 37
    attention = (torch.arange(L)[None] < torch.randint(1, L + 1, (bs, 1), generator=g)).to(device)
    attention = attention.long() if lengths else attention
    mask = (torch.rand(bs, L, generator=g) < 0.7).to(device)
    logp = (-2.0 * torch.rand(bs, L, generator=g)).to(device)
    rewards = (3.0 * torch.randn(bs, generator=g)).to(device)
    norm = None
    if levels is not None:
        norm = Normalization(NormConfig(mean_level=levels[0], mean_leave1out=levels[1], std_level=levels[2],
                                        std_unbiased=levels[3], group_size=group))
    args = (rewards, -0.5, 2.0, 5.0, norm)
    scores = score_step(*args)
    grouped = levels is not None and "group" in levels
    assert (scores is None) == (grouped and group > 64)

    def rows(score, step=None):
        return advantage_rows(mask, logp, True, None, attention, score, None, 0.1, "k1", 1.0, 0.95, False, None, step)

    want = rows(reward_scores(*args))
    data = dict(attention_mask=attention, loss_mask=mask, logprobs=logp, rewards=rewards)
    out = engine_glue.compute_advantages(data, kl_ctl=0.1, gae_lambda=0.95, reward_bias=-0.5, reward_scaling=2.0,
                                         reward_clip=5.0, reward_norm=norm)
    assert torch.equal(out["tot_rewards"], want[3]) and torch.equal(out["advantages"], want[4])
    if scores is not None:
        for a, b in zip(rows(rewards, scores), want):
            assert torch.equal(a, b)


@pytest.mark.parametrize("bs,L,offset", [(5, 1021, 0), (5, 1022, 0), (3, 1025, 0), (5, 2045, 0), (5, 2047, 0), (4, 2048, 0),
                                         (3, 2051, 0), (3, 6143, 0), (1030, 5, 0), (2050, 1022, 0), (5, 61, 1), (3, 2049, 3),
                                         (3, 1024, 0), (3, 1028, 1), (3, 1277, 0), (3, 1278, 2), (3, 1533, 0), (3, 1534, 0),
                                         (3, 1790, 1), (3, 2052, 0), (3, 2557, 3), (3, 4095, 0), (3, 4096, 1), (3, 4100, 0),
                                         (1024, 2049, 1), (1024, 2051, 0), (4096, 1027, 3)])
@pytest.mark.parametrize("gamma,lam", [(1.0, 0.95), (1.0, 1.0), (0.99, 0.999)])
def test_advantage_rows_at_the_edges_of_their_blocks(device, bs, L, offset, gamma, lam):
    """Rows around the sizes of a block of 1024 and of 2048 positions, few rows and so many that they go in several blocks of
    1024, at every place in a 16-byte piece, more rows than the last workgroup holds, and arrays that do not start on 16 bytes
    (``offset`` elements into a larger one): advantages and returns against the recurrence in float64 with the float32
    factors.  The maps are composed in float64; a state is rounded once where it enters a piece of four positions and four
    times (product, two sums with reward and value, sum with the last advantage) at each of them: 17 times 2^-24 of the
    largest state, reward and value.  Over all tokens it is a few times less: 2^-22 of the 2-norm (a composition in float32 is
    off by 4e-7 for lam = 1 and 1e-6 for gamma lam = 0.989)."""
    from areal_amd import engine_glue

    g = torch.Generator().manual_seed(bs + L)
    lens = torch.randint((L + 1) // 2, L + 1, (bs, 1), generator=g)
    at = torch.arange(L)[None]
    attention = at < lens
    mask = attention & (torch.rand(bs, L, generator=g) < 0.8)
    logp = -2.0 * torch.rand(bs, L, generator=g)
    base = dict(attention_mask=attention, loss_mask=mask, logprobs=logp, rewards=torch.randn(bs, generator=g),
                ref_logp=logp + 0.05 * torch.randn(bs, L, generator=g), prox_logp=logp.clone(),
                values=torch.randn(bs, L, generator=g))

    def placed(t):
        if offset == 0 or t.dim() != 2:
            return t.clone().to(device)
        flat = torch.empty(t.numel() + offset, dtype=t.dtype, device=device)
        flat[offset:] = t.flatten().to(device)
        return flat[offset:].view(t.shape)

    kw = dict(kl_ctl=0.1, kl_estimator="k1", discount=gamma, gae_lambda=lam, use_decoupled_loss=True)
    out = engine_glue.compute_advantages({k: placed(v) for k, v in base.items()}, **kw)
    norm = Normalization(NormConfig(mean_level="batch", std_level="batch"))
    normed = engine_glue.compute_advantages({k: placed(v) for k, v in base.items()}, adv_norm=norm, **kw)
    m, v, r = out["loss_mask"].cpu().double(), base["values"].double(), out["tot_rewards"].cpu().double()
    no_eos = (lens[:, 0] == L)
    nv, lg = torch.where(no_eos, v[:, -1], 0.0), torch.zeros(bs, dtype=torch.float64)
    adv, biggest = torch.zeros(bs, L, dtype=torch.float64), 1.0
    f32 = lambda x: float(torch.tensor(x, dtype=torch.float32))
    gamma, gl = f32(gamma), f32(f32(gamma) * f32(lam))
    for t in range(L - 2, -1, -1):
        new = r[:, t] + gamma * nv - v[:, t] + gl * lg
        nv, lg = torch.where(m[:, t] > 0, v[:, t], nv), torch.where(m[:, t] > 0, new, lg)
        adv[:, t] = lg
        biggest = max(biggest, float(lg.abs().max()))
    bound = 17 * 2.0 ** -24 * (biggest + float(r.abs().max()) + 2 * float(v.abs().max()))
    assert float((out["advantages"].cpu().double() - adv).norm()) <= 2.0 ** -22 * float(adv.norm())
    assert float((out["advantages"].cpu().double() - adv).abs().max()) <= bound
    ret = adv + v
    assert float((out["returns"].cpu().double() - ret).abs().max()) <= bound + 2.0 ** -24 * float(ret.abs().max())
    # the separate two-pass normalisation of the same advantages: float64 sums in another order, then one rounding to float32
    want = norm(out["advantages"], out["loss_mask"])
    assert float((normed["advantages"] - want).abs().max()) <= 4 * 2.0 ** -23 * max(float(want.abs().max()), 1.0)


@pytest.mark.parametrize("bs,L", [(1, 1), (1, 3), (3, 2047), (257, 5), (513, 9), (700, 2051), (1024, 33), (1025, 33), (9, 4097)])
@pytest.mark.parametrize("std_unbiased", [True, False])
@pytest.mark.parametrize("masked", [0.0, 0.6, 1.0])
def test_batch_normalisation_from_the_sums_of_the_rows(device, bs, L, std_unbiased, masked):
    """Up to 1 024 rows the kernel that normalises folds their sums itself: sizes either side of a thread's rows, of a piece of
    four elements and of that limit, with nothing and everything under the mask, against the separate two-pass normalisation of
    the same advantages.  float64 sums in another order, then one rounding to float32: 4 ulps of the largest."""
    from areal_amd import engine_glue

    g = torch.Generator().manual_seed(bs * 101 + L)
    mask = torch.rand(bs, L, generator=g) >= masked if masked < 1.0 else torch.zeros(bs, L, dtype=torch.bool)
    data = dict(attention_mask=torch.ones(bs, L, dtype=torch.bool), loss_mask=mask, logprobs=-torch.rand(bs, L, generator=g),
                values=torch.randn(bs, L, generator=g) + 2.0, rewards=torch.rand(bs, generator=g))
    norm = Normalization(NormConfig(mean_level="batch", std_level="batch", std_unbiased=std_unbiased))

    def run(adv_norm):
        d = {k: v.clone().to(device) for k, v in data.items()}
        return engine_glue.compute_advantages(d, adv_norm=adv_norm, discount=0.99, gae_lambda=0.95, use_decoupled_loss=True)

    plain, got, again = run(None), run(norm)["advantages"], run(norm)["advantages"]
    want = norm(plain["advantages"], plain["loss_mask"])
    assert torch.equal(got, again)
    assert float((got - want).abs().max()) <= 4 * 2.0 ** -23 * max(float(want.abs().max()), 1.0)


@pytest.mark.parametrize("bs,L", [(1, 64), (3, 33), (3, 1025), (3, 4097)])
@pytest.mark.parametrize("levels", [("group", "batch"), ("group", None), ("group", "group"), (None, "group"), ("batch", "group"),
                                    (None, "batch"), ("batch", "batch")])
def test_normalised_advantage_rows_of_a_batch_smaller_than_a_group(device, bs, L, levels):
    """No group is full, so a mean of the group is no mean (0), in the squares of a batch-wide deviation as well.  The
    one-pass kernel against the separate two-pass normalisation and against the oracle, with advantages far from their
    mean: float64 sums in another order, then one rounding to float32, 4 ulps of the largest."""
    from areal_amd import engine_glue

    g = torch.Generator().manual_seed(bs + L)
    mask = torch.rand(bs, L, generator=g) < 0.8
    data = dict(attention_mask=torch.ones(bs, L, dtype=torch.bool), loss_mask=mask, logprobs=-torch.rand(bs, L, generator=g),
                values=-4.0 + torch.rand(bs, L, generator=g), rewards=torch.rand(bs, generator=g))
    cfg = dict(mean_level=levels[0], std_level=levels[1], group_size=4)
    norm = Normalization(NormConfig(**cfg))

    def run(adv_norm):
        d = {k: v.clone().to(device) for k, v in data.items()}
        return engine_glue.compute_advantages(d, adv_norm=adv_norm, discount=0.0, gae_lambda=0.0, use_decoupled_loss=True)

    plain, got, want = run(None), run(norm)["advantages"], run(lambda x, m: norm(x, m))["advantages"]
    counted = plain["advantages"][plain["loss_mask"].bool()]
    assert counted.numel() > L // 4 and float(counted[counted != 0].abs().min()) > 1.0
    bound = 4 * 2.0 ** -23 * max(float(want.abs().max()), 1.0)
    assert float(want.abs().max()) > 0.5 and float((got - want).abs().max()) <= bound
    by_oracle = O.normalization(plain["advantages"].cpu(), plain["loss_mask"].cpu(), mean_leave1out=False, std_unbiased=True,
                                eps=1e-5, **cfg)
    assert float((got.cpu() - by_oracle).abs().max()) <= 2e-6 * (float(by_oracle.abs().max()) + 1.0)


@pytest.mark.parametrize("shared", ["ref_logp is logprobs", "ref_logp is values", "prox_logp is values"])
def test_advantages_of_arrays_that_share_memory(device, shared):
    """Log-probs are masked in place: with a second role for the same memory the result is that of separate kernels that
    run one after the other, and autograd's version of what was written goes up."""
    from areal_amd import engine_glue

    bs, L = 5, 300
    g = torch.Generator().manual_seed(3)
    lens = torch.randint(L // 2, L + 1, (bs, 1), generator=g)
    attention = torch.arange(L)[None] < lens
    mask = attention & (torch.rand(bs, L, generator=g) < 0.7)
    one, two, three = (-2.0 * torch.rand(bs, L, generator=g) for _ in range(3))
    score = torch.randn(bs, generator=g)
    recomputed = shared.startswith("prox_logp")

    def run(reward_norm):
        a, b, c = (t.clone().to(device) for t in (one, two, three))
        data = dict(attention_mask=attention.to(device), loss_mask=mask.to(device), rewards=score.to(device), logprobs=a,
                    ref_logp=b, prox_logp=c, values=torch.zeros(bs, L, device=device))
        first, second = shared.split(" is ")
        data[first] = data[second] = data[first]
        before = b._version
        out = engine_glue.compute_advantages(data, kl_ctl=0.1, adv_norm=None, reward_norm=reward_norm, gae_lambda=0.9,
                                             use_decoupled_loss=not recomputed, recompute_logprob=recomputed)
        assert data["ref_logp"]._version > (before if data["ref_logp"] is b else 0)
        return {k: out[k].clone() for k in ("logprobs", "ref_logp", "kl_rewards", "tot_rewards", "returns", "advantages")}

    got = run(None)
    # masks, products and KL by torch, in the order of the reference
    a, b, c = one.clone(), two.clone(), three.clone()
    arrays = dict(logprobs=a, ref_logp=b, prox_logp=c, values=torch.zeros(bs, L))
    first, second = shared.split(" is ")
    arrays[first] = arrays[second] = arrays[first]
    m = torch.roll(mask.float(), -1, -1)
    old = arrays["prox_logp"] if recomputed else torch.roll(arrays["logprobs"], -1, -1)
    old.mul_(m)
    arrays["ref_logp"].mul_(m)
    assert torch.equal(got["logprobs"].cpu(), old) and torch.equal(got["ref_logp"].cpu(), arrays["ref_logp"])
    rewards = got["tot_rewards"]
    adv, ret = areal_amd.gae_advantages(rewards, arrays["values"].to(device), m.to(device),
                                        (lens.squeeze(1) == L).to(device), 1.0, 0.9)
    assert torch.equal(got["advantages"], adv) and torch.equal(got["returns"], ret)
    want = -0.1 * (old - arrays["ref_logp"])  # one product and one difference of float32: 2 ulps
    assert float((got["kl_rewards"].cpu() - want).abs().max()) <= 2 * 2.0 ** -23 * float(want.abs().max())


def test_moments_in_a_graph_beside_eager_ones(device):
    """The counters that the workgroups of a launch share are the graph's own: nothing that was captured stays in the
    buffer kept for eager calls, and replays give the eager result."""
    from areal_amd import functional
    from areal_amd.advantages import moments_table

    n = 300001
    x, m = torch.zeros(n, device=device), torch.zeros(n, dtype=torch.bool, device=device)
    N = functional.N
    N.load()
    kept = dict(functional._WORK)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = moments_table([("x", x, m), ("all", x, None)])
    assert functional._WORK.keys() == kept.keys()
    for seed in (1, 2, 3):
        g = torch.Generator().manual_seed(seed)
        x.copy_(torch.randn(n, generator=g))
        m.copy_(torch.rand(n, generator=g) < 0.4)
        graph.replay()
        torch.cuda.synchronize()
        eager = moments_table([("x", x, m), ("all", x, None)])
        for name in eager:
            for k in eager[name]:
                assert torch.equal(eager[name][k], captured[name][k]), (seed, name, k)


@pytest.mark.parametrize("levels", [("group", "batch"), (None, "batch"), (None, "group"), ("batch", "batch"),
                                    ("batch", "group"), ("group", "group")])
@pytest.mark.parametrize("L", [60, 5000])
@pytest.mark.parametrize("what", ["nan", "inf", "-inf"])
def test_advantages_that_are_not_finite_reach_the_deviation(device, levels, L, what):
    """A NaN or an infinity in one row (at its first position, the last one of the scan, so that it does not spread along
    the row by itself) does to every other row what it does in the separate kernels: in a mean or deviation that it enters
    it stays, the rest of the batch agrees to the rounding of sums in another order."""
    from areal_amd import engine_glue

    bs = 12
    g = torch.Generator().manual_seed(L)
    values = torch.randn(bs, L, generator=g)
    big = {"nan": float("nan"), "inf": -3e38, "-inf": 3e38}[what]
    values[5, 0], values[5, 1] = big, (0.0 if what == "nan" else -big)
    mask = torch.rand(bs, L, generator=g) < 0.7
    mask[5, 1:3] = True  # after the roll: positions 0 and 1 count
    logp = -torch.rand(bs, L, generator=g)
    data = dict(attention_mask=torch.ones(bs, L, dtype=torch.bool), loss_mask=mask, logprobs=logp, values=values,
                rewards=torch.randn(bs, generator=g))
    norm = Normalization(NormConfig(mean_level=levels[0], std_level=levels[1], group_size=4))
    kw = dict(kl_ctl=0.1, discount=0.99, gae_lambda=0.0, use_decoupled_loss=True)

    def run(adv_norm):
        return engine_glue.compute_advantages({k: v.clone().to(device) for k, v in data.items()}, adv_norm=adv_norm, **kw)

    plain = run(None)["advantages"]
    hit = plain[5, 0].isnan() if what == "nan" else plain[5, 0] == float(what)
    assert bool(hit) and int((~plain.isfinite()).sum()) == 1
    got, want = run(norm)["advantages"], run(lambda x, m: norm(x, m))["advantages"]
    assert torch.allclose(got, want, rtol=1e-6, atol=1e-6, equal_nan=True)


def test_advantages_of_one_array_as_both_policies(device):
    """Recomputed log-probs that are also the reference policy's are masked twice, as in the reference: with a mask of
    fractions that shows."""
    from areal_amd import engine_glue

    bs, L = 4, 33
    g = torch.Generator().manual_seed(8)
    mask, one = torch.rand(bs, L, generator=g), -torch.rand(bs, L, generator=g)
    shared = one.clone().to(device)
    data = dict(attention_mask=torch.ones(bs, L, dtype=torch.bool, device=device), loss_mask=mask.to(device),
                logprobs=one.to(device), prox_logp=shared, ref_logp=shared, rewards=torch.zeros(bs, device=device))
    engine_glue.compute_advantages(data, use_decoupled_loss=False, recompute_logprob=True)
    m = torch.roll(mask, -1, -1)
    assert torch.equal(shared.cpu(), one * m * m)


def test_reward_scores_with_a_bias_per_sequence(device):
    """Bias, scaling and clip may be tensors, as in the torch expressions of the reference."""
    from areal_amd import engine_glue

    bs, L = 6, 12
    g = torch.Generator().manual_seed(5)
    bias, scaling = torch.randn(bs, generator=g), torch.rand(bs, generator=g)
    data = dict(attention_mask=torch.ones(bs, L, dtype=torch.bool), loss_mask=torch.ones(bs, L, dtype=torch.bool),
                logprobs=torch.zeros(bs, L), rewards=torch.randn(bs, generator=g))
    norm = Normalization(NormConfig(mean_level="group", std_level="group", group_size=3))
    for reward_norm in (None, norm):
        out = engine_glue.compute_advantages({k: v.clone().to(device) for k, v in data.items()}, reward_bias=bias.to(device),
                                             reward_scaling=scaling.to(device), reward_norm=reward_norm)
        want = (data["rewards"] + bias) * scaling
        if reward_norm is not None:
            want = O.normalization(want, None, mean_level="group", std_level="group", group_size=3, eps=1e-5)
        assert torch.allclose(out["tot_rewards"][:, L - 2].cpu(), want, rtol=1e-5, atol=1e-6)


@pytest.mark.parametrize("bs,inner,gs", [(512, 1, 16), (2049, 1, 8), (3000, 1, 63), (3000, 1, 64), (3001, 1, 65), (8, 1024, 4),
                                         (8, 1023, 3), (4097, 1, 1), (8192, 1, 4096), (8192, 1, 2), (1, 5120, 1)])
@pytest.mark.parametrize("masked", [False, True])
def test_normalization_of_a_few_thousand_values(device, bs, inner, gs, masked):
    """Either side of the line between one launch and several, groups of less than, as many as and more than a wave, rows
    past the last group; a group mean with a batch-wide deviation, where long groups used to be summed once per value
    ([8, 1024] in groups of 4: 10.6 ms).  The float32 output has one rounding; 2e-6 of the largest, as above."""
    from areal_amd import engine_glue

    g = torch.Generator().manual_seed(bs + inner)
    x = torch.randn(bs, inner, generator=g) * 2.0 + 0.5
    mask = (torch.rand(bs, inner, generator=g) < 0.6).float() if masked else None
    for mean, std, loo in (("group", "batch", False), ("group", "batch", True), ("batch", "batch", False), ("group", "group", False),
                           (None, "batch", False), ("batch", "group", True)):
        cfg = dict(mean_level=mean, std_level=std, mean_leave1out=loo, eps=1e-5, group_size=gs)
        want = O.normalization(x, mask, **cfg)
        norm = Normalization(NormConfig(**cfg))
        got = norm(x.to(device), None if mask is None else mask.to(device)).cpu()
        assert float((got - want).abs().max()) <= 2e-6 * (float(want.abs().max()) + 1.0), cfg
        if inner == 1 and not masked:  # the same as reward scores: two positions, the scores land on the first
            data = dict(attention_mask=torch.ones(bs, 2, dtype=torch.bool), loss_mask=torch.ones(bs, 2, dtype=torch.bool),
                        logprobs=torch.zeros(bs, 2), rewards=x[:, 0].clone())
            out = engine_glue.compute_advantages({k: v.to(device) for k, v in data.items()}, reward_norm=norm)
            got = out["tot_rewards"][:, 0].cpu()
            assert float((got - want[:, 0]).abs().max()) <= 2e-6 * (float(want.abs().max()) + 1.0), cfg


def test_group_means_with_a_batch_deviation_are_linear_in_the_values(device):
    """[8, 1024] in groups of 4 rows: some 20 us a call; summing a value's whole group per value took 10 ms."""
    x, m = torch.randn(8, 1024, device=device), torch.ones(8, 1024, device=device)
    norm = Normalization(NormConfig(mean_level="group", std_level="batch", group_size=4))
    begin, end = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    norm(x, m)
    begin.record()
    for _ in range(20):
        norm(x, m)
    end.record()
    end.synchronize()
    assert begin.elapsed_time(end) < 20 * 2.0


def test_masked_moments_read_their_mask_once(device, monkeypatch):
    """A mask that is not bool is converted once, not once per tensor."""
    from areal_amd import advantages as A
    from areal_amd import functional as F

    n, calls = 777, []
    g = torch.Generator().manual_seed(2)
    mask = (torch.rand(n, generator=g) < 0.5).long()
    values = {f"v{i}": torch.randn(n, generator=g) for i in range(5)}
    plain = F._mask_u8
    monkeypatch.setattr(F, "_mask_u8", lambda m: calls.append(m.dtype) or plain(m))
    got = A.masked_moments({k: v.to(device) for k, v in values.items()}, mask.to(device))
    assert len([c for c in calls if c is not torch.bool]) <= 1
    for k, v in values.items():
        assert float(got[k]["sum"]) == pytest.approx(float(v.double()[mask.bool()].sum()), abs=1e-4)
        assert int(got[k]["count"]) == int(mask.sum())


def test_advantages_of_rows_with_a_long_masked_tail(device):
    """Rows whose last blocks (2 048 positions or fewer) have no token with a loss: the squares of such a row are taken about
    the mean of the tokens that count all the same, so a mean a million times the spread costs no digits."""
    from areal_amd import engine_glue

    bs, L = 6, 9000
    g = torch.Generator().manual_seed(4)
    mask = torch.zeros(bs, L, dtype=torch.bool)
    mask[:, 1:3001] = True
    data = dict(attention_mask=torch.ones(bs, L, dtype=torch.bool), loss_mask=mask, logprobs=torch.zeros(bs, L),
                values=-4096.0 - 2.0 ** -8 * torch.rand(bs, L, generator=g), rewards=torch.zeros(bs))
    for levels in (("batch", "batch"), ("group", "group")):
        norm = Normalization(NormConfig(mean_level=levels[0], std_level=levels[1], group_size=3, eps=0.0))

        def run(adv_norm):
            d = {k: v.clone().to(device) for k, v in data.items()}
            return engine_glue.compute_advantages(d, adv_norm=adv_norm, discount=0.0, gae_lambda=0.0, use_decoupled_loss=True)

        got, want = run(norm)["advantages"], run(lambda x, m: norm(x, m))["advantages"]
        # the float64 rounding of a shifted sum of squares would be 2^-53 (mean / spread)^2, some 1e-4; what remains is
        # that of the sums, then one rounding to float32
        assert float((got - want).abs().max()) <= 4 * 2.0 ** -23 * float(want.abs().max())
