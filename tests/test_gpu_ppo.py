"""GPU parity of apply_rejection_sampling and ppo_actor_loss_fn against the oracle and against the
reference's own known-answer cases."""
import itertools
import math

import pytest
import torch

import areal_amd
import oracle
from areal_amd import RejectionSamplingConfig
from helpers import cosine
from test_oracle_pins import _ppo_case_tensors, _run_rs_case, check_ppo_expectations, check_rs_expectations

pytestmark = pytest.mark.gpu


def _to(dev, *ts):
    return [None if t is None else t.to(dev) for t in ts]


def test_rejection_sampling_reference_known_answers(device, known_answers):
    def fn(prox, old, mask, cu, cfg):
        return areal_amd.apply_rejection_sampling(*_to(device, prox, old, mask, cu), cfg)

    for case in known_answers["rejection_sampling"]:
        check_rs_expectations(case, _run_rs_case(case, fn, RejectionSamplingConfig))


def test_ppo_loss_reference_known_answers(device, known_answers):
    for case in known_answers["ppo_actor_loss"]:
        lp, prox, old, adv, mask, cu = _to(device, *_ppo_case_tensors(case))
        loss, stat = areal_amd.ppo_actor_loss_fn(
            lp, prox, old, adv, case["eps_clip"], mask, importance_sampling_level=case["level"], cu_seqlens=cu
        )
        check_ppo_expectations(case, loss.cpu(), {k: (v.cpu() if torch.is_tensor(v) else v) for k, v in stat.items()})


def _random_packed(seed, n_seqs=9, lo=1, hi=40, all_masked_seq=True):
    g = torch.Generator().manual_seed(seed)
    lengths = torch.randint(lo, hi + 1, (n_seqs,), generator=g).tolist()
    T = sum(lengths)
    cu = torch.tensor([0] + list(itertools.accumulate(lengths)), dtype=torch.int32)
    prox = -2 + 0.5 * torch.randn(T, generator=g)
    old = prox + 0.6 * torch.randn(T, generator=g)
    lp = prox + 0.3 * torch.randn(T, generator=g)
    adv = torch.randn(T, generator=g)
    mask = torch.rand(T, generator=g) < 0.7
    if all_masked_seq:
        mask[int(cu[2]) : int(cu[3])] = False
    return lengths, cu, lp, prox, old, adv, mask


RS_GRID = [
    dict(level=lv, action=ac, metric=me, agg=ag, upper=up, lower=lo)
    for lv in ("token", "sequence")
    for ac, me in (("mask", "ratio"), ("mask", "kl_k1"), ("mask", "kl_k2"), ("mask", "kl_k3"), ("clamp", "ratio"))
    for ag in (("mean",) if lv == "token" else ("sum", "mean", "max"))
    for up, lo in (((1.6, None), (1.6, 0.7)) if me == "ratio" else ((0.15, None), (0.15, -0.2)))
]


@pytest.mark.parametrize("kw", RS_GRID, ids=lambda k: "-".join(str(v) for v in k.values()))
def test_rejection_sampling_matches_oracle_packed_and_padded(device, kw):
    cfg = RejectionSamplingConfig(**kw)
    _, cu, _, prox, old, _, mask = _random_packed(seed=17)
    prox[5] = float("-inf"); old[5] = float("-inf")  # NaN difference is sanitised (functional.py:231-233)
    for mask_t in (mask, mask.float()):
        want = oracle.rejection_sampling(prox, old, mask_t, cu, cfg)
        got = areal_amd.apply_rejection_sampling(*_to(device, prox, old, mask_t, cu), cfg)
        assert got.loss_mask.dtype == mask_t.dtype
        assert torch.equal(got.loss_mask.cpu(), want.loss_mask)                      # masks: bit-exact
        assert torch.allclose(got.behave_imp_weight.cpu(), want.behave_imp_weight, rtol=2e-6, atol=1e-7)
        assert got.filtered_fraction == pytest.approx(want.filtered_fraction, abs=1e-12)
    # 2-D padded layout
    g = torch.Generator().manual_seed(23)
    p2 = -2 + 0.5 * torch.randn(6, 11, generator=g)
    o2 = p2 + 0.6 * torch.randn(6, 11, generator=g)
    m2 = torch.rand(6, 11, generator=g) < 0.6
    m2[4] = False
    want = oracle.rejection_sampling(p2, o2, m2, None, cfg)
    got = areal_amd.apply_rejection_sampling(*_to(device, p2, o2, m2), None, cfg)
    assert torch.equal(got.loss_mask.cpu(), want.loss_mask)
    assert torch.allclose(got.behave_imp_weight.cpu(), want.behave_imp_weight, rtol=2e-6, atol=1e-7)
    assert got.filtered_fraction == pytest.approx(want.filtered_fraction, abs=1e-12)


PPO_GRID = [
    dict(eps_clip=0.2),
    dict(eps_clip=0.2, eps_clip_higher=0.28, c_clip=3.0),
    dict(eps_clip=0.1, c_clip=1.2),
    dict(eps_clip=0.2, rs=dict(level="token", metric="ratio", upper=1.5)),
    dict(eps_clip=0.2, c_clip=3.0, eps_clip_higher=0.28, rs=dict(level="token", action="clamp", metric="ratio", upper=1.5)),
    dict(eps_clip=0.2, rs=dict(level="sequence", agg="mean", metric="kl_k2", upper=0.2)),
    dict(eps_clip=0.2, rs=dict(level="sequence", action="clamp", agg="max", metric="ratio", upper=1.4, lower=0.8)),
]


@pytest.mark.parametrize("level", ["token", "sequence"])
@pytest.mark.parametrize("kw", PPO_GRID, ids=lambda k: "-".join(f"{a}={b}" for a, b in k.items() if a != "rs") + ("-rs" if "rs" in k else ""))
def test_ppo_loss_and_gradient_match_oracle(device, kw, level):
    kw = dict(kw)
    rs = kw.pop("rs", None)
    cfg = RejectionSamplingConfig(**rs) if rs else None
    _, cu, lp, prox, old, adv, mask = _random_packed(seed=29)
    for packed in (True, False):
        if packed:
            args, cu_arg = (lp, prox, old, adv, mask), cu
        else:
            n = (lp.numel() // 7) * 7
            args, cu_arg = tuple(t[:n].reshape(-1, 7) for t in (lp, prox, old, adv, mask)), None
        lp_o = args[0].clone().requires_grad_(True)
        want_loss, want = oracle.ppo_actor_loss(
            lp_o, args[1], args[2], args[3], loss_mask=args[4], rejection_sampling_cfg=cfg,
            importance_sampling_level=level, cu_seqlens=cu_arg, **kw
        )
        want_loss.backward()
        lp_d = args[0].to(device).requires_grad_(True)
        got_loss, got = areal_amd.ppo_actor_loss_fn(
            lp_d, *_to(device, args[1], args[2], args[3]), loss_mask=args[4].to(device), rejection_sampling=cfg,
            importance_sampling_level=level, cu_seqlens=None if cu_arg is None else cu_arg.to(device), **kw
        )
        (got_loss * 1.0).backward()
        assert got_loss.ndim == 0 and got_loss.dtype == torch.float32
        assert float(got_loss.detach()) == pytest.approx(float(want_loss.detach()), rel=1e-3, abs=1e-6)   # stated tolerance
        assert float(got_loss.detach()) == pytest.approx(float(want_loss.detach()), rel=2e-5, abs=1e-6)   # what it delivers
        assert set(got) == set(want)
        for k in ("clip_mask", "dual_clip_mask") + (("behave_mask",) if cfg else ()):
            assert got[k].dtype == torch.bool and torch.equal(got[k].cpu(), want[k]), k
        for k in ("loss", "importance_weight", "approx_kl") + (("behave_approx_kl", "behave_imp_weight") if cfg else ()):
            assert got[k].dtype == torch.float32 and got[k].shape == args[0].shape
            assert torch.allclose(got[k].cpu(), want[k], rtol=1e-5, atol=1e-6), k
        if cfg:
            assert got["filtered_fraction"] == pytest.approx(want["filtered_fraction"], abs=1e-12)
        assert torch.allclose(lp_d.grad.cpu(), lp_o.grad, rtol=2e-5, atol=1e-7)
        assert cosine(lp_d.grad.cpu(), lp_o.grad) > 0.99999


def test_gradient_ties_match_autograd(device):
    """Exact ties: ratio on a clip bound, zero advantage, dual-clip equality."""
    lo, hi = 1.0 - 0.25, 1.0 + 0.25   # exactly representable
    ratios = torch.tensor([lo, hi, 1.0, 2.0, 0.5, 4.0, 3.0, 1.0])
    adv = torch.tensor([1.0, -1.0, 0.0, 1.0, -1.0, -1.0, -1.0, 2.0])
    lp = ratios.log()
    # make exp(lp) land exactly on the intended ratios where that matters
    prox = torch.zeros_like(lp)
    mask = torch.ones_like(lp, dtype=torch.bool)
    lp_o = lp.clone().requires_grad_(True)
    want_loss, want = oracle.ppo_actor_loss(lp_o, prox, prox, adv, 0.25, mask, None, 3.0)
    want_loss.backward()
    lp_d = lp.to(device).requires_grad_(True)
    got_loss, got = areal_amd.ppo_actor_loss_fn(lp_d, *_to(device, prox, prox, adv), 0.25, mask.to(device), None, 3.0)
    got_loss.backward()
    same_ratio = got["importance_weight"].cpu() == want["importance_weight"]
    assert same_ratio[2] and same_ratio[7]
    # compare wherever both sides computed the same ratio bit for bit (exp may differ by an ulp elsewhere)
    assert torch.allclose(lp_d.grad.cpu()[same_ratio], lp_o.grad[same_ratio], rtol=1e-6, atol=1e-8)
    assert torch.equal(got["clip_mask"].cpu()[same_ratio], want["clip_mask"][same_ratio])
    assert torch.equal(got["dual_clip_mask"].cpu()[same_ratio], want["dual_clip_mask"][same_ratio])


def test_edge_cases(device):
    z = torch.randn(2, 4, device=device)
    none = torch.zeros(2, 4, dtype=torch.bool, device=device)
    loss, stat = areal_amd.ppo_actor_loss_fn(z.clone().requires_grad_(True), z, z, z, 0.2, none)
    assert float(loss.detach()) == 0.0 and float(stat["importance_weight"].abs().sum()) == 0.0
    assert "behave_imp_weight" not in stat and "filtered_fraction" not in stat
    with pytest.raises(ValueError, match="cu_seqlens is required for 1D tensors"):
        areal_amd.ppo_actor_loss_fn(z[0], z[0], z[0], z[0], 0.2, ~none[0], importance_sampling_level="sequence")
    with pytest.raises(AssertionError):
        areal_amd.ppo_actor_loss_fn(z, z, z, z, 0.2, ~none, c_clip=1.0)
    # sequences of length one, and a batch of one
    cu = torch.tensor([0, 1, 2, 3], dtype=torch.int32, device=device)
    t = torch.randn(3, device=device)
    loss, stat = areal_amd.ppo_actor_loss_fn(t, t - 0.1, t, torch.ones(3, device=device), 0.2,
                                             torch.ones(3, dtype=torch.bool, device=device),
                                             importance_sampling_level="sequence", cu_seqlens=cu)
    assert torch.allclose(stat["importance_weight"], torch.full((3,), math.exp(0.1), device=device), atol=1e-5)


def test_masked_positions_and_denominator_keep_reference_semantics(device):
    """stat['loss'] keeps its pre-mask value, the ratio is zero where masked, and the denominator is the
    ORIGINAL mask count even when rejection sampling drops tokens (functional.py:479-483)."""
    _, cu, lp, prox, old, adv, mask = _random_packed(seed=31)
    cfg = RejectionSamplingConfig(level="token", metric="ratio", upper=1.3)
    loss, stat = areal_amd.ppo_actor_loss_fn(*_to(device, lp, prox, old, adv), 0.2, mask.to(device), rejection_sampling=cfg)
    kept = stat["behave_mask"].cpu()
    assert kept.sum() < mask.sum()
    manual = float(stat["loss"].cpu()[kept].double().sum()) / int(mask.sum())
    assert float(loss) == pytest.approx(manual, rel=1e-5)
    assert float(stat["importance_weight"].cpu()[~kept].abs().sum()) == 0.0


def test_empty_batches_do_not_raise(device):
    """Zero tokens (a data-parallel rank without work): empty results, zero counts, no launch over null pointers."""
    from areal_amd import RejectionSamplingConfig

    e = torch.zeros(0, device=device)
    eb = torch.zeros(0, dtype=torch.bool, device=device)
    cu0 = torch.zeros(1, dtype=torch.int32, device=device)
    for level in ("token", "sequence"):
        res = areal_amd.apply_rejection_sampling(e, e, eb, cu0, RejectionSamplingConfig(level=level, metric="ratio",
                                                                                         upper=2.0))
        assert res.loss_mask.numel() == 0 and res.filtered_fraction == 0.0
    loss, stat = areal_amd.ppo_actor_loss_fn(e.clone().requires_grad_(True), e, e, e, 0.2, eb)
    assert float(loss.detach()) == 0.0 and stat["importance_weight"].numel() == 0
    adv, ret = areal_amd.gae_advantages(torch.zeros(0, 8, device=device), torch.zeros(0, 8, device=device),
                                        torch.zeros(0, 8, device=device), eb, 1.0, 0.95)
    assert adv.shape == (0, 8) and ret.shape == (0, 8)


@pytest.mark.parametrize("n", [1, 255, 1025, 4096, 4097, 8200, 262144, 1048577])
@pytest.mark.parametrize("rs", [None, dict(level="token", upper=1.3), dict(level="sequence", upper=1.02)])
def test_step_launches_at_the_edges_of_their_slices(device, n, rs):
    """One workgroup, whole and ragged slices of 4096 tokens, and more tokens than the largest grid takes one slice of:
    counts, per-token outputs and loss of the launches around the loss, twice on one work buffer (it comes back zero).
    Whole numbers exactly; the loss is an fp64 sum of fp32 terms rounded once (and the terms differ by a few ulps of
    expf): 1e-5 relative to the mean absolute term."""
    g = torch.Generator().manual_seed(n)
    prox = -2 + 0.5 * torch.randn(n, generator=g)
    old, lp = prox + 0.3 * torch.randn(n, generator=g), prox + 0.3 * torch.randn(n, generator=g)
    adv, mask = torch.randn(n, generator=g), torch.rand(n, generator=g) < 0.7
    cu = torch.tensor([0] + sorted({n // 3, n // 2, n}), dtype=torch.int32)
    cfg = None if rs is None else RejectionSamplingConfig(action="mask", metric="ratio", **rs)
    want_loss, want = oracle.ppo_actor_loss(lp, prox, old, adv, 0.2, mask, rejection_sampling_cfg=cfg, cu_seqlens=cu, c_clip=3.0)
    d = _to(device, lp, prox, old, adv, mask, cu)
    for _ in range(2):
        x = d[0].clone().requires_grad_(True)
        loss, stat = areal_amd.ppo_actor_loss_fn(x, d[1], d[2], d[3], 0.2, d[4], c_clip=3.0, rejection_sampling=cfg, cu_seqlens=d[5])
        loss.backward()
        scale = float(want["loss"].abs().mean()) + 1e-6
        assert abs(float(loss.detach()) - float(want_loss)) <= 1e-5 * scale
        for k in ("clip_mask", "dual_clip_mask") + (("behave_mask",) if rs else ()):
            assert torch.equal(stat[k].cpu(), want[k]), k
        for k in ("loss", "importance_weight", "approx_kl"):
            assert torch.allclose(stat[k].cpu(), want[k], rtol=1e-5, atol=1e-5), k
        if rs:
            assert stat["filtered_fraction"] == want["filtered_fraction"]
        kept = mask if not rs else want["behave_mask"]
        assert float(x.grad[~kept.to(device)].abs().sum()) == 0.0


@pytest.mark.parametrize("n,covered", [(1, 1), (300, 300), (5000, 4321)])
@pytest.mark.parametrize("rs", [None, dict(level="token", upper=1.3), dict(level="sequence", upper=1.02)])
@pytest.mark.parametrize("level", ["token", "sequence"])
def test_separate_entry_points_of_the_c_abi_agree_with_the_step(device, n, covered, rs, level):
    """aa_rejection_sampling / aa_count_nonzero_u8, aa_ppo_loss, aa_ppo_stat_outputs and aa_masked_sum against the one call
    that does the same, and its first launch alone (counts_only).  The same expressions: whole numbers and masks exactly,
    floats to 4 ulps (a product or quotient taken in another order); the loss is one fp64 sum in two orders."""
    import ctypes

    from areal_amd import _native as N
    from areal_amd import functional as F

    lib = N.load()
    g = torch.Generator().manual_seed(n)
    prox = -2 + 0.5 * torch.randn(n, generator=g)
    old, lp, adv = prox + 0.3 * torch.randn(n, generator=g), prox + 0.3 * torch.randn(n, generator=g), torch.randn(n, generator=g)
    mask = torch.rand(n, generator=g) < 0.7
    mask[-1] = True
    cu = torch.tensor([0] + sorted({covered // 3, covered // 2, covered} - {0}), dtype=torch.int32)
    lp, prox, old, adv, mask, cu = _to(device, lp, prox, old, adv, mask, cu)
    B, seq = cu.numel() - 1, level == "sequence"
    cfg = None if rs is None else RejectionSamplingConfig(action="mask", metric="ratio", **rs)
    params = F._ppo_params(0.2, 0.28, 3.0, cfg is not None)
    P, st = (lambda t: None if t is None else t.data_ptr()), torch.cuda.current_stream().cuda_stream

    def new_step():
        return F._Step(device, n, n, mask, prox, old, adv, params, cfg, cu, B)

    step, g_step = new_step(), torch.empty_like(lp)
    N.check(lib.aa_ppo_loss_step(step.struct, P(lp), int(seq), 0, P(g_step), st), "aa_ppo_loss_step")
    counted = new_step()
    N.check(lib.aa_ppo_loss_step(counted.struct, None, 0, 1, None, st), "aa_ppo_loss_step")
    three = lambda s: s.floats.view(torch.int32)[9, :3].tolist()

    floats = lambda k: [torch.empty(n, device=device) for _ in range(k)]
    m8, w, mask_eff, counts = mask.view(torch.uint8), None, mask.view(torch.uint8), torch.empty(3, dtype=torch.int32, device=device)
    if cfg is None:
        N.check(lib.aa_count_nonzero_u8(P(m8), n, P(counts), st), "aa_count_nonzero_u8")
        assert three(step)[0] == three(counted)[0] == int(counts[0])
    else:
        mask_eff, w = torch.empty_like(m8), torch.empty(n, device=device)
        N.check(lib.aa_rejection_sampling(P(prox), P(old), P(m8), n, P(cu), B, N.RS_LEVEL[cfg.level], N.RS_ACTION[cfg.action],
                                          N.RS_METRIC[cfg.metric], N.RS_AGG[cfg.agg], float(cfg.upper), 0.0, 0, P(mask_eff),
                                          P(w), P(counts), st), "aa_rejection_sampling")
        assert three(step) == three(counted) == counts.tolist()
        outside = int(mask[covered:].sum()) if cfg.level == "sequence" else 0
        assert counts.tolist()[0] + outside == int(mask.sum()) and counts.tolist()[2] == outside
        for s in (step, counted):
            assert torch.equal(s.bools[1, :n], mask_eff.bool()) and torch.equal(s.floats[8, :n], w)
    stat_loss, ratio, g_logp, approx_kl, behave_kl = floats(5)
    flags, clip, dual, behave = (torch.empty(n, dtype=torch.uint8, device=device) for _ in range(4))
    N.check(lib.aa_ppo_loss(P(lp), P(prox), P(adv), P(mask_eff), P(w), n, P(cu), B, int(seq), ctypes.byref(params), P(counts),
                            P(stat_loss), P(ratio), P(flags), P(g_logp), st), "aa_ppo_loss")
    N.check(lib.aa_ppo_stat_outputs(P(lp), P(prox), P(old), P(flags), P(w), P(mask_eff), n, P(approx_kl), P(clip), P(dual),
                                    P(behave) if cfg else None, P(behave_kl) if cfg else None, st), "aa_ppo_stat_outputs")
    loss = torch.empty((), device=device)
    N.check(lib.aa_masked_sum(P(stat_loss), P(mask_eff), n, P(counts), None, P(loss), st), "aa_masked_sum")
    stat = step.stats(rows=False)
    for got, want in ((clip, stat["clip_mask"]), (dual, stat["dual_clip_mask"])) + (((behave, stat["behave_mask"]),) if cfg else ()):
        assert torch.equal(got.bool(), want)
    ulps = 4 * 2.0 ** -23
    for got, want in ((stat_loss, stat["loss"]), (ratio, stat["importance_weight"]), (g_logp, g_step), (approx_kl, stat["approx_kl"]),
                      *(((behave_kl, stat["behave_approx_kl"]),) if cfg else ())):
        assert torch.allclose(got, want, rtol=ulps, atol=0.0)
    assert abs(float(loss) - float(step.loss)) <= ulps * float((stat_loss.abs() * mask_eff).sum()) / max(int(counts[0]), 1) + 1e-30


@pytest.mark.parametrize("n", [1, 512, 513, 140001])
@pytest.mark.parametrize("methods,with_errors", [(0, 0), (1, 0), (7, 1)])
def test_logging_stats_with_and_without_the_mean(device, n, methods, with_errors):
    """aa_logging_stats (a launch to fold the slices) against aa_logging_stats_table (the last workgroup folds them): the
    same slices in the same order, so the same bits; the mean is the quotient."""
    from areal_amd import _native as N
    from areal_amd import functional as F

    lib = N.load()
    g = torch.Generator().manual_seed(n)
    old, lp, gt = (-torch.rand(n, generator=g) for _ in range(3))
    versions, mask = torch.randint(-1, 6, (n,), generator=g, dtype=torch.int32), torch.rand(n, generator=g) < 0.7
    old, lp, gt, versions, mask = _to(device, old, lp, gt, versions, mask)
    args = [t.data_ptr() for t in (old, lp, gt, versions, mask)] + [n, 6, methods, with_errors]
    scratch, st = torch.empty(lib.aa_logging_stats_scratch_bytes(n), dtype=torch.uint8, device=device), torch.cuda.current_stream().cuda_stream
    four, five = torch.empty(36, 4, device=device), torch.empty(36, 5, device=device)
    N.check(lib.aa_logging_stats(*args, four.data_ptr(), scratch.data_ptr(), scratch.numel(), st), "aa_logging_stats")
    N.check(lib.aa_logging_stats_table(*args, five.data_ptr(), scratch.data_ptr(), scratch.numel(), F._work_words(device).data_ptr(), st),
            "aa_logging_stats_table")
    assert torch.equal(four, five[:, :4])
    assert torch.allclose(five[:, 4], four[:, 0] / four[:, 3], rtol=2.0 ** -23, atol=0.0, equal_nan=True)
    assert int(four[0, 3]) == int(mask.sum())
