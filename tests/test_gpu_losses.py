"""GPU parity: GRPO / DPO loss kernels and masked reductions against the CPU oracle and the
reference's known-answer vectors (tests/golden/reference_known_answers.json)."""

import numpy as np
import pytest
import torch

from conftest import make_grpo_config
from open_instruct_amd import _lib, dpo_utils, grpo_utils, model_utils, padding_free_collator, rl_utils
from oracle import dpo as o_dpo
from oracle import grpo as o_grpo
from oracle import logprob as o_logprob
from oracle import reductions as o_red

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOL = 1e-5


def _close(a, b, tol=TOL):
    a, b = a.detach().float().cpu(), b.detach().float().cpu()
    assert a.shape == b.shape, (a.shape, b.shape)
    scale = max(1.0, b.abs().max().item()) if b.numel() else 1.0
    err = (a - b).abs().max().item() if b.numel() else 0.0
    assert err <= tol * scale, err


# ------------------------------------------------------------------ masked_mean
def test_masked_mean_reference_known_answers(golden):
    for case in golden["masked_mean"]:
        out = rl_utils.masked_mean(torch.tensor(case["values"], device=DEV), torch.tensor(case["mask"], device=DEV), axis=case["axis"])
        exp = torch.tensor(case["expected"])
        assert out.shape == exp.shape, case["source"]
        assert torch.allclose(out.cpu(), exp, rtol=1e-6, atol=0), case["source"]


@pytest.mark.parametrize("axis", [None, 1, 0, -1])
@pytest.mark.parametrize("denominator", [None, 37.5])
@pytest.mark.parametrize("bool_mask", [True, False])
def test_masked_mean_random_and_gradient(axis, denominator, bool_mask):
    g = torch.Generator().manual_seed(0)
    values = torch.randn(4, 6, 2500, generator=g)
    mask = torch.rand(6, 2500, generator=g) > 0.4
    mask[2] = False  # an empty row
    m = mask if bool_mask else mask.float()
    ref_v = values.clone().requires_grad_(True)
    ref = o_red.masked_mean(ref_v, m, axis, denominator)
    upstream = torch.randn(4, generator=g)
    ref.backward(upstream)
    dv = values.clone().to(DEV).requires_grad_(True)
    out = rl_utils.masked_mean(dv, m.to(DEV), axis, denominator)
    out.backward(upstream.to(DEV))
    _close(out, ref)
    # Slices whose mask is empty: the reference's torch.where(denom > 0, num / denom, 0) has a
    # 0 * (1/0) = NaN gradient there; the kernel defines that gradient as 0.
    exp_grad = ref_v.grad
    undefined = torch.isnan(exp_grad)
    assert (dv.grad.cpu()[undefined] == 0).all()
    exp_grad = torch.where(undefined, torch.zeros_like(exp_grad), exp_grad)
    assert (dv.grad.cpu() - exp_grad).abs().max().item() <= 1e-7 + 1e-5 * exp_grad.abs().max().item()


# both sides of the sizes that go in one launch: elements, rows and columns of a mean per row
@pytest.mark.parametrize("rows,cols,axis", [(1, 1, None), (1, 16384, None), (1, 16385, None), (3, 5461, None), (1, 2048, 1),
                                            (1, 2049, 1), (16, 1024, 1), (16, 1025, 1), (17, 900, 1), (15, 63, 1)])  # fmt: skip
def test_masked_mean_sizes_of_one_launch(rows, cols, axis):
    g = torch.Generator().manual_seed(rows * cols)
    values = torch.randn(3, rows, cols, generator=g)
    mask = torch.rand(rows, cols, generator=g) > 0.3
    mask[rows // 2] = rows == 1  # an empty row where there is another
    ref_v = values.double().requires_grad_(True)
    if axis is None:
        ref = (ref_v * mask).sum((1, 2)) / mask.sum()
    else:
        ref = ((ref_v * mask).sum(2) / mask.sum(1).clamp(min=1)).mean(1)
    ref.sum().backward()
    dv = values.to(DEV).requires_grad_(True)
    out = rl_utils.masked_mean(dv, mask.to(DEV), axis)
    out.sum().backward()
    # chunks of 1024 in fp32 at most: 10 roundings of partial sums no larger than the sum of magnitudes
    bound = 10 * 2.0**-24 * values.abs().amax().item()
    assert (out.detach().cpu().double() - ref.detach()).abs().max().item() <= bound
    assert (dv.grad.cpu().double() - ref_v.grad).abs().max().item() <= 2.0**-22 * ref_v.grad.abs().max().item()


# both sides of the leading entries that go in one launch
@pytest.mark.parametrize("extra,axis", [(512, None), (513, None), (256, 1), (257, 1), (65535, 1)])
def test_masked_mean_of_many_leading_entries(extra, axis):
    g = torch.Generator().manual_seed(extra)
    values = torch.randn(extra, 2, 33, generator=g)
    mask = torch.rand(2, 33, generator=g) > 0.3
    kept = values.double() * mask
    ref = kept.sum((1, 2)) / mask.sum() if axis is None else (kept.sum(2) / mask.sum(1)).mean(1)
    out = rl_utils.masked_mean(values.to(DEV), mask.to(DEV), axis)
    # fp32 at most: 6 roundings of a wave's sum, 3 of the four waves', and that of the result, none of more than the largest
    assert (out.cpu().double() - ref).abs().max().item() <= 10 * 2.0**-24 * values.abs().amax().item()


def test_masked_mean_scalar_cases():
    v = torch.tensor([[1.0, 2.0, 3.0], [4.0, 5.0, 6.0]], device=DEV)
    m = torch.tensor([[True, True, False], [True, False, False]], device=DEV)
    assert rl_utils.masked_mean(v, m, None, 10.0).item() == pytest.approx(0.7)
    assert rl_utils.masked_mean(v, m, None, 0.0).item() == 0.0
    assert rl_utils.masked_mean(v, torch.zeros_like(m)).item() == 0.0


# ------------------------------------------------------------------ compute_grpo_loss
def test_grpo_known_answers_on_device(golden):
    case = golden["dapo_clipping"]
    cfg = make_grpo_config(clip_lower=case["clip_lower"], clip_higher=case["clip_higher"])
    ratio = torch.tensor(case["ratio"], device=DEV)
    pg, clipfrac, kl = grpo_utils.compute_grpo_loss(
        torch.randn(1, 3, device=DEV), ratio, torch.tensor(case["advantages"], device=DEV), None, cfg, torch.ones_like(ratio)
    )
    assert torch.allclose(pg.cpu(), torch.tensor(case["expected_pg_loss"]))
    assert torch.equal(clipfrac.cpu(), torch.tensor(case["expected_clipfrac"]))
    assert torch.equal(kl.cpu(), torch.zeros(1, 3))
    case = golden["dapo_negative_advantages"]
    cfg = make_grpo_config(clip_lower=case["clip_lower"], clip_higher=case["clip_higher"])
    ratio = torch.tensor(case["ratio"], device=DEV)
    pg, _, _ = grpo_utils.compute_grpo_loss(
        torch.zeros_like(ratio), ratio, torch.full_like(ratio, case["advantage"]), None, cfg, torch.ones_like(ratio)
    )
    assert torch.allclose(pg.cpu(), torch.tensor(case["expected_pg_loss"]))
    case = golden["cispo"]
    cfg = make_grpo_config(loss_fn="cispo", clip_higher=case["clip_higher"])
    ratio = torch.tensor(case["ratio"], device=DEV, requires_grad=True)
    new = torch.randn(1, 3, device=DEV, requires_grad=True)
    pg, clipfrac, _ = grpo_utils.compute_grpo_loss(new, ratio, torch.tensor(case["advantages"], device=DEV), None, cfg, torch.ones(1, 3, device=DEV))
    pg.sum().backward()
    assert new.grad is not None and (ratio.grad is None or (ratio.grad == 0).all())
    assert torch.equal(clipfrac.cpu(), torch.tensor(case["expected_clipfrac"]))


def _grpo_inputs(seed, shape=(5, 300), edge=False):
    g = torch.Generator().manual_seed(seed)
    new = -torch.rand(shape, generator=g) * 5
    old = new + 0.3 * torch.randn(shape, generator=g)
    ref = new + 0.5 * torch.randn(shape, generator=g)
    adv = torch.randn(shape, generator=g)
    adv[0, :10] = 0.0
    mask = torch.rand(shape, generator=g) > 0.3
    rho = torch.rand(shape, generator=g) * 2
    rho[1, :20] = 0.0
    if edge:
        ref[2, :5] = new[2, :5] - 100.0  # outside the +-40 clamp
        old[3, :5] = new[3, :5]  # ratio exactly 1
    return new, old, ref, adv, mask, rho


@pytest.mark.parametrize("loss_fn", ["dapo", "cispo"])
@pytest.mark.parametrize("kl_estimator", [0, 1, 2, 3])
@pytest.mark.parametrize("with_ref", [True, False])
def test_compute_grpo_loss_parity_and_gradients(loss_fn, kl_estimator, with_ref):
    new, old, ref, adv, _, rho = _grpo_inputs(1, edge=True)
    cfg = make_grpo_config(loss_fn=loss_fn, clip_higher=0.28, kl_estimator=kl_estimator)
    g = torch.Generator().manual_seed(2)
    up_pg, up_kl = torch.randn(new.shape, generator=g), torch.randn(new.shape, generator=g)

    def run(mod, dev):
        n = new.clone().to(dev).requires_grad_(True)
        ratio = torch.exp(n - old.to(dev))
        pg, cf, kl = mod.compute_grpo_loss(n, ratio, adv.to(dev), ref.to(dev) if with_ref else None, cfg, rho.to(dev))
        (pg * up_pg.to(dev) + kl * up_kl.to(dev)).sum().backward()
        return pg, cf, kl, n.grad

    e_pg, e_cf, e_kl, e_grad = run(o_grpo, "cpu")
    pg, cf, kl, grad = run(grpo_utils, DEV)
    _close(pg, e_pg)
    assert torch.equal(cf.cpu(), e_cf)
    _close(kl, e_kl, 2e-5)
    _close(grad, e_grad, 2e-5)
    assert pg.requires_grad and not cf.requires_grad


def test_rho_correction_known_answers_on_device(golden):
    case = golden["rho_mask"]
    cfg = make_grpo_config(use_rho_correction=True, rho_mask_lower_bound=case["mask_lower"], rho_mask_upper_bound=case["mask_upper"])
    old = torch.log(torch.tensor(case["rho"])).to(DEV)
    zeros, ones = torch.zeros_like(old), torch.ones_like(old)
    c = grpo_utils.compute_rho_correction(old, zeros, torch.tensor(case["response_mask"], device=DEV), ones, cfg)
    assert torch.allclose(c.weights.cpu(), torch.tensor(case["expected_weights"]))
    assert torch.equal(c.metrics["val/rho_drop_low_frac"].cpu(), torch.tensor(case["expected_drop_low"]))
    assert torch.equal(c.metrics["val/rho_drop_high_frac"].cpu(), torch.tensor(case["expected_drop_high"]))
    c = grpo_utils.compute_rho_correction(old, zeros, torch.tensor(case["response_mask_with_pad"], device=DEV), ones, cfg)
    assert torch.allclose(c.weights.cpu(), torch.tensor(case["expected_weights_with_pad"]))
    assert torch.equal(c.metrics["val/rho_drop_low_frac"].cpu(), torch.tensor(case["expected_drop_low_with_pad"]))
    for key, extra in (("rho_mask_sequence_level", {"rho_mask_sequence_level": True}), ("rho_mask_tv_divergence", {"rho_mask_tv_divergence": True})):
        case = golden[key]
        cfg = make_grpo_config(use_rho_correction=True, rho_mask_lower_bound=case["mask_lower"], rho_mask_upper_bound=case["mask_upper"], **extra)
        old = torch.log(torch.tensor(case["rho"])).to(DEV)
        c = grpo_utils.compute_rho_correction(old, torch.zeros_like(old), torch.ones_like(old, dtype=torch.bool), torch.ones_like(old), cfg)
        assert torch.allclose(c.weights.cpu(), torch.tensor(case["expected_weights"])), key
        assert torch.equal(c.metrics["val/rho_drop_high_frac"].cpu(), torch.tensor(case["expected_drop_high"])), key


@pytest.mark.parametrize("seq_level,tv", [(False, False), (True, False), (False, True)])
def test_rho_correction_random_parity(seq_level, tv):
    new, old, _, adv, mask, _ = _grpo_inputs(3, shape=(7, 700))
    vl = old + 0.4 * torch.randn(old.shape, generator=torch.Generator().manual_seed(4))
    vl[~mask] = float("nan")  # vLLM logprobs are NaN on query tokens
    cfg = make_grpo_config(
        use_rho_correction=True, rho_mask_sequence_level=seq_level, rho_mask_tv_divergence=tv, rho_mask_lower_bound=0.6,
        rho_mask_upper_bound=1.6 if not tv else 0.3, rho_clamp_lower_bound=0.7, rho_clamp_upper_bound=1.4,
    )  # fmt: skip
    exp = o_grpo.compute_rho_correction(old, vl, mask, adv, cfg)
    got = grpo_utils.compute_rho_correction(old.to(DEV), vl.to(DEV), mask.to(DEV), adv.to(DEV), cfg)
    _close(got.weights, exp.weights)
    for k in exp.metrics:
        _close(got.metrics[k], exp.metrics[k])
    _close(got.histogram_metrics["val/rho_hist"], exp.histogram_metrics["val/rho_hist"])
    off = grpo_utils.compute_rho_correction(old.to(DEV), vl.to(DEV), mask.to(DEV), adv.to(DEV), make_grpo_config())
    assert (off.weights == 1).all() and off.metrics == {}


def test_mask_logprobs_and_estimate_kl():
    lp = torch.tensor([[0.5, float("nan"), -3.0, -1.0]], device=DEV, requires_grad=True)
    mask = torch.tensor([[True, True, False, True]], device=DEV)
    out = grpo_utils.mask_logprobs(lp, mask)
    assert out.tolist() == [[0.5, 1.0, 1.0, -1.0]]
    out.sum().backward()
    assert lp.grad.tolist() == [[1.0, 0.0, 0.0, 1.0]]
    assert (grpo_utils.mask_logprobs(lp.detach(), torch.zeros_like(mask)) == grpo_utils.INVALID_LOGPROB).all()
    g = torch.Generator().manual_seed(5)
    d = (torch.randn(3, 50, generator=g) * 3).clamp(-40, 40)
    ratio = torch.randn(3, 50, generator=g).exp()
    up = torch.randn(4, 3, 50, generator=g)
    rd, rr = d.clone().requires_grad_(True), ratio.clone().requires_grad_(True)
    exp = o_logprob.estimate_kl(rd, rr)
    exp.backward(up)
    gd, gr = d.to(DEV).requires_grad_(True), ratio.to(DEV).requires_grad_(True)
    got = model_utils.estimate_kl(gd, gr)
    got.backward(up.to(DEV))
    assert got.shape == (4, 3, 50)
    _close(got, exp)
    _close(gd.grad, rd.grad)
    _close(gr.grad, rr.grad)


# ------------------------------------------------------------------ fused scalar loss
@pytest.mark.parametrize("loss_fn", ["dapo", "cispo"])
@pytest.mark.parametrize("axis,denominator", [(None, None), (None, 1234.0), (1, None)])
@pytest.mark.parametrize("with_old", [True, False])
def test_grpo_loss_fused_parity(loss_fn, axis, denominator, with_old):
    new, old, ref, adv, mask, rho = _grpo_inputs(6, shape=(9, 2100), edge=True)
    mask[4] = False  # a row without response tokens
    ent = torch.rand(new.shape, generator=torch.Generator().manual_seed(7)) * 3
    cfg = make_grpo_config(loss_fn=loss_fn, clip_higher=0.28, beta=0.05)
    rn = new.clone().requires_grad_(True)
    o_old = old if with_old else rn.detach()
    e_loss, e_pg, e_cf, _, e_ratio = o_grpo.grpo_token_loss(rn, o_old, ref, adv, mask, cfg, rho, denominator, axis, dp_scale=2.0)
    e_loss.backward()
    dn = new.clone().to(DEV).requires_grad_(True)
    loss, stats = grpo_utils.grpo_loss_fused(
        dn, old.to(DEV) if with_old else None, ref.to(DEV), adv.to(DEV), mask.to(DEV), cfg, rho.to(DEV), ent.to(DEV),
        loss_denominator=denominator, axis=axis, dp_scale=2.0,
    )  # fmt: skip
    loss.backward()
    _close(loss, e_loss, 2e-5)
    # rows without response tokens under axis=1: NaN gradient in the reference (0 * 1/0), 0 here
    exp_grad = rn.grad
    undefined = torch.isnan(exp_grad)
    assert (dn.grad.cpu()[undefined] == 0).all() and (axis == 1 or not undefined.any())
    exp_grad = torch.where(undefined, torch.zeros_like(exp_grad), exp_grad)
    assert (dn.grad.cpu() - exp_grad).abs().max().item() <= 2e-5 * max(1e-6, exp_grad.abs().max().item()) + 1e-9
    # statistics recorded by populate_sample_loss_stats in the reference
    d = (rn.detach() - ref).clamp(-40, 40)
    kl4 = o_red.masked_mean(o_logprob.estimate_kl(d, e_ratio.detach()), mask)
    for j in range(4):
        _close(stats[f"objective/kl{j}_avg"], kl4[j], 2e-5)
    _close(stats["loss/policy_avg"], o_red.masked_mean(e_pg.detach(), mask), 2e-5)
    _close(stats["policy/clipfrac_avg"], o_red.masked_mean(e_cf, mask), 2e-5)
    _close(stats["val/ratio"], o_red.masked_mean(e_ratio.detach(), mask), 2e-5)
    _close(stats["policy/entropy_avg"], o_red.masked_mean(ent, mask), 2e-5)
    assert stats["num_response_tokens"].item() == float(mask.sum())
    assert stats["loss/total_avg"].item() == loss.item()


def test_grpo_loss_fused_empty_mask_is_zero():
    new, old, ref, adv, mask, _ = _grpo_inputs(8, shape=(2, 50))
    cfg = make_grpo_config()
    dn = new.to(DEV).requires_grad_(True)
    loss, stats = grpo_utils.grpo_loss_fused(dn, old.to(DEV), ref.to(DEV), adv.to(DEV), torch.zeros_like(mask).to(DEV), cfg)
    loss.backward()
    assert loss.item() == 0.0 and (dn.grad == 0).all() and stats["num_response_tokens"].item() == 0.0


@pytest.mark.parametrize("load_ref,with_rho,with_entropy", [(True, True, True), (False, True, False), (True, False, False)])
@pytest.mark.parametrize("route", ["tensors", "fused", "plain_dict"])
def test_populate_sample_loss_stats_parity(load_ref, with_rho, with_entropy, route):
    """open_instruct/grpo_utils.py:674-742 on the device against the oracle's restatement: from the
    per-token tensors (the reference's call; one pass, written into the table column), from the
    statistics of the fused loss kernels (nothing recomputed) and into a plain dict of tensors."""
    new, old, ref, adv, mask, _ = _grpo_inputs(16, shape=(5, 1300), edge=True)
    cfg = make_grpo_config(
        loss_fn="dapo", clip_higher=0.28, beta=0.05, kl_estimator=2, load_ref_policy=load_ref, use_rho_correction=True,
        rho_mask_lower_bound=0.7, rho_mask_upper_bound=1.4, rho_clamp_lower_bound=0.8, rho_clamp_upper_bound=1.2,
    )  # fmt: skip
    g = torch.Generator().manual_seed(17)
    vllm = old + 0.3 * torch.randn(old.shape, generator=g)
    ent = torch.rand(new.shape, generator=g) * 3 if with_entropy else None
    o_rho = o_grpo.compute_rho_correction(old, vllm, mask, adv, cfg)
    e_loss, e_pg, e_cf, _, e_ratio = o_grpo.grpo_token_loss(new, old, ref, adv, mask, cfg, o_rho.weights)
    exp = o_grpo.create_loss_stats(3, record_entropy=with_entropy)
    o_grpo.populate_sample_loss_stats(
        exp, 1, e_pg, e_cf, e_ratio, e_loss, mask, new, ref, ent, cfg, o_rho.metrics if with_rho else None
    )

    d = lambda t: None if t is None else t.to(DEV)  # noqa: E731
    rho = grpo_utils.compute_rho_correction(d(old), d(vllm), d(mask), d(adv), cfg)
    stats = grpo_utils.create_loss_stats(3, torch.device(DEV), record_entropy=with_entropy)
    assert set(stats) == set(exp) and all(v.shape == (3,) and v.is_cuda for v in stats.values())
    if route == "plain_dict":
        stats = {k: torch.zeros(3, device=DEV) for k in stats}
    rho_metrics = rho.metrics if with_rho else None
    if route == "fused":
        loss, fused = grpo_utils.grpo_loss_fused(
            d(new), d(old), d(ref), d(adv), d(mask), cfg, rho.weights, d(ent), rho_metrics=rho_metrics
        )
        grpo_utils.populate_sample_loss_stats(
            stats, 1, None, None, None, loss, d(mask), d(new), d(ref), d(ent), cfg, rho_metrics, fused_stats=fused
        )
    else:
        ratio = torch.exp(d(new) - d(old))
        pg, cf, _ = grpo_utils.compute_grpo_loss(d(new), ratio, d(adv), d(ref), cfg, rho.weights)
        loss = d(e_loss)
        grpo_utils.populate_sample_loss_stats(stats, 1, pg, cf, ratio, loss, d(mask), d(new), d(ref), d(ent), cfg, rho_metrics)
    for key, value in exp.items():
        got = stats[key].cpu()
        assert got[0].item() == 0.0 and got[2].item() == 0.0, key  # other samples untouched
        tol = 2e-5 * max(1.0, abs(value[1].item()))
        assert abs(got[1].item() - value[1].item()) <= tol, (key, got[1].item(), value[1].item())
    # the epoch summary: token-weighted means and the weighted variance of val/ratio
    counts = torch.tensor([3.0, 5.0, 0.0])
    for k in stats:
        stats[k][0] = 0.25
    exp_summary = o_grpo.compute_metrics_from_loss_stats({k: v.cpu() for k, v in stats.items()}, counts)
    summary = grpo_utils.compute_metrics_from_loss_stats(stats, counts.to(DEV))
    assert set(summary) == set(exp_summary)
    for k, v in exp_summary.items():
        assert summary[k] == pytest.approx(v, rel=1e-5, abs=1e-7), k
    zero = grpo_utils.compute_metrics_from_loss_stats(stats, torch.zeros(3, device=DEV))
    assert all(v == 0.0 for v in zero.values())


def test_group_advantages_on_device():
    rng = np.random.default_rng(0)
    scores = (rng.random(64) < 0.3).astype(np.float64)
    scores[8:16] = 1.0
    for mode in ("standard", "centered"):
        exp = o_grpo.group_advantages(scores, 8, mode).astype(np.float32)
        got = grpo_utils.group_advantages(torch.tensor(scores, device=DEV), 8, mode).cpu().numpy()
        assert np.array_equal(got, exp), mode  # Bernoulli rewards: sums are exact, so fp32 results are bit-equal
    assert (got[8:16] == 0).all()
    cont = rng.normal(size=48)
    got = grpo_utils.group_advantages(torch.tensor(cont, device=DEV), 16).cpu().numpy()
    assert np.abs(got - o_grpo.group_advantages(cont, 16)).max() <= 1e-6


# ------------------------------------------------------------------ per-sequence logps and DPO
def test_get_batch_logps_padded_known_answers(golden):
    for case in golden["get_batch_logps_padded_average"]:
        out = dpo_utils._get_batch_logps(
            torch.tensor(case["per_token_logps"], device=DEV), torch.tensor(case["labels"], device=DEV), average_log_prob=True
        )
        assert torch.equal(out.cpu(), torch.tensor(case["expected"])), case["source"]


@pytest.mark.parametrize("average", [False, True])
def test_seq_logps_packed_and_padded_parity(average):
    g = torch.Generator().manual_seed(9)
    lens = [700, 1, 1300, 64, 5, 2048]
    rows, labs = [], []
    for n in lens:
        rows.append(-torch.rand(n, generator=g) * 4)
        lab = torch.randint(0, 1000, (n,), generator=g)
        lab[: max(1, n // 3)] = -100
        labs.append(lab)
    labs[3][:] = -100  # a fully masked sequence
    per_token = torch.cat(rows).unsqueeze(0)
    labels = torch.cat(labs).unsqueeze(0)
    cu = torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32)
    up = torch.randn(len(lens), generator=g)
    rp = per_token.clone().requires_grad_(True)
    exp = o_red.get_batch_logps_packed(rp, labels, cu, average)
    exp.backward(up)
    dp = per_token.to(DEV).requires_grad_(True)
    got = padding_free_collator.get_batch_logps(dp, labels.to(DEV), cu.to(DEV), average)
    got.backward(up.to(DEV))
    _close(got, exp, 2e-6)
    assert not torch.isnan(got).any()
    assert torch.equal(dp.grad.cpu(), rp.grad)  # each position gets its sequence's upstream value (or 0): bit-exact
    # padded layout
    tmax = max(lens)
    pt = torch.zeros(len(lens), tmax)
    lb = torch.full((len(lens), tmax), -100)
    for i, n in enumerate(lens):
        pt[i, :n], lb[i, :n] = rows[i], labs[i]
    rp2 = pt.clone().requires_grad_(True)
    exp2 = o_red.get_batch_logps_padded(rp2, lb, average)
    exp2.backward(up)
    dp2 = pt.to(DEV).requires_grad_(True)
    got2 = dpo_utils._get_batch_logps(dp2, lb.to(DEV), average)
    got2.backward(up.to(DEV))
    _close(got2, exp2, 2e-6)
    assert torch.equal(dp2.grad.cpu(), rp2.grad)
    _close(got2, got, 2e-6)  # packed == padded


def test_packed_all_masked_segment(golden):
    case = golden["packed_cu_seq_lens"]
    g = torch.Generator().manual_seed(10)
    logits = torch.randn(1, case["seq_len"], 100, generator=g)
    labels = torch.ones(1, case["seq_len"], dtype=torch.long)
    lo, hi = case["masked_label_range"]
    labels[0, lo:hi] = -100
    cu = torch.tensor(case["cu_seq_lens"])
    per_token = padding_free_collator.calculate_per_token_logps(logits.to(DEV), labels.to(DEV))
    out = padding_free_collator.get_batch_logps(per_token, labels.to(DEV), cu.to(DEV), average_log_prob=True)
    exp = o_red.get_batch_logps_packed(o_logprob.calculate_per_token_logps(logits, labels), labels, cu, True)
    assert out.shape[0] == case["expected_num_outputs"] and not torch.isnan(out).any()
    _close(out, exp)


@pytest.mark.parametrize("label_smoothing", [0.0, 0.1])
@pytest.mark.parametrize("reference_free", [False, True])
def test_dpo_loss_parity_and_gradients(label_smoothing, reference_free, golden):
    g = torch.Generator().manual_seed(11)
    pc, pr = torch.randn(8, generator=g) * 30 - 400, torch.randn(8, generator=g) * 30 - 400
    rc, rr = torch.randn(8, generator=g) * 50 - 400, torch.randn(8, generator=g) * 50 - 400
    up = torch.randn(8, generator=g)

    def run(mod, dev):
        a, b = pc.clone().to(dev).requires_grad_(True), pr.clone().to(dev).requires_grad_(True)
        losses, cr, rj = mod.dpo_loss(a, b, rc.to(dev), rr.to(dev), 0.1, reference_free, label_smoothing)
        losses.backward(up.to(dev))
        return losses, cr, rj, a.grad, b.grad

    e = run(o_dpo, "cpu")
    o = run(dpo_utils, DEV)
    for got, exp in zip(o, e):
        _close(got, exp, 2e-6)
    assert not o[1].requires_grad and not o[2].requires_grad
    case = golden["dpo_loss_zero_margin"]
    losses, _, _ = dpo_utils.dpo_loss(*(torch.tensor(case[k], device=DEV) for k in ("policy_chosen", "policy_rejected", "ref_chosen", "ref_rejected")), beta=case["beta"])
    assert torch.allclose(losses.cpu(), torch.tensor(case["expected_losses"]), atol=1e-7)


def test_simpo_wpo_and_compute_loss_dispatch():
    g = torch.Generator().manual_seed(12)
    pc, pr = -torch.rand(1, generator=g) * 2, -torch.rand(1, generator=g) * 2
    rc, rr = -torch.rand(1, generator=g) * 2, -torch.rand(1, generator=g) * 2
    exp = o_dpo.simpo_loss(pc, pr, 2.0, 0.5, 0.1)
    got = dpo_utils.simpo_loss(pc.to(DEV), pr.to(DEV), 2.0, 0.5, 0.1)
    for a, b in zip(got, exp):
        _close(a, b, 2e-6)
    mask = torch.tensor([[True, False, True, True]])
    a = pc.clone().requires_grad_(True)
    exp = o_dpo.wpo_loss(a, pr, rc, rr, 0.3, mask, mask)
    exp[0].sum().backward()
    b = pc.to(DEV).requires_grad_(True)
    got = dpo_utils.wpo_loss(b, pr.to(DEV), rc.to(DEV), rr.to(DEV), 0.3, mask.to(DEV), mask.to(DEV))
    got[0].sum().backward()
    _close(got[0], exp[0], 2e-6)
    _close(b.grad, a.grad, 2e-6)

    class Args:
        loss_type, beta, label_smoothing, gamma_beta_ratio = "dpo_norm", 0.1, 0.0, 0.3

    class Cache:
        def __getitem__(self, index):
            return {"chosen_logps": rc.to(DEV)[index], "rejected_logps": rr.to(DEV)[index]}

    out = dpo_utils.compute_loss(Args, {"index": torch.tensor([0], device=DEV)}, pc.to(DEV), pr.to(DEV), Cache())
    _close(out[0], o_dpo.dpo_loss(pc, pr, rc, rr, 0.1)[0], 2e-6)
    Args.loss_type = "bogus"
    with pytest.raises(ValueError):
        dpo_utils.compute_loss(Args, {}, pc.to(DEV), pr.to(DEV), None)


def test_forward_for_logprobs_and_compute_logprobs_with_mock_model():
    """Mirrors open_instruct/test_olmo_core_train_modules.py:49-131 with a stub model returning fixed logits."""
    from open_instruct_amd.data_types import CollatedBatchData

    g = torch.Generator().manual_seed(13)
    b, t, v = 2, 5, 10
    logits = torch.randn(b, t, v, generator=g)

    class Model(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.z = torch.nn.Parameter(logits.to(DEV))

        def forward(self, input_ids, attention_mask=None, position_ids=None):
            return self.z[: input_ids.shape[0]]

    model = Model()
    qr = torch.randint(1, v, (b, t), generator=g)
    pos = torch.arange(t).unsqueeze(0).expand(b, -1)
    lp1, ent1 = grpo_utils.forward_for_logprobs(model, qr.to(DEV), None, pos.to(DEV), 0, 1.0, return_entropy=True)
    lp2, _ = grpo_utils.forward_for_logprobs(model, qr.to(DEV), None, pos.to(DEV), 0, 0.5)
    e_lp, e_ent = o_grpo.forward_for_logprobs(logits, qr, 0, 1.0, True)
    assert lp1.shape == (b, t - 1) and ent1.shape == (b, t - 1)
    assert (lp1 <= 0).all() and (ent1 >= 0).all() and lp1.requires_grad and not ent1.requires_grad
    assert not torch.allclose(lp1, lp2)
    _close(lp1, e_lp)
    _close(ent1, e_ent)
    mask = torch.ones(b, t, dtype=torch.bool)
    mask[:, :2] = False
    data = CollatedBatchData(
        query_responses=[qr.to(DEV), qr.to(DEV)], attention_masks=[torch.ones(b, t, dtype=torch.long, device=DEV)] * 2,
        position_ids=[pos.to(DEV)] * 2, advantages=[torch.randn(b, t, device=DEV)] * 2,
        response_masks=[mask.to(DEV), torch.zeros_like(mask).to(DEV)], vllm_logprobs=[torch.randn(b, t - 1, device=DEV)] * 2,
    )  # fmt: skip
    model1 = Model()
    out = grpo_utils.compute_logprobs(model1, data, pad_token_id=0, temperature=1.0, use_grad=True)
    assert len(out) == 2 and out[0].shape == (b, t - 1) and out[0].requires_grad
    assert (out[0] <= grpo_utils.INVALID_LOGPROB).all()
    assert (out[1] == grpo_utils.INVALID_LOGPROB).all()  # all-masked sample
    assert (out[0][:, 0] == grpo_utils.INVALID_LOGPROB).all()
    counts = grpo_utils.calculate_token_counts(1, data, torch.device(DEV))
    assert counts == {0: float(mask[:, 1:].sum()), 1: 0.0}

    # models with the olmo-core interface get doc_lens / max_doc_lens instead of the attention mask
    seen = {}

    class OlmoModel(Model):
        def forward(self, input_ids, attention_mask=None, position_ids=None, doc_lens=None, max_doc_lens=None):
            seen.update(attention_mask=attention_mask, doc_lens=doc_lens, max_doc_lens=max_doc_lens)
            return self.z[: input_ids.shape[0]]

    att = torch.tensor([[1, 1, 2, 2, 0], [1, 2, 2, 2, 2]], device=DEV)
    lp3, _ = grpo_utils.forward_for_logprobs(OlmoModel(), qr.to(DEV), att, pos.to(DEV), 0, 1.0, pass_olmo_core_doc_lens=True)
    assert seen["attention_mask"] is None and seen["doc_lens"].tolist() == [[2, 2, 1], [1, 4, 0]] and seen["max_doc_lens"] == [2, 4]
    assert torch.equal(lp3, lp1)
    data.attention_masks[:] = [att, att]
    out3 = grpo_utils.compute_logprobs(OlmoModel(), data, pad_token_id=0, temperature=1.0, pass_olmo_core_doc_lens=True)
    assert torch.equal(out3[0], out[0].detach()) and seen["doc_lens"].shape[0] == b


def test_separate_and_concatenated_forward_agree_and_pass_aux_loss():
    """open_instruct/dpo_utils.py:826-956: two forwards or one give the same per-sequence logps; with
    output_router_logits the model's aux_loss is handed on (concatenated: as is, separate: both sides
    concatenated)."""
    torch.manual_seed(5)
    vocab = 50
    table = torch.randn(vocab, vocab, device=DEV)

    class Out:
        def __init__(self, logits, aux):
            self.logits, self.aux_loss = logits, aux

    class Model(torch.nn.Module):
        def forward(self, input_ids, attention_mask=None, output_router_logits=False):
            return Out(table[input_ids], torch.tensor([0.25], device=DEV) if output_router_logits else None)

    batch = {
        "chosen_input_ids": torch.randint(1, vocab, (3, 9), device=DEV), "rejected_input_ids": torch.randint(1, vocab, (3, 6), device=DEV),
        "chosen_attention_mask": torch.ones(3, 9, dtype=torch.long, device=DEV),
        "rejected_attention_mask": torch.ones(3, 6, dtype=torch.long, device=DEV),
    }  # fmt: skip
    batch["chosen_labels"] = batch["chosen_input_ids"].clone()
    batch["rejected_labels"] = batch["rejected_input_ids"].clone()
    batch["chosen_labels"][:, :3] = -100
    batch["rejected_labels"][:, :2] = -100
    for average in (False, True):
        c1, r1, aux1 = dpo_utils.concatenated_forward(Model(), batch, average_log_prob=average)
        c2, r2, aux2 = dpo_utils.separate_forward(Model(), batch, average_log_prob=average)
        assert aux1 is None and aux2 is None
        _close(c1, c2)
        _close(r1, r2)
        for side, got in (("chosen", c1), ("rejected", r1)):
            per_token = o_logprob.calculate_per_token_logps(table[batch[f"{side}_input_ids"]].cpu(), batch[f"{side}_labels"].cpu())
            _close(got, o_red.get_batch_logps_padded(per_token, batch[f"{side}_labels"].cpu(), average), 1e-5)
    _, _, aux = dpo_utils.concatenated_forward(Model(), batch, output_router_logits=True)
    assert aux.tolist() == [0.25]
    _, _, aux = dpo_utils.separate_forward(Model(), batch, output_router_logits=True)
    assert aux.tolist() == [0.25, 0.25]


@pytest.mark.parametrize("shape", [(3, 9), (1, 1), (4, 5000)])
def test_vllm_local_debug_metrics_parity(shape):
    """open_instruct/grpo_utils.py:345-369 in one launch; fp64 accumulation on the device, so the
    comparison is against the oracle run in fp64 (1e-5) and in fp32 (loose: fp32 summation order)."""
    g = torch.Generator().manual_seed(23)
    local = -torch.rand(shape, generator=g) * 5
    vllm = local + 0.1 * torch.randn(shape, generator=g)
    mask = torch.rand(shape, generator=g) > 0.3
    if shape[1] > 4:
        vllm[0, 2] = float("nan")
        mask[0, 2] = True
    got = grpo_utils.compute_vllm_local_debug_metrics(local.to(DEV), vllm.to(DEV), mask.to(DEV))
    exp = o_grpo.compute_vllm_local_debug_metrics(local.double(), vllm.double(), mask)
    assert set(got) == set(exp)
    for k in exp:
        assert abs(got[k] - exp[k]) <= 1e-5 * max(1.0, abs(exp[k])), (k, got[k], exp[k])
    none = grpo_utils.compute_vllm_local_debug_metrics(local.to(DEV), vllm.to(DEV), torch.zeros_like(mask).to(DEV))
    assert all(x == 0.0 for x in none.values())
    vec = grpo_utils.vllm_local_debug_stats(local.to(DEV), vllm.to(DEV), mask.to(DEV))
    assert vec.shape == (4,) and vec.is_cuda
    with pytest.raises(ValueError):
        grpo_utils.vllm_local_debug_stats(local.to(DEV), vllm.to(DEV)[..., :-1], mask.to(DEV))


def test_reference_cache_build_through_concatenated_forward(tmp_path):
    """open_instruct/dpo_utils.py:405-520 over open_instruct/dpo_utils.py:826-878 with a stub model:
    the cache holds, per dataset index, what a direct oracle evaluation of that sample gives."""
    g = torch.Generator().manual_seed(24)
    v, t, n_samples = 50, 12, 4
    table = torch.randn(64, v, generator=g)  # logits depend on the token id only

    class Model(torch.nn.Module):
        def forward(self, input_ids, attention_mask=None, **kw):
            return table.to(input_ids.device)[input_ids]

    def sample(i):
        ids_c = torch.randint(0, 64, (1, t), generator=g)
        ids_r = torch.randint(0, 64, (1, t), generator=g)
        lab_c, lab_r = ids_c.clone() % v, ids_r.clone() % v
        lab_c[:, :3] = -100
        lab_r[:, :5] = -100
        return {
            "chosen_input_ids": ids_c, "chosen_labels": lab_c, "chosen_attention_mask": torch.ones_like(ids_c),
            "rejected_input_ids": ids_r, "rejected_labels": lab_r, "rejected_attention_mask": torch.ones_like(ids_r),
            "index": torch.tensor([i]),
        }  # fmt: skip

    samples = [sample(i) for i in (2, 0, 3, 1)]
    batches = [{k: val.to(DEV) for k, val in s.items()} for s in samples]
    cache = dpo_utils.build_reference_logprobs_cache(
        model=Model(), dataloader=batches, average_log_prob=False, forward_fn=dpo_utils.concatenated_forward,
        full_dataset_size=n_samples, device=torch.device(DEV), cache_path=tmp_path / "reference_logps.pt",
        is_main_process=True, model_dims=None,
    )  # fmt: skip
    assert (tmp_path / "reference_logps.pt").exists()
    for s in samples:
        i = int(s["index"])
        for side in ("chosen", "rejected"):
            per_token = o_logprob.calculate_per_token_logps(table[s[f"{side}_input_ids"]], s[f"{side}_labels"])
            exp = o_red.get_batch_logps_padded(per_token, s[f"{side}_labels"])
            got = cache.tensors[f"{side}_logps"][i].item()
            assert abs(got - exp.item()) <= 1e-4, (side, i, got, exp.item())
    picked = cache[torch.tensor([1, 3], device=DEV)]
    assert picked["chosen_logps"].shape == (2,)


@pytest.mark.parametrize("dtype,vocab", [
    (torch.float32, 64), (torch.bfloat16, 4096), (torch.bfloat16, 4099), (torch.float16, 1000),
    # rows longer than what a workgroup parks on its CU (16384 16-byte pieces): the rest is read twice
    (torch.bfloat16, 151936), (torch.float32, 70000),
])  # fmt: skip
@pytest.mark.parametrize("loss_fn,axis,denominator,with_old,with_ref,drop_last", [
    ("dapo", None, None, True, True, False),
    ("dapo", 1, None, True, True, True),
    ("cispo", None, 77.0, True, False, False),
    ("dapo", None, None, False, True, True),
])  # fmt: skip
def test_grpo_loss_on_logits_single_pass(dtype, vocab, loss_fn, axis, denominator, with_old, with_ref, drop_last):
    """One read + one write of the logits (open_instruct/grpo_utils.py:541-574 -> :504-538 ->
    open_instruct/grpo_fast.py:702-724 fused) against the CPU oracle chain and against the two-pass
    kernels.  vocab 4099 does not fit the single-pass kernel and must fall back with equal results."""
    g = torch.Generator().manual_seed(41)
    b, t = 3, 6
    rows_t = t + 1 if drop_last else t
    logits = (torch.randn(b, rows_t, vocab, generator=g) * 2.0).to(dtype)
    labels = torch.randint(0, vocab, (b, t), generator=g)
    adv = torch.randn(b, t, generator=g)
    mask = torch.rand(b, t, generator=g) > 0.3
    mask[1] = False  # a row without response tokens
    rho = torch.rand(b, t, generator=g) + 0.5
    cfg = make_grpo_config(loss_fn=loss_fn, beta=0.05, kl_estimator=2, clip_higher=0.28)
    temperature = 0.9
    # oracle chain in fp32 on the same (rounded) logits
    ref_in = logits.float().clone().requires_grad_(True)
    z = ref_in[:, :-1] if drop_last else ref_in
    lp_o = o_logprob.log_softmax_and_gather(z, labels, None, temperature)
    ent_o = o_logprob.entropy_from_logits(z.detach(), None, temperature)
    old = lp_o.detach() + 0.05 * torch.randn(b, t, generator=g) if with_old else None
    ref = lp_o.detach() + 0.1 * torch.randn(b, t, generator=g) if with_ref else None
    loss_o, *_ = o_grpo.grpo_token_loss(
        lp_o, old if with_old else lp_o.detach(), ref, adv, mask.float(), cfg, rho_weights=rho,
        loss_denominator=denominator, axis=axis, dp_scale=0.5,
    )  # fmt: skip
    # rows without tokens give NaN gradients in the reference formulation (0 * 1/0); the kernels define 0
    torch.nan_to_num(loss_o, nan=0.0).backward()
    exp_grad = torch.nan_to_num(ref_in.grad, nan=0.0)

    dev = lambda x: None if x is None else x.to(DEV)  # noqa: E731
    lg = logits.to(DEV).requires_grad_(True)
    loss, stats, lp, ent = grpo_utils.grpo_loss_on_logits(
        lg, dev(labels), dev(old), dev(ref), dev(adv), dev(mask), cfg, temperature=temperature, rho_weights=dev(rho),
        loss_denominator=denominator, axis=axis, dp_scale=0.5, drop_last=drop_last,
    )  # fmt: skip
    loss.backward()
    tol = 1e-5 if dtype == torch.float32 else 2e-3
    assert not lp.requires_grad and lp.shape == (b, t)
    assert (lp.cpu() - lp_o.detach()).abs().max().item() <= tol
    assert (ent.cpu() - ent_o).abs().max().item() <= tol
    if axis is None:  # with axis=1 the reference value itself is NaN-free only without empty rows
        assert abs(loss.item() - loss_o.item()) <= tol
    assert lg.grad.dtype == dtype and lg.grad.shape == logits.shape
    assert (lg.grad.float().cpu() - exp_grad).abs().max().item() <= tol
    if drop_last:
        assert (lg.grad[:, -1] == 0).all()
    # the two-pass kernels give the same numbers
    lg2 = logits.to(DEV).requires_grad_(True)
    lp2, ent2 = model_utils.logprob_and_entropy(lg2, dev(labels), temperature=temperature, drop_last=drop_last)
    loss2, stats2 = grpo_utils.grpo_loss_fused(
        lp2, dev(old), dev(ref), dev(adv), dev(mask), cfg, rho_weights=dev(rho), entropy=ent2,
        loss_denominator=denominator, axis=axis, dp_scale=0.5,
    )  # fmt: skip
    loss2.backward()
    # another workgroup size, another merge order of the per-lane statistics: last-bit differences
    assert (lp - lp2.detach()).abs().max().item() <= 4e-6 and (ent - ent2).abs().max().item() <= 4e-6
    assert abs(loss.item() - loss2.item()) <= 4e-6 * max(1.0, abs(loss2.item()))
    for k in stats2:
        assert abs(stats[k].item() - stats2[k].item()) <= 4e-6 * max(1.0, abs(stats2[k].item())), k
    step = 2.0**-7 if dtype != torch.float32 else 1e-5
    assert (lg.grad.float() - lg2.grad.float()).abs().max().item() <= step * max(1e-3, lg2.grad.float().abs().max().item())
    # an upstream gradient other than 1 scales the stored gradient
    lg3 = logits.to(DEV).requires_grad_(True)
    loss3, *_ = grpo_utils.grpo_loss_on_logits(
        lg3, dev(labels), dev(old), dev(ref), dev(adv), dev(mask), cfg, temperature=temperature, rho_weights=dev(rho),
        loss_denominator=denominator, axis=axis, dp_scale=0.5, drop_last=drop_last,
    )  # fmt: skip
    (loss3 * 2.0).backward()
    assert (lg3.grad.float() - 2.0 * lg.grad.float()).abs().max().item() <= 2.0 * step * max(1e-3, lg.grad.float().abs().max().item())


def test_grpo_on_logits_raw_c_abi_rows_with_scalar_tail():
    """oi_lsg_grpo_fwd_bwd through ctypes on rows whose length is not a multiple of the 16-byte piece
    (a [rows, 4099] view of a [rows, 4104] buffer, gradient into a buffer of the same pitch), more rows
    than workgroups' first round, labels in the last whole piece, in the scalar tail and at 0; against
    the oracle's autograd (open_instruct/grpo_utils.py:504-538 on open_instruct/model_utils.py:587-603)."""
    lib = _lib.load()
    g = torch.Generator().manual_seed(17)
    rows, vocab, pitch = 700, 4099, 4104
    buf = (torch.randn(rows, pitch, generator=g) * 2.0).bfloat16()
    labels = torch.randint(0, vocab, (rows,), generator=g)
    labels[:4] = torch.tensor([0, vocab - 1, vocab - 3, 4095])
    adv = torch.randn(rows, generator=g)
    mask = torch.rand(rows, generator=g) > 0.3
    cfg = make_grpo_config(loss_fn="dapo", beta=0.05, kl_estimator=2, clip_higher=0.28)
    ref_in = buf[:, :vocab].float().clone().requires_grad_(True)
    lp_o = o_logprob.log_softmax_and_gather(ref_in, labels, None, 1.0)
    ent_o = o_logprob.entropy_from_logits(ref_in.detach(), None, 1.0)
    old = lp_o.detach() + 0.05 * torch.randn(rows, generator=g)
    ref = lp_o.detach() + 0.1 * torch.randn(rows, generator=g)
    loss_o, *_ = o_grpo.grpo_token_loss(
        lp_o[None], old[None], ref[None], adv[None], mask.float()[None], cfg, rho_weights=torch.ones(1, rows),
        loss_denominator=None, axis=None, dp_scale=1.0,
    )  # fmt: skip
    loss_o.backward()
    d = lambda x: x.to(DEV).contiguous()  # noqa: E731
    lg, out = d(buf), torch.full((rows, pitch), 7.0, device=DEV).bfloat16()
    coef = d(mask.float() / mask.sum())
    lp, ent = torch.empty(rows, device=DEV), torch.empty(rows, device=DEV)
    lab, old_d, ref_d, adv_d = d(labels), d(old), d(ref), d(adv)
    rc = lib.oi_lsg_grpo_fwd_bwd(
        lg.data_ptr(), 1, rows, 1, pitch, pitch, vocab, lab.data_ptr(), 1.0, old_d.data_ptr(), ref_d.data_ptr(),
        adv_d.data_ptr(), None, coef.data_ptr(), 0, 1.0 - cfg.clip_lower, 1.0 + cfg.clip_higher, 2, cfg.beta,
        lp.data_ptr(), ent.data_ptr(), None, out.data_ptr(), pitch, pitch, torch.cuda.current_stream().cuda_stream,
    )  # fmt: skip
    assert rc == 0
    torch.cuda.synchronize()
    assert (lp.cpu() - lp_o.detach()).abs().max().item() <= 2e-3
    assert (ent.cpu() - ent_o).abs().max().item() <= 2e-3
    assert (out[:, :vocab].float().cpu() - ref_in.grad).abs().max().item() <= 2e-3
    assert (out[:, :vocab].float().cpu() - ref_in.grad).abs().max().item() <= 2.0**-7 * ref_in.grad.abs().max().item()
    assert (out[:, vocab:] == 7.0).all()  # the padding of the gradient buffer is not touched
    # rows shorter than one piece are refused, as are unaligned pitches
    args = lambda v, so: (lg.data_ptr(), 1, rows, 1, so, so, v, lab.data_ptr(), 1.0, None, None, adv_d.data_ptr(), None,  # noqa: E731
                          coef.data_ptr(), 0, 0.8, 1.28, 2, 0.0, lp.data_ptr(), ent.data_ptr(), None, out.data_ptr(), so, so,
                          torch.cuda.current_stream().cuda_stream)  # fmt: skip
    assert lib.oi_lsg_grpo_fwd_bwd(*args(5, pitch)) < 0
    assert lib.oi_lsg_grpo_fwd_bwd(*args(vocab, vocab)) < 0


def test_grpo_loss_on_logits_full_vocabulary_rows():
    """Llama-3 vocabulary (128256, bf16), 300 rows: the single-launch path against the two-pass
    kernels on the device (the CPU oracle covers small shapes above)."""
    torch.manual_seed(42)
    b, t, vocab = 3, 100, 128256
    logits = (torch.randn(b, t, vocab, device=DEV) * 3.0).bfloat16()
    labels = torch.randint(0, vocab, (b, t), device=DEV)
    adv = torch.randn(b, t, device=DEV)
    mask = torch.rand(b, t, device=DEV) > 0.2
    cfg = make_grpo_config(loss_fn="dapo", beta=0.05, kl_estimator=2, clip_higher=0.28)
    with torch.no_grad():
        lp0 = model_utils.log_softmax_and_gather(logits, labels)
    old, ref = lp0 + 0.05 * torch.randn_like(lp0), lp0 + 0.1 * torch.randn_like(lp0)
    a = logits.clone().requires_grad_(True)
    loss_a, stats_a, lp_a, ent_a = grpo_utils.grpo_loss_on_logits(a, labels, old, ref, adv, mask, cfg)
    loss_a.backward()
    c = logits.clone().requires_grad_(True)
    lp_c, ent_c = model_utils.logprob_and_entropy(c, labels)
    loss_c, stats_c = grpo_utils.grpo_loss_fused(lp_c, old, ref, adv, mask, cfg, entropy=ent_c)
    loss_c.backward()
    assert (lp_a - lp_c.detach()).abs().max().item() <= 1e-5 and (ent_a - ent_c).abs().max().item() <= 1e-5
    assert abs(loss_a.item() - loss_c.item()) <= 1e-6 + 1e-5 * abs(loss_c.item())
    ga, gc = a.grad.float(), c.grad.float()
    assert (ga - gc).abs().max().item() <= 2.0**-7 * gc.abs().max().item()
    assert (ga[~mask] == 0).all()
    # every gradient row sums to ~0 and the statistics agree
    assert ga.sum(-1).abs().max().item() <= 0.05 * ga.abs().max().item() * 8
    for k in stats_c:
        assert abs(stats_a[k].item() - stats_c[k].item()) <= 1e-5 * max(1.0, abs(stats_c[k].item())), k


def test_grpo_loss_on_logits_broadcast_side_tensors():
    """Side tensors that only broadcast to [B, T] ([B, 1] advantages, a 0-dim rho weight, [1, T] old
    logprobs) are accepted by the reference's elementwise code; the single-launch route must expand
    them like the two-pass route does and give the same loss and gradient."""
    g = torch.Generator().manual_seed(51)
    b, t, vocab = 4, 9, 4096
    logits = (torch.randn(b, t, vocab, generator=g) * 2.0).bfloat16()
    labels = torch.randint(0, vocab, (b, t), generator=g)
    mask = torch.rand(b, t, generator=g) > 0.2
    adv = torch.randn(b, 1, generator=g)
    rho = torch.tensor(0.75)
    ref = -10.3 + 0.5 * torch.randn(1, t, generator=g)  # near the logprobs of N(0, 2) logits at this vocabulary
    cfg = make_grpo_config(loss_fn="dapo", beta=0.05, kl_estimator=2, clip_higher=0.28)
    d = lambda x: x.to(DEV)  # noqa: E731
    one = d(logits).requires_grad_(True)
    loss1, _, lp1, _ = grpo_utils.grpo_loss_on_logits(one, d(labels), None, d(ref), d(adv), d(mask), cfg, rho_weights=d(rho))
    loss1.backward()
    two = d(logits).requires_grad_(True)
    lp2, ent2 = model_utils.logprob_and_entropy(two, d(labels))
    loss2, _ = grpo_utils.grpo_loss_fused(lp2, None, d(ref), d(adv), d(mask), cfg, rho_weights=d(rho), entropy=ent2)
    loss2.backward()
    rl = logits.float().requires_grad_(True)
    lp_o = o_logprob.log_softmax_and_gather(rl, labels, None)
    loss_o, *_ = o_grpo.grpo_token_loss(
        lp_o, lp_o.detach(), ref.expand(b, t), adv.expand(b, t), mask.float(), cfg, rho_weights=rho.expand(b, t)
    )
    loss_o.backward()
    assert abs(loss1.item() - loss2.item()) <= 1e-5 and abs(loss1.item() - loss_o.item()) <= 2e-3
    assert (one.grad.float() - two.grad.float()).abs().max().item() <= 2.0**-7 * two.grad.float().abs().max().item()
    assert (one.grad.float().cpu() - rl.grad).abs().max().item() <= 2e-3 + 2.0**-7 * rl.grad.abs().max().item()
    with pytest.raises(ValueError, match="does not broadcast"):
        grpo_utils.grpo_loss_on_logits(one, d(labels), None, None, d(adv.reshape(1, b)), d(mask), cfg)
    # an evaluation call builds no gradient tensor and still returns the loss
    with torch.no_grad():
        loss3, _, lp3, _ = grpo_utils.grpo_loss_on_logits(one, d(labels), None, d(ref), d(adv), d(mask), cfg, rho_weights=d(rho))
    assert not loss3.requires_grad and abs(loss3.item() - loss1.item()) <= 1e-5


def test_rho_correction_broadcast_advantages():
    new, old, _, _, mask, _ = _grpo_inputs(23, shape=(4, 60))
    adv = torch.randn(4, 1, generator=torch.Generator().manual_seed(3))
    cfg = make_grpo_config(use_rho_correction=True, rho_mask_tv_divergence=True, rho_mask_lower_bound=0.05, rho_mask_upper_bound=0.2)
    exp = o_grpo.compute_rho_correction(old, new, mask, adv.expand(4, 60), cfg)
    got = grpo_utils.compute_rho_correction(old.to(DEV), new.to(DEV), mask.to(DEV), adv.to(DEV), cfg)
    _close(got.weights, exp.weights)
    for k, v in exp.metrics.items():
        _close(got.metrics[k], v)


@pytest.mark.parametrize("shape", [(1, 1), (1, 255), (1, 257), (3, 1365), (1, 4096), (1, 4097), (2, 16384), (1, 32769)])
@pytest.mark.parametrize("kept", [0.0, 0.6, 1.0])
def test_rho_histogram_is_the_selection_in_order(shape, kept):
    g = torch.Generator().manual_seed(shape[1])
    old, vllm = torch.randn(shape, generator=g).to(DEV), torch.randn(shape, generator=g).to(DEV)
    mask = (torch.rand(shape, generator=g) < kept).to(DEV)
    cfg = make_grpo_config(use_rho_correction=True)
    hist = grpo_utils.compute_rho_correction(old, vllm, mask, torch.ones(shape, device=DEV), cfg).histogram_metrics["val/rho_hist"]
    expected = torch.exp((old - vllm).clamp(-10, 10))[mask]
    assert hist.shape == expected.shape and torch.allclose(hist, expected, rtol=1e-5, atol=0)


@pytest.mark.parametrize("sample_idx", [0, 6, -1])  # the last by the general way
def test_recorded_column_equals_the_general_way(sample_idx, monkeypatch):
    g = torch.Generator().manual_seed(5)
    t = lambda: torch.randn(2, 70, generator=g).to(DEV)  # noqa: E731
    mask = (torch.rand(2, 70, generator=g) < 0.7).to(DEV)
    cfg = make_grpo_config(load_ref_policy=True, beta=0.05)
    new, old, ref, adv, ent = t(), t(), t(), t(), t()
    loss, stats = grpo_utils.grpo_loss_fused(new, old, ref, adv, mask, cfg, entropy=ent)
    tables, calls, call = [], [], _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *args: (calls.append(name), call(name, *args))[1])
    for recorded in (stats, {k: v for k, v in stats.items()}):
        table = grpo_utils.create_loss_stats(7, DEV, record_entropy=True)
        table.table.fill_(7.0)
        total = loss if recorded is stats else loss.double()  # the general way
        grpo_utils.populate_sample_loss_stats(table, sample_idx, None, None, None, total, mask, new, ref, ent, cfg, fused_stats=recorded)
        tables.append(table.table)
    assert calls.count("oi_record_stats") == (1 if sample_idx >= 0 else 0)
    assert torch.equal(*tables)
