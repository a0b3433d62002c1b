"""The backward that reads the forward's logits against the one that computes them again: the same products in
the same order, so both gradients must agree to the bit, at the edges of the tiles (rows and columns that are
no multiple of anything, a single row, masks that leave few rows or none)."""

import pytest
import torch

from open_instruct_amd import _lib, lm_head, olmo_core_train_modules

DEV = "cuda:0"


def test_kept_bytes_limits():
    lib = _lib.load()
    assert lib.oi_lmhead_kept_bytes(1, 1) == 256 * 256 * 4
    assert lib.oi_lmhead_kept_bytes(8192, 131072) == 4 << 30
    assert lib.oi_lmhead_kept_bytes(8193, 131072) == 0
    assert lib.oi_lmhead_kept_bytes(8192, 131073) == 0
    assert lib.oi_lmhead_kept_bytes(0, 1000) == lib.oi_lmhead_kept_bytes(1 << 23, 1) == 0
    # refused before anything is launched: nothing to keep there, or less memory than that
    args = [1 << 4] * 3 + [None]
    assert lib.oi_lmhead_logp_fwd_kept(*args, 8193, 64, 131072, 1.0, 256, None, 256, 256, 1 << 40, 256, 1 << 40, None) == -5
    assert lib.oi_lmhead_logp_fwd_kept(*args, 10, 64, 300, 1.0, 256, None, 256, 256, 512 * 256 * 4 - 1, 256, 1 << 40, None) == -5


@pytest.mark.gpu
@pytest.mark.parametrize(
    "n,h,v,share",
    [(1, 64, 50, None), (256, 64, 256, None), (257, 192, 1001, None), (700, 256, 2047, 0.4), (513, 128, 300, 0.002),
     (90, 64, 777, 0.0)],
)  # fmt: skip
def test_kept_logits_match_recomputed_logits(n, h, v, share):
    print("case kept logits", n, h, v, share, flush=True)
    g = torch.Generator().manual_seed(n + v)
    hidden = torch.randn(n, h, generator=g).bfloat16().to(DEV)
    weight = (torch.randn(v, h, generator=g) * 0.2).bfloat16().to(DEV)
    labels = torch.randint(-3, v + 3, (n,), generator=g).to(DEV)
    up = (torch.rand(n, generator=g) + 0.5).to(DEV)  # never 0: both routes multiply the same rows
    mask = None if share is None else (torch.rand(n, generator=g) < share).to(DEV)
    results = []
    for compact in (False, True):  # leaving out rows without a gradient is the recomputing route
        dh, dw = hidden.clone().requires_grad_(True), weight.clone().requires_grad_(True)
        out, ent = lm_head.fused_lm_head_logprobs(dh, dw, labels, 0.8, mask=mask, return_entropy=True, compact_backward=compact)
        kept = [t for t in out.grad_fn.next_functions[0][0].saved_tensors if t is not None and t.numel() >= 256 * 256]
        assert any(t.dtype == torch.float32 for t in kept) != compact
        for _ in range(2):  # the kept logits survive a backward pass
            dh.grad = dw.grad = None
            out.backward(up, retain_graph=True)
        results.append((out.detach(), ent, dh.grad, dw.grad))
    for a, b in zip(*results):
        assert torch.equal(a, b)


# ---- where the logits are not kept --------------------------------------------------------------------------
def _ask(n=300, h=64, v=1000):
    return lm_head._kept_logits(n, h, v, torch.device("cpu"), False)


@pytest.fixture
def plenty(monkeypatch):
    """A device with all the memory in the world and no graph alive, seen from the CPU."""
    monkeypatch.setattr(lm_head, "_free_bytes", lambda dev: 1 << 50)
    monkeypatch.setattr(lm_head, "_kept_alive", [])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)


def test_live_graphs_share_one_budget(plenty, monkeypatch):
    first = _ask()
    monkeypatch.setattr(lm_head, "KEPT_BUDGET", first.numel() * 4 * 2 + 1)
    second = _ask()
    assert second is not None and _ask() is None
    del first  # its graph is through
    third = _ask()
    assert third is not None and _ask() is None and len(lm_head._kept_alive) == 2
    del second, third
    assert _ask(1, 64, 1) is not None


def test_kept_only_out_of_plenty(plenty, monkeypatch):
    lib = _lib.load()
    n, h, v = 300, 64, 1000
    monkeypatch.setattr(lm_head, "_free_bytes", lambda dev: 0)
    assert _ask(n, h, v) is not None  # a little is kept without asking
    monkeypatch.setattr(lm_head, "KEPT_UNASKED", 0)
    needs = 8 * lib.oi_lmhead_kept_bytes(n, v) + lib.oi_lmhead_bwd_workspace_bytes(n, h, v, 1, 0) + 2 * h * (n + v)
    monkeypatch.setattr(lm_head, "_free_bytes", lambda dev: needs - 1)
    assert _ask(n, h, v) is None
    monkeypatch.setattr(lm_head, "_free_bytes", lambda dev: needs)
    assert _ask(n, h, v) is not None


def test_not_kept_where_saved_tensors_are_packed_or_a_stream_captures(plenty, monkeypatch):
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, lambda t: t):
        assert _ask() is None
    assert _ask() is not None
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    assert _ask() is None


def test_an_allocation_that_fails_is_not_kept(plenty, monkeypatch):
    def refuse(*args, **kwargs):
        raise torch.cuda.OutOfMemoryError("no block of that size")

    monkeypatch.setattr(torch, "empty", refuse)
    assert _ask() is None


@pytest.mark.parametrize("n,h,v", [(300, 64, 1001)])
@pytest.mark.gpu
def test_calls_without_kept_logits_give_the_same_bits(n, h, v, monkeypatch):
    """Refused memory, a budget that another graph holds, checkpointing and the caller's own choice."""
    print("case not kept", n, h, v, flush=True)
    g = torch.Generator().manual_seed(n + v)
    hidden = torch.randn(n, h, generator=g).bfloat16().to(DEV)
    weight = (torch.randn(v, h, generator=g) * 0.2).bfloat16().to(DEV)
    labels = torch.randint(0, v, (n,), generator=g).to(DEV)
    up = (torch.rand(n, generator=g) + 0.5).to(DEV)
    monkeypatch.setattr(lm_head, "_kept_alive", [])

    def run(expect_kept, call=lm_head.fused_lm_head_logprobs, **kw):
        dh, dw = hidden.clone().requires_grad_(True), weight.clone().requires_grad_(True)
        out, _ = call(dh, dw, labels, **kw)
        assert (sum(r() is not None for r in lm_head._kept_alive) == 1) == expect_kept
        out.backward(up)
        assert all(r() is None for r in lm_head._kept_alive)  # given back with the graph
        return out.detach(), dh.grad, dw.grad

    def checkpointed(*args, **kw):
        return torch.utils.checkpoint.checkpoint(lm_head.fused_lm_head_logprobs, *args, use_reentrant=False, **kw)

    kept = run(True)
    others = [run(False, keep_logits=False), run(False, call=checkpointed)]
    with monkeypatch.context() as m:
        m.setattr(lm_head, "KEPT_UNASKED", 0)
        m.setattr(lm_head, "_free_bytes", lambda dev: 0)
        others.append(run(False))
    with monkeypatch.context() as m:
        m.setattr(lm_head, "KEPT_BUDGET", 0)
        others.append(run(False))
    for other in others:
        for a, b in zip(kept, other):
            assert torch.equal(a, b)


@pytest.mark.gpu
def test_the_wrappers_pass_the_choice_on(monkeypatch):
    monkeypatch.setattr(lm_head, "_kept_alive", [])
    hidden = torch.randn(1, 40, 64, device=DEV).bfloat16().requires_grad_(True)
    labels = torch.randint(0, 300, (1, 40), device=DEV)
    head = olmo_core_train_modules.DPOLMHead(64, 300, device=DEV)
    head.keep_logits = False
    outs = [head(hidden, labels=labels).loss, lm_head.fused_linear_cross_entropy(hidden, head.w_out.weight, labels, keep_logits=False)]
    assert not lm_head._kept_alive
    head.keep_logits = True
    outs.append(head(hidden, labels=labels).loss)
    assert len(lm_head._kept_alive) == 1 and all(o.requires_grad for o in outs)
