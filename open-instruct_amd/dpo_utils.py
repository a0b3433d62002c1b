"""DPO-family sequence losses on the GPU.

Names and signatures follow open_instruct/dpo_utils.py in the reference (``dpo_loss`` :523-563,
``wpo_loss`` :566-613, ``simpo_loss`` :617-642, ``compute_loss`` :645-686, ``_get_batch_logps``
:689-712, ``process_batch`` :715-731, ``concatenated_inputs`` :734-763, ``concatenated_forward``
:826-878, ``separate_forward`` :881-956, ``concatenated_forward_olmo`` :959-1019,
``build_reference_logprobs_cache`` :405-520).
"""

from __future__ import annotations

import contextlib
import dataclasses
import enum
import pathlib
from collections.abc import Callable, Iterable

import torch
import torch.distributed as dist

from . import _lib, lm_head, model_utils, olmo_core_utils, padding_free_collator
from .padding_free_collator import get_batch_logps_padded


class DPOLossType(str, enum.Enum):
    """The preference losses of the reference and what each one needs; open_instruct/dpo_utils.py:76-92.
    A string enum: members compare equal to their names, which is also what :func:`compute_loss` and
    :func:`fused_loss_olmo` accept in ``args.loss_type``."""

    dpo = "dpo"
    dpo_norm = "dpo_norm"
    simpo = "simpo"
    wpo = "wpo"

    def __str__(self) -> str:
        return self.value

    @property
    def is_average_loss(self) -> bool:
        """Per-sequence logprobs are token means rather than sums."""
        return self.value in ("simpo", "dpo_norm")

    @property
    def needs_reference_model(self) -> bool:
        return self.value in ("dpo", "dpo_norm", "wpo")

    @property
    def computes_reward_metrics(self) -> bool:
        return self.value in ("dpo", "dpo_norm")


class _SigmoidPairLoss(torch.autograd.Function):
    @staticmethod
    def forward(ctx, pc, pr, rc, rr, weights, beta, label_smoothing, margin):
        dev = _lib.require_gpu(pc, pr, rc, rr, weights)
        shape = pc.shape
        pc_c, pr_c = _lib.f32c(pc).reshape(-1), _lib.f32c(pr).reshape(-1)
        rc_c = _lib.f32c(rc).reshape(-1) if rc is not None else None
        rr_c = _lib.f32c(rr).reshape(-1) if rr is not None else None
        w_c = _lib.f32c(weights).reshape(-1) if weights is not None else None
        n = pc_c.numel()
        out = torch.empty((3, n), dtype=torch.float32, device=dev)
        at = out.data_ptr()
        _lib.call(
            "oi_dpo_sigmoid_fwd", pc_c.data_ptr(), pr_c.data_ptr(), _lib.ptr(rc_c), _lib.ptr(rr_c), _lib.ptr(w_c), n,
            beta, label_smoothing, margin, at, at + 4 * n, at + 8 * n, _lib.stream_of(pc_c),
        )  # fmt: skip
        ctx.save_for_backward(pc_c, pr_c, rc_c, rr_c, w_c)
        ctx.meta = (beta, label_smoothing, margin, shape, pc.dtype, pr.dtype)
        losses, cr, rj = (t.reshape(shape) for t in out.unbind(0))
        ctx.mark_non_differentiable(cr, rj)
        ctx.set_materialize_grads(False)  # of the rewards: two fills that nobody reads
        return losses, cr, rj

    @staticmethod
    def backward(ctx, g_losses, _g_cr, _g_rj):
        pc_c, pr_c, rc_c, rr_c, w_c = ctx.saved_tensors
        beta, ls, margin, shape, dt_c, dt_r = ctx.meta
        n = pc_c.numel()
        g = _lib.f32c(g_losses).reshape(-1) if g_losses is not None else torch.zeros_like(pc_c)
        d = torch.empty((2, n), dtype=torch.float32, device=g.device)
        _lib.call(
            "oi_dpo_sigmoid_bwd", pc_c.data_ptr(), pr_c.data_ptr(), _lib.ptr(rc_c), _lib.ptr(rr_c), _lib.ptr(w_c),
            g.data_ptr(), n, beta, ls, margin, d.data_ptr(), d.data_ptr() + 4 * n, _lib.stream_of(g),
        )  # fmt: skip
        d_c, d_r = d.unbind(0)
        return d_c.reshape(shape).to(dt_c), d_r.reshape(shape).to(dt_r), None, None, None, None, None, None


def dpo_loss(
    policy_chosen_logps: torch.Tensor,
    policy_rejected_logps: torch.Tensor,
    reference_chosen_logps: torch.Tensor,
    reference_rejected_logps: torch.Tensor,
    beta: float,
    reference_free: bool = False,
    label_smoothing: float = 0.0,
) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """Sigmoid DPO loss per pair and detached rewards; drop-in for open_instruct/dpo_utils.py:523-563.

    ``reference_free`` drops the reference log-ratio from the loss only; the rewards still use the
    provided reference logps, as in the reference.
    """
    if reference_free:
        losses, _, _ = _SigmoidPairLoss.apply(
            policy_chosen_logps, policy_rejected_logps, None, None, None, float(beta), float(label_smoothing), 0.0
        )
        with torch.no_grad():
            _, cr, rj = _SigmoidPairLoss.apply(
                policy_chosen_logps.detach(), policy_rejected_logps.detach(), reference_chosen_logps.detach(),
                reference_rejected_logps.detach(), None, float(beta), float(label_smoothing), 0.0,
            )  # fmt: skip
        return losses, cr, rj
    return _SigmoidPairLoss.apply(
        policy_chosen_logps, policy_rejected_logps, reference_chosen_logps.detach(),
        reference_rejected_logps.detach(), None, float(beta), float(label_smoothing), 0.0,
    )  # fmt: skip


def simpo_loss(
    policy_chosen_logps: torch.Tensor,
    policy_rejected_logps: torch.Tensor,
    beta: float,
    gamma_beta_ratio: float,
    label_smoothing: float = 0.0,
) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """SimPO loss (margin ``gamma/beta``, no reference model); open_instruct/dpo_utils.py:617-642."""
    return _SigmoidPairLoss.apply(
        policy_chosen_logps, policy_rejected_logps, None, None, None, float(beta), float(label_smoothing),
        float(gamma_beta_ratio),
    )  # fmt: skip


def wpo_loss(
    policy_chosen_logps: torch.Tensor,
    policy_rejected_logps: torch.Tensor,
    reference_chosen_logps: torch.Tensor,
    reference_rejected_logps: torch.Tensor,
    beta: float,
    chosen_loss_mask: torch.Tensor,
    rejected_loss_mask: torch.Tensor,
    label_smoothing: float = 0.0,
) -> tuple[torch.Tensor, torch.Tensor, torch.Tensor]:
    """WPO: the DPO pair loss times ``min(1, exp(avg_c + avg_r))``; open_instruct/dpo_utils.py:566-613.

    Follows the reference literally, including that the weights are not detached: the gradient
    flows through them as well, so the weight factor is assembled with differentiable tensor ops on
    the ``[bs]`` vectors and multiplied onto the kernel's per-pair loss.
    """
    avg_c = (policy_chosen_logps * chosen_loss_mask).sum(-1) / chosen_loss_mask.sum(-1)
    avg_r = (policy_rejected_logps * rejected_loss_mask).sum(-1) / rejected_loss_mask.sum(-1)
    weights = torch.clamp(torch.exp(avg_c + avg_r), max=1)
    base, cr, rj = _SigmoidPairLoss.apply(
        policy_chosen_logps, policy_rejected_logps, reference_chosen_logps.detach(),
        reference_rejected_logps.detach(), None, float(beta), float(label_smoothing), 0.0,
    )  # fmt: skip
    return base * weights, cr, rj


def compute_loss(args, batch: dict, policy_chosen_logps, policy_rejected_logps, reference_cache=None):
    """Dispatch on ``args.loss_type``; open_instruct/dpo_utils.py:645-686.

    ``reference_cache[batch["index"]]`` must return a mapping with ``chosen_logps`` /
    ``rejected_logps`` (the reference's ``TensorCache``, open_instruct/model_utils.py:92-115).
    """
    loss_type = str(getattr(args.loss_type, "value", args.loss_type))
    if loss_type in ("dpo", "dpo_norm"):
        assert reference_cache is not None
        ref = reference_cache[batch["index"]]
        return dpo_loss(
            policy_chosen_logps, policy_rejected_logps, ref["chosen_logps"], ref["rejected_logps"], beta=args.beta,
            label_smoothing=args.label_smoothing,
        )  # fmt: skip
    if loss_type == "simpo":
        return simpo_loss(
            policy_chosen_logps, policy_rejected_logps, beta=args.beta, gamma_beta_ratio=args.gamma_beta_ratio,
            label_smoothing=args.label_smoothing,
        )  # fmt: skip
    if loss_type == "wpo":
        assert reference_cache is not None
        ref = reference_cache[batch["index"]]
        return wpo_loss(
            policy_chosen_logps, policy_rejected_logps, ref["chosen_logps"], ref["rejected_logps"], beta=args.beta,
            label_smoothing=args.label_smoothing, chosen_loss_mask=batch["chosen_labels"] != -100,
            rejected_loss_mask=batch["rejected_labels"] != -100,
        )  # fmt: skip
    raise ValueError(f"Unknown loss type: {args.loss_type}")


def _get_batch_logps(
    per_token_logps: torch.Tensor, labels: torch.Tensor, average_log_prob: bool = False
) -> torch.Tensor:
    """Per-row sum or mean of kept per-token logps; drop-in for open_instruct/dpo_utils.py:689-712."""
    return get_batch_logps_padded(per_token_logps, labels, average_log_prob)


def _pad_to(t: torch.Tensor, length: int, value: int) -> torch.Tensor:
    if t.shape[1] == length:
        return t
    pad = torch.full((t.shape[0], length - t.shape[1]), value, dtype=t.dtype, device=t.device)
    return torch.cat([t, pad], dim=1)


def concatenated_inputs(batch: dict) -> dict:
    """Chosen and rejected stacked along the batch dim, padded to a common length.

    Integer plumbing of open_instruct/dpo_utils.py:734-763: ``labels`` pad with -100, everything
    else with 0.
    """
    keys = [k for k in batch if k.startswith("chosen_") and isinstance(batch[k], torch.Tensor)]
    max_len = max(batch["chosen_input_ids"].shape[1], batch["rejected_input_ids"].shape[1])
    out = {}
    for k in keys:
        name = k[len("chosen_") :]
        pad = -100 if "labels" in name else 0
        out[f"concatenated_{name}"] = torch.cat(
            [_pad_to(batch[k], max_len, pad), _pad_to(batch[f"rejected_{name}"], max_len, pad)], dim=0
        )
    return out


def _split_pairs(logps: torch.Tensor, bs: int) -> tuple[torch.Tensor, torch.Tensor]:
    """Chosen sequences come first in every concatenated batch, rejected ones after them."""
    return logps[:bs], logps[bs:]


def _sequence_logps(per_token, labels, concat: dict, packing: bool, average_log_prob: bool) -> torch.Tensor:
    if packing:
        return padding_free_collator.get_batch_logps(
            per_token, labels, concat["concatenated_cu_seq_lens_k"], average_log_prob
        )
    return _get_batch_logps(per_token, labels, average_log_prob)


def concatenated_forward(
    model, batch: dict, average_log_prob: bool = False, output_router_logits: bool = False, packing: bool = False,
    fused_head: bool = False,
):  # fmt: skip
    """One model forward over chosen+rejected, then per-sequence logps; open_instruct/dpo_utils.py:826-878.

    HuggingFace interface: ``model(**inputs).logits``; with ``output_router_logits`` the model is
    asked for its router logits and the ``aux_loss`` of its output is passed through.  Returns
    ``(chosen_logps, rejected_logps, aux_loss)``.  ``fused_head=True`` (not in the reference) runs
    the model's trunk only and sends its hidden states through the fused lm_head, so the model never forms
    its ``[B, T, V]`` logits and prompt / padding positions are not multiplied; same results.
    """
    if packing:
        concat, bs = padding_free_collator.concatenated_inputs(batch)
    else:
        concat = concatenated_inputs(batch)
        bs = batch["chosen_input_ids"].shape[0]
    inputs = {
        k.replace("concatenated_", ""): v
        for k, v in concat.items()
        if k.startswith("concatenated_") and not k.endswith("labels")
    }
    aux_loss = None
    labels = concat["concatenated_labels"]
    if fused_head:
        if output_router_logits:
            raise ValueError("fused_head runs the trunk only: the router's aux_loss is not available")
        per_token = lm_head.per_token_logps_from_trunk(model, labels, **inputs)
    else:
        if output_router_logits:
            output = model(**inputs, output_router_logits=True)
            aux_loss = output.aux_loss
        else:
            output = model(**inputs)
        logits = getattr(output, "logits", output)
        per_token = padding_free_collator.calculate_per_token_logps(logits, labels)
    chosen, rejected = _split_pairs(_sequence_logps(per_token, labels, concat, packing, average_log_prob), bs)
    return chosen, rejected, aux_loss


def process_batch(batch: dict, prefix: str, pad_value: int = 0) -> dict[str, torch.Tensor]:
    """The tensors of one side (``"chosen"`` / ``"rejected"``) under their un-prefixed names;
    open_instruct/dpo_utils.py:715-731 (``pad_value`` is unused there as well)."""
    del pad_value
    lead = prefix + "_"
    return {k[len(lead) :]: v for k, v in batch.items() if k.startswith(prefix) and isinstance(v, torch.Tensor)}


def separate_forward(
    model, batch: dict, average_log_prob: bool = False, output_router_logits: bool = False, fused_head: bool = False
):
    """Chosen and rejected sequences in two model forwards (selectable through ``forward_fn``);
    open_instruct/dpo_utils.py:881-956.  The logits are read in their own dtype with fp32
    accumulation, so the reference's fp32 copy of them is not made.  ``fused_head`` as in
    :func:`concatenated_forward`."""
    if fused_head and output_router_logits:
        raise ValueError("fused_head runs the trunk only: the router's aux_loss is not available")
    logps, aux = [], []
    for side in ("chosen", "rejected"):
        part = process_batch(batch, side)
        if fused_head:
            per_token = lm_head.per_token_logps_from_trunk(
                model, part["labels"], input_ids=part["input_ids"], attention_mask=part["attention_mask"]
            )
            output = None
        else:
            kwargs = {"output_router_logits": True} if output_router_logits else {}
            output = model(input_ids=part["input_ids"], attention_mask=part["attention_mask"], **kwargs)
            per_token = padding_free_collator.calculate_per_token_logps(output.logits, part["labels"])
        logps.append(_get_batch_logps(per_token, part["labels"], average_log_prob))
        aux.append(output.aux_loss if output_router_logits else None)
        del output, per_token
    aux_loss = torch.cat(aux, dim=0) if output_router_logits and all(a is not None for a in aux) else None
    return logps[0], logps[1], aux_loss


def concatenated_forward_olmo(
    model,
    batch: dict,
    average_log_prob: bool = False,
    packing: bool = False,
    output_router_logits: bool = False,
):
    """Chosen+rejected in one forward of a model with the olmo-core interface;
    open_instruct/dpo_utils.py:959-1019.

    The labels go INTO the model: its LM head (:class:`~open_instruct_amd.olmo_core_train_modules.DPOLMHead`)
    returns the per-token logps as ``output.loss`` instead of logits.
    Packed batches pass ``position_ids`` and the document lengths derived from ``cu_seq_lens_k``.
    ``output_router_logits`` is accepted and unused, ``aux_loss`` is always None, as in the reference.
    """
    del output_router_logits
    if packing:
        concat, bs = padding_free_collator.concatenated_inputs(batch)
    else:
        concat = concatenated_inputs(batch)
        bs = batch["chosen_input_ids"].shape[0]
    labels = concat["concatenated_labels"]
    input_ids = concat["concatenated_input_ids"]
    if packing:
        doc_lens, max_doc_lens = olmo_core_utils.doc_lens_from_cu_seq_lens(
            concat["concatenated_cu_seq_lens_k"], seq_len=input_ids.shape[-1]
        )
        output = model(
            input_ids, labels=labels, position_ids=concat.get("concatenated_position_ids"), doc_lens=doc_lens,
            max_doc_lens=max_doc_lens,
        )  # fmt: skip
    else:
        output = model(input_ids, labels=labels)
    chosen, rejected = _split_pairs(_sequence_logps(output.loss, labels, concat, packing, average_log_prob), bs)
    return chosen, rejected, None


def separate_forward_olmo(model, batch: dict, average_log_prob: bool = False, output_router_logits: bool = False):
    """Chosen and rejected sequences in two forwards of a model with the olmo-core interface;
    open_instruct/dpo_utils.py:1022-1054.

    As in :func:`concatenated_forward_olmo` the labels go into the model and its
    :class:`~open_instruct_amd.olmo_core_train_modules.DPOLMHead` returns the per-token logps as
    ``output.loss``; only one side's activations are alive at a time.  ``output_router_logits`` is accepted
    and unused, ``aux_loss`` is always None, as in the reference.  (The reference empties the allocator's
    cache after each side, to give back a side's logits.  Here no block of that kind is free between the sides: what a
    trained head may keep, at most 4 GiB over both, is in use until the backward; its ``keep_logits = False`` keeps
    nothing.)
    """
    del output_router_logits
    sides = []
    for side in ("chosen", "rejected"):
        part = process_batch(batch, side)
        output = model(part["input_ids"], labels=part["labels"])
        sides.append(_get_batch_logps(output.loss, part["labels"], average_log_prob=average_log_prob))
        del output, part
    return sides[0], sides[1], None


@dataclasses.dataclass
class FusedDPOResult:
    """What :func:`dpo_loss_on_hidden` returns.  ``loss`` (``losses.mean()``) carries the graph: its
    ``backward()`` hands the gradients computed inside the call to ``hidden`` and ``weight``; every
    other field is detached."""

    loss: torch.Tensor
    losses: torch.Tensor
    chosen_logps: torch.Tensor
    rejected_logps: torch.Tensor
    chosen_rewards: torch.Tensor
    rejected_rewards: torch.Tensor
    per_token_logps: torch.Tensor | None


# slab size of the no-recompute DPO step when the caller names none (scored tokens per slab); a slab holds
# whole chosen / rejected pairs, so it should not be smaller than the largest pair of the batch
DEFAULT_DPO_SLAB_TOKENS = 8192


def dpo_loss_on_hidden(
    hidden: torch.Tensor,
    weight: torch.Tensor,
    labels: torch.Tensor,
    reference_chosen_logps: torch.Tensor | None,
    reference_rejected_logps: torch.Tensor | None,
    beta: float,
    *,
    cu_seq_lens: torch.Tensor | None = None,
    average_log_prob: bool = False,
    reference_free: bool = False,
    label_smoothing: float = 0.0,
    gamma_beta_ratio: float = 0.0,
    token_slabs: bool | int = True,
) -> FusedDPOResult:
    """Sigmoid preference loss straight from the final hidden states of a concatenated chosen + rejected
    batch, with both gradients and nothing recomputed.

    One call for the reference's sequence "``DPOLMHead`` (``w_out``, ``calculate_per_token_logps``:
    open_instruct/olmo_core_train_modules.py:71-76) -> per-sequence logps
    (open_instruct/padding_free_collator.py:202-229 / open_instruct/dpo_utils.py:689-712) -> ``dpo_loss`` /
    ``simpo_loss`` (open_instruct/dpo_utils.py:523-563, :617-642) -> ``losses.mean().backward()``
    (open_instruct/olmo_core_train_modules.py:190-207)".  Because the loss is known inside the call, a
    slab of token rows can be finished (forward, upstream gradient, ``d_hidden``, its share of ``d_weight``)
    before the next one starts, so a trainable lm_head costs 6·N·H·V of matrix work instead of the 8·N·H·V of
    the differentiable route through :class:`~open_instruct_amd.olmo_core_train_modules.DPOLMHead`, whose
    backward recomputes the logits of all but small batches.  The ``[tokens, vocab]`` logits never exist; the scratch is a
    ``[slab, vocab]`` bf16 buffer and an fp32 ``[vocab, hidden]``.

    ``hidden`` is ``[2 * bs, T, H]`` bf16 with ``labels`` ``[2 * bs, T]`` (padded; chosen rows first:
    open_instruct/dpo_utils.py:734-763), or ``[1, T_total, H]`` with ``labels`` ``[1, T_total]`` and
    ``cu_seq_lens`` int32 ``[2 * bs + 1]`` (packed: open_instruct/padding_free_collator.py:166-199).  The
    labels are the batch's own, unshifted; position ``t`` is scored against ``labels[t + 1]`` where that
    is not -100, other positions are not multiplied.  ``average_log_prob`` as in ``dpo_norm`` / ``simpo``;
    ``reference_free`` drops the reference term from the loss (the rewards keep it, as in the reference);
    ``gamma_beta_ratio`` is simpo's margin (pass no reference logps for simpo).

    ``token_slabs``: ``True`` = slabs of ``DEFAULT_DPO_SLAB_TOKENS`` scored tokens, or a number.  A slab
    is filled with whole pairs (a token's upstream gradient needs the logprob sums of both sequences of
    its pair); a pair that is larger than a slab still gives the right result but its tokens go through a
    recomputing backward, so pass at least the largest pair's scored tokens.  ``result.loss.backward()``
    may be called once.
    """
    from . import grpo_utils

    if hidden.ndim != 3 or labels.ndim != 2 or tuple(hidden.shape[:2]) != tuple(labels.shape):
        raise ValueError(f"hidden {tuple(hidden.shape)} and labels {tuple(labels.shape)} must be [B, T, H] and [B, T]")
    packed = cu_seq_lens is not None
    if packed and labels.shape[0] != 1:
        raise ValueError("a packed batch is one row: hidden [1, T, H], labels [1, T]")
    n_seqs = int(cu_seq_lens.numel()) - 1 if packed else int(labels.shape[0])
    if n_seqs < 2 or n_seqs % 2:
        raise ValueError(f"{n_seqs} sequences: a concatenated batch holds the chosen and the rejected half")
    if (reference_chosen_logps is None) != (reference_rejected_logps is None):
        raise ValueError("pass both reference logps or neither")
    bs, total = n_seqs // 2, int(labels.shape[1])
    dev = _lib.require_gpu(hidden, weight, labels, cu_seq_lens, reference_chosen_logps, reference_rejected_logps)
    if hidden.dtype != torch.bfloat16 or weight.dtype != torch.bfloat16:
        raise ValueError("the fused lm_head expects bf16 hidden states and weight")
    h, v = int(hidden.shape[-1]), int(weight.shape[0])
    if weight.ndim != 2 or weight.shape[1] != h or h % 64:
        raise ValueError(f"weight {tuple(weight.shape)} does not fit hidden size {h} (a multiple of 64)")
    ref_c = None if reference_chosen_logps is None else _lib.f32c(reference_chosen_logps.detach()).reshape(-1)
    ref_r = None if reference_rejected_logps is None else _lib.f32c(reference_rejected_logps.detach()).reshape(-1)
    if ref_c is not None and (ref_c.numel() != bs or ref_r.numel() != bs):
        raise ValueError(f"reference logps must hold {bs} entries each")
    loss_ref_c, loss_ref_r = (None, None) if reference_free else (ref_c, ref_r)
    slab_tokens = DEFAULT_DPO_SLAB_TOKENS if token_slabs is True else int(token_slabs)
    if slab_tokens < 256:
        raise ValueError("token_slabs must be True or a number of tokens (at least 256)")
    n = labels.numel()
    hid = hidden.detach().reshape(n, h).contiguous()
    w = weight.detach().contiguous()
    lab = labels.to(torch.int64).contiguous()
    cu = None if not packed else cu_seq_lens.to(torch.int32).contiguous()
    per_token = torch.empty(labels.shape, dtype=torch.float32, device=dev)
    seq_logps = torch.empty(n_seqs, dtype=torch.float32, device=dev)
    out = torch.empty((3, bs), dtype=torch.float32, device=dev)
    wants_grad = torch.is_grad_enabled() and (hidden.requires_grad or weight.requires_grad)
    if not wants_grad:
        shifted = padding_free_collator.shift_labels(lab)
        with torch.no_grad():
            lp, _ = lm_head.fused_lm_head_logprobs(hidden, weight, shifted, mask=shifted != -100)
            logps = _sequence_logps(lp, lab, {"concatenated_cu_seq_lens_k": cu}, packed, average_log_prob)
            losses, _, _ = _SigmoidPairLoss.apply(
                logps[:bs], logps[bs:], loss_ref_c, loss_ref_r, None, float(beta), float(label_smoothing),
                float(gamma_beta_ratio),
            )  # fmt: skip
            _, cr, rj = _SigmoidPairLoss.apply(logps[:bs], logps[bs:], ref_c, ref_r, None, float(beta), 0.0, 0.0)
        return FusedDPOResult(losses.mean(), losses, logps[:bs], logps[bs:], cr, rj, lp)
    d_hidden = torch.empty_like(hid)
    d_weight = torch.empty_like(w) if weight.requires_grad else None
    lib = _lib.load()
    ws_bytes = lib.oi_lmhead_dpo_workspace_bytes(n_seqs, total, int(packed), h, v, int(d_weight is not None), slab_tokens)
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
    _lib.call(
        "oi_lmhead_dpo_fwd_bwd", hid.data_ptr(), w.data_ptr(), lab.data_ptr(), _lib.ptr(cu), n_seqs, total, h, v, 1.0,
        _lib.ptr(loss_ref_c), _lib.ptr(loss_ref_r), float(beta), float(label_smoothing), float(gamma_beta_ratio),
        int(bool(average_log_prob)), 1.0 / bs, per_token.data_ptr(), seq_logps.data_ptr(), out[0].data_ptr(),
        out[1].data_ptr(), out[2].data_ptr(), d_hidden.data_ptr(), _lib.ptr(d_weight), slab_tokens, ws.data_ptr(),
        ws_bytes, _lib.stream_of(hid),
    )  # fmt: skip
    losses, cr, rj = out.unbind(0)
    if reference_free and ref_c is not None:  # the rewards keep the reference term
        cr, rj = float(beta) * (seq_logps[:bs] - ref_c), float(beta) * (seq_logps[bs:] - ref_r)
    loss = grpo_utils._AttachHeadGrads.apply(losses.mean(), hidden, weight, d_hidden.reshape(hidden.shape), d_weight)
    return FusedDPOResult(loss, losses, seq_logps[:bs], seq_logps[bs:], cr, rj, per_token)


def fused_loss_olmo(
    model,
    batch: dict,
    args,
    reference_cache=None,
    average_log_prob: bool | None = None,
    packing: bool = False,
    token_slabs: bool | int = True,
) -> FusedDPOResult:
    """``concatenated_forward_olmo`` -> ``compute_loss`` -> ``losses.mean()`` (the body of
    open_instruct/olmo_core_train_modules.py:190-207) with the lm_head, the per-sequence sums and the
    pair loss in one no-recompute call.

    The model must follow the olmo-core interface with a
    :class:`~open_instruct_amd.olmo_core_train_modules.DPOLMHead` as ``model.lm_head``: the labels go into
    the model, the head receives the final hidden states and, because a loss specification is set on it for
    the duration of this call, computes the loss and both gradients right there (see
    :func:`dpo_loss_on_hidden`).  ``args`` is duck-typed like the reference's (``loss_type``, ``beta``,
    ``label_smoothing``, ``gamma_beta_ratio``); ``loss_type`` ``dpo``, ``dpo_norm`` and ``simpo`` take the
    one-call form.  ``wpo`` (whose weight puts the finished sequence sums of a pair inside the gradient)
    takes the reference's own sequence here, :func:`concatenated_forward_olmo` -> :func:`compute_loss` ->
    ``losses.mean()`` on the differentiable fused head (its backward recomputes the logits), and comes
    back in the same result type with ``per_token_logps=None``.
    ``result.loss.backward()`` continues into the trunk through the hidden states.
    """
    loss_type = str(getattr(args.loss_type, "value", args.loss_type))
    if loss_type not in ("dpo", "dpo_norm", "simpo", "wpo"):
        raise ValueError(f"Unknown loss type: {args.loss_type}")
    if average_log_prob is None:
        average_log_prob = loss_type in ("dpo_norm", "simpo")
    if loss_type == "wpo":
        chosen, rejected, _ = concatenated_forward_olmo(model, batch, average_log_prob=average_log_prob, packing=packing)
        losses, chosen_rewards, rejected_rewards = compute_loss(args, batch, chosen, rejected, reference_cache)
        return FusedDPOResult(
            loss=losses.mean(), losses=losses.detach(), chosen_logps=chosen.detach(), rejected_logps=rejected.detach(),
            chosen_rewards=chosen_rewards, rejected_rewards=rejected_rewards, per_token_logps=None,
        )  # fmt: skip
    if packing:
        concat, _ = padding_free_collator.concatenated_inputs(batch)
    else:
        concat = concatenated_inputs(batch)
    labels = concat["concatenated_labels"]
    input_ids = concat["concatenated_input_ids"]
    ref_c = ref_r = None
    if loss_type != "simpo":
        assert reference_cache is not None
        ref = reference_cache[batch["index"]]
        ref_c, ref_r = ref["chosen_logps"], ref["rejected_logps"]
    head = model.lm_head
    head.fused_loss = dict(
        reference_chosen_logps=ref_c, reference_rejected_logps=ref_r, beta=args.beta,
        cu_seq_lens=concat["concatenated_cu_seq_lens_k"] if packing else None, average_log_prob=average_log_prob,
        label_smoothing=getattr(args, "label_smoothing", 0.0),
        gamma_beta_ratio=getattr(args, "gamma_beta_ratio", 0.0) if loss_type == "simpo" else 0.0,
        token_slabs=token_slabs,
    )  # fmt: skip
    try:
        if packing:
            doc_lens, max_doc_lens = olmo_core_utils.doc_lens_from_cu_seq_lens(
                concat["concatenated_cu_seq_lens_k"], seq_len=input_ids.shape[-1]
            )
            model(
                input_ids, labels=labels, position_ids=concat.get("concatenated_position_ids"), doc_lens=doc_lens,
                max_doc_lens=max_doc_lens,
            )  # fmt: skip
        else:
            model(input_ids, labels=labels)
        result = head.fused_result
    finally:
        head.fused_loss = None
        head.fused_result = None
    if result is None:
        raise RuntimeError("the model's lm_head did not run the fused loss (is it a DPOLMHead?)")
    return result


def build_reference_logprobs_cache(
    model: torch.nn.Module,
    dataloader: Iterable[dict],
    average_log_prob: bool,
    forward_fn: Callable,
    full_dataset_size: int,
    device: torch.device,
    cache_path: pathlib.Path | str,
    is_main_process: bool,
    model_dims=None,
    use_lora: bool = False,
    disable_adapter_context: Callable[[], contextlib.AbstractContextManager] | None = None,
    forward_kwargs: dict | None = None,
) -> model_utils.TensorCache:
    """Reference-policy logps of every sample, computed once; open_instruct/dpo_utils.py:405-520,
    same parameters in the same order (both reference callers pass them by keyword:
    open_instruct/dpo_tune_cache.py:522-534, open_instruct/dpo.py:310).

    One no-grad pass over ``dataloader``: ``forward_fn(model, batch, average_log_prob=...)`` returns
    ``(chosen_logps, rejected_logps, aux)``, which are scattered to ``batch["index"]``.  Batches
    flagged ``is_padding`` are skipped; an index that no batch covered raises, as in the reference.
    An existing ``cache_path`` is loaded instead of recomputed.  ``is_main_process`` gates the
    directory check and the write of the new cache; with ``use_lora`` the forward runs inside
    ``disable_adapter_context()`` when one is given; ``model_dims`` only feeds the reference's
    progress-bar MFU read-out and is accepted and unused.  The barriers and the MAX all-reduce across
    ranks (open_instruct/dpo_utils.py:456,494-495,518) run when a process group is initialised.
    """
    del model_dims
    cache_path = pathlib.Path(cache_path)
    if cache_path.exists():
        return model_utils.TensorCache.from_disk(cache_path, device=device)
    if is_main_process:
        cache_path.parent.mkdir(parents=True, exist_ok=True)
        probe = cache_path.parent / f".write_test_{cache_path.stem}"
        try:
            probe.touch()
            probe.unlink()
        except (OSError, PermissionError) as e:
            raise RuntimeError(
                f"Cannot write to cache directory {cache_path.parent}: {e}. "
                f"Set REFERENCE_LOGPROBS_CACHE_PATH to a writable location."
            ) from e
    distributed = dist.is_available() and dist.is_initialized()
    if distributed:
        dist.barrier()
    model.eval()
    chosen = torch.full((full_dataset_size,), float("-inf"), dtype=torch.float32, device=device)
    rejected = torch.full((full_dataset_size,), float("-inf"), dtype=torch.float32, device=device)
    with torch.no_grad():
        for batch in dataloader:
            adapter_off = disable_adapter_context() if use_lora and disable_adapter_context is not None else None
            with adapter_off if adapter_off is not None else contextlib.nullcontext():
                chosen_logps, rejected_logps, _ = forward_fn(
                    model, batch, average_log_prob=average_log_prob, **(forward_kwargs or {})
                )
            if batch.get("is_padding", False):
                continue
            index = batch["index"].to(device).long()
            chosen[index] = chosen_logps.float()
            rejected[index] = rejected_logps.float()
    if distributed:
        dist.all_reduce(chosen, op=dist.ReduceOp.MAX)
        dist.all_reduce(rejected, op=dist.ReduceOp.MAX)
    missing = torch.where((chosen == float("-inf")) | (rejected == float("-inf")))[0]
    if len(missing) > 0:
        raise RuntimeError(
            f"Missing {len(missing)} indices during reference logprobs caching. First 10: {missing[:10].tolist()}"
        )
    model.train()
    cache = model_utils.TensorCache(tensors={"chosen_logps": chosen, "rejected_logps": rejected})
    if is_main_process:
        cache.to_disk(cache_path)
    if distributed:
        dist.barrier()
    return cache
