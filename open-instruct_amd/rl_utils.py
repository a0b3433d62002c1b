"""Masked mean and sequence packing on the GPU; same names and signatures as
open_instruct/rl_utils.py (``masked_mean`` :426-448, ``pack_sequences`` :227-375,
``PackedSequences`` :181-213)."""

from __future__ import annotations

import itertools
from dataclasses import dataclass

import numpy as np
import torch

from . import _lib


def _as_rows(values: torch.Tensor, mask: torch.Tensor, axis: int | None):
    """Reshape to values [extra, rows, cols] / mask [rows, cols] for the two reduction modes.

    axis=None: one row holding every mask element.  axis=k: the reduced mask dim becomes the
    column dim (moved last when it is not already), every other mask dim is a row.
    """
    extra_dims = values.ndim - mask.ndim
    if extra_dims < 0:
        raise ValueError(f"values {tuple(values.shape)} has fewer dims than mask {tuple(mask.shape)}")
    if tuple(values.shape[extra_dims:]) != tuple(mask.shape):
        try:  # the reference relies on broadcasting; make it explicit
            mask = mask.expand(values.shape[extra_dims:])
        except RuntimeError:
            raise ValueError(f"mask shape {tuple(mask.shape)} does not match values {tuple(values.shape)}") from None
    extra = 1
    for d in values.shape[:extra_dims]:
        extra *= d
    if axis is None:
        cols = mask.numel()
        return values.reshape(extra, 1, cols), mask.reshape(1, cols), extra_dims, 0
    ax = axis if axis >= 0 else axis + mask.ndim
    if not 0 <= ax < mask.ndim:
        raise IndexError(f"axis {axis} out of range for a mask with {mask.ndim} dims")
    if ax != mask.ndim - 1:
        mask = mask.movedim(ax, -1)
        values = values.movedim(extra_dims + ax, -1)
    cols = mask.shape[-1]
    rows = mask.numel() // max(cols, 1)
    return values.reshape(extra, rows, cols), mask.reshape(rows, cols), extra_dims, 1


class _MaskedMean(torch.autograd.Function):
    @staticmethod
    def forward(ctx, values3, mask2, axis_mode, denominator):
        dev = _lib.require_gpu(values3, mask2)
        v = _lib.f32c(values3)
        is_float = mask2.dtype.is_floating_point
        m = _lib.f32c(mask2) if is_float else _lib.mask_u8(mask2)
        extra, rows, cols = v.shape
        out = torch.empty(extra, dtype=torch.float32, device=dev)
        row_denoms = torch.empty(rows, dtype=torch.float32, device=dev)
        ws_bytes = _lib.load().oi_masked_mean_workspace_bytes(extra, rows, cols)
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
        _lib.call(
            "oi_masked_mean_fwd", v.data_ptr(), m.data_ptr(), int(is_float), extra, rows, cols, axis_mode,
            float(denominator), out.data_ptr(), row_denoms.data_ptr(), ws.data_ptr(), ws_bytes, _lib.stream_of(v),
        )  # fmt: skip
        ctx.save_for_backward(m, row_denoms)
        ctx.is_float = is_float
        ctx.shape = (extra, rows, cols)
        ctx.in_dtype = values3.dtype
        return out

    @staticmethod
    def backward(ctx, grad_out):
        m, row_denoms = ctx.saved_tensors
        extra, rows, cols = ctx.shape
        g = _lib.f32c(grad_out)
        dv = torch.empty(ctx.shape, dtype=torch.float32, device=g.device)
        _lib.call(
            "oi_masked_mean_bwd", g.data_ptr(), m.data_ptr(), int(ctx.is_float), row_denoms.data_ptr(), extra, rows,
            cols, dv.data_ptr(), _lib.stream_of(g),
        )  # fmt: skip
        return dv.to(ctx.in_dtype), None, None, None


def masked_mean(
    values: torch.Tensor, mask: torch.Tensor, axis: int | None = None, denominator: float | None = None
) -> torch.Tensor:
    """Mean of ``values`` over the positions selected by ``mask``.

    Drop-in for open_instruct/rl_utils.py:426-448: extra leading dims of ``values`` are kept;
    ``axis=None`` divides the masked sum by ``mask.sum()`` (or ``denominator``); ``axis=k`` takes
    per-slice means along mask dim ``k`` and averages them; an empty mask gives 0.
    """
    if denominator is not None and not isinstance(denominator, (int, float)):
        denominator = float(denominator)
    if values.numel() == 0 or mask.numel() == 0:
        raise ValueError("masked_mean needs non-empty tensors")
    v3, m2, extra_dims, axis_mode = _as_rows(values, mask, axis)
    if denominator is not None and denominator <= 0:
        # the reference returns zeros for a non-positive constant denominator
        return (v3.sum(dim=(1, 2)) * 0.0).reshape(values.shape[:extra_dims])
    out = _MaskedMean.apply(v3, m2, axis_mode, 0.0 if denominator is None else float(denominator))
    return out.reshape(values.shape[:extra_dims])


# ----------------------------------------------------------------------------------------------
# sequence packing
# ----------------------------------------------------------------------------------------------
@dataclass
class PackedSequences:
    """Same fields as open_instruct/rl_utils.py:181-213; every tensor lives on the GPU and the
    per-row tensors of one field are views into one flat buffer (rows back to back)."""

    query_responses: list[torch.Tensor]
    attention_masks: list[torch.Tensor]
    response_masks: list[torch.Tensor]
    original_responses: list[list[int]]
    advantages: list[torch.Tensor] | None = None
    num_actions: list[torch.Tensor] | None = None
    position_ids: list[torch.Tensor] | None = None
    packed_seq_lens: list[torch.Tensor] | None = None
    vllm_logprobs: list[torch.Tensor] | None = None
    dones: list[torch.Tensor] | None = None
    rewards: list[torch.Tensor] | None = None


_INT64 = range(-(2**63), 2**63)


def _native(name: str, *args) -> bool:
    """Whether the native reader took these lists (otherwise its outputs mean nothing)."""
    lib = _lib.pylists()
    return lib is not None and getattr(lib, name)(*args) == 0


def _offsets(seqs) -> np.ndarray:
    """Where each sequence starts in the flat array, and the end."""
    n = len(seqs)
    offsets = np.empty(n + 1, dtype=np.int64)
    if not _native("oi_py_offsets", seqs, n, offsets.ctypes.data):
        offsets[0] = 0
        np.cumsum(np.fromiter((len(x) for x in seqs), dtype=np.int64, count=n), out=offsets[1:])
    return offsets


def _walk(seqs, offsets: np.ndarray, dtype) -> np.ndarray:
    """Sequences of any kind, flattened element by element."""
    return np.fromiter(itertools.chain.from_iterable(seqs), dtype=dtype, count=int(offsets[-1]))


def _fill_ints(seqs, offsets: np.ndarray, out: np.ndarray, skip) -> np.ndarray:
    """Flattens integer sequences into ``out``; returns how many elements of each differ from ``skip``."""
    n = len(offsets) - 1
    others = np.empty(n, dtype=np.int64)
    if type(skip) is int and skip in _INT64:
        if _native("oi_py_flatten_ints", seqs, n, offsets.ctypes.data, skip, out.ctypes.data, others.ctypes.data):
            return others
    out[:] = _walk(seqs, offsets, np.int64)
    before = np.zeros(len(out) + 1, dtype=np.int64)
    np.cumsum(out != skip, out=before[1:])
    return before[offsets[1:]] - before[offsets[:-1]]


def _fill_flags(seqs, offsets: np.ndarray, out: np.ndarray) -> None:
    if not _native("oi_py_flatten_flags", seqs, len(offsets) - 1, offsets.ctypes.data, out.ctypes.data):
        out[:] = _walk(seqs, offsets, np.int64) != 0


def _fill_floats(seqs, offsets: np.ndarray, out: np.ndarray) -> None:
    if not _native("oi_py_flatten_floats", seqs, len(offsets) - 1, offsets.ctypes.data, out.ctypes.data):
        out[:] = _walk(seqs, offsets, np.float32)


class _Staging:
    """Arrays that go to the device together: sections of one pinned buffer, 16-byte aligned, and one copy."""

    def __init__(self, sizes: list[tuple[int, type]]):
        self.at, end = [], 0
        for count, dtype in sizes:
            self.at.append(end)
            end += (count * np.dtype(dtype).itemsize + 15) // 16 * 16
        self.host = torch.empty(max(end, 16), dtype=torch.uint8, pin_memory=True)
        raw = self.host.numpy()
        self.arrays = [
            raw[at : at + count * np.dtype(dtype).itemsize].view(dtype) for at, (count, dtype) in zip(self.at, sizes)
        ]

    def upload(self, dev) -> torch.Tensor:
        # the allocator of pinned memory hands the buffer out again only when the copy is through
        return self.host.to(dev, non_blocking=True)


def pack_sequences(
    queries: list[list[int]],
    responses: list[list[int]],
    masks: list[list[int]],
    pack_length: int,
    pad_token_id: int,
    vllm_logprobs: list[list[float]],
    min_num_batches: int = 1,
    mask_tool_use: bool = False,
    advantages=None,
    device: torch.device | str = "cuda",
) -> PackedSequences:
    """Pack query-response pairs into rows of at most ``pack_length`` tokens.

    Drop-in for open_instruct/rl_utils.py:227-375 (same greedy rule: a sequence that does not fit
    the current row starts a new one; ``min_num_batches`` shrinks the row length to
    ``total_tokens // min_num_batches``).  The ragged lists are flattened once on the host; the
    seven per-token outputs are written by one kernel launch and returned as GPU tensors.
    ``advantages`` (one value per sequence, optional) fills ``PackedSequences.advantages`` with
    the broadcast of open_instruct/data_loader.py:1509-1514 in the same launch; response masks
    keep the reference's int64 document ids (``.bool()`` them after use, as the reference does).
    """
    n = len(queries)
    if not (len(responses) == len(masks) == len(vllm_logprobs) == n):
        raise ValueError("queries, responses, masks and vllm_logprobs must have one length")
    q_off = _offsets(queries)
    r_off = _offsets(responses)
    dev = torch.device(device)
    with_adv = advantages is not None
    # queries, responses, tool mask, logprobs, their offsets, destinations, row bases, advantages, lengths
    staging = None
    if dev.type == "cuda" and n and torch.cuda.is_current_stream_capturing():
        # a recorded copy would read the pinned buffer at every replay, when it has long been handed out again
        raise RuntimeError("pack_sequences reads Python lists and cannot be captured into a graph")
    if dev.type == "cuda" and n:
        n_q, n_r = int(q_off[-1]), int(r_off[-1])
        staging = _Staging(
            [(n_q, np.int64), (n_r, np.int64), (n_r if mask_tool_use else 0, np.uint8), (n_r, np.float32), (n + 1, np.int64),
             (n + 1, np.int64), (n, np.int64), (n, np.int32), (n if with_adv else 0, np.float32), (2 * n, np.int64)]
        )  # fmt: skip
        q_flat, r_flat, tool, lp_flat, q_off_s, r_off_s, dst_s, mask_base, adv_s, lens = staging.arrays
    else:
        q_flat = np.empty(int(q_off[-1]), dtype=np.int64)
    others = _fill_ints(queries, q_off, q_flat, pad_token_id)
    q_len = q_off[1:] - q_off[:-1]
    assert (others == q_len).all()  # no padding token in a query
    lp_off, m_off = _offsets(vllm_logprobs), _offsets(masks)
    for i in np.flatnonzero((np.diff(lp_off) != np.diff(r_off)) | (np.diff(m_off) != np.diff(r_off))):
        assert len(vllm_logprobs[i]) == len(responses[i]), (
            f"Response {i}: logprobs length ({len(vllm_logprobs[i])}) != response length ({len(responses[i])})"
        )
        raise ValueError(f"Response {i}: mask length ({len(masks[i])}) != response length ({len(responses[i])})")
    if dev.type != "cuda":
        raise RuntimeError("pack_sequences writes its outputs on an AMD GPU; there is no CPU implementation")
    if n:
        r_len = _fill_ints(responses, r_off, r_flat, pad_token_id)
        if mask_tool_use:  # only read when tool tokens are masked out
            _fill_flags(masks, r_off, tool)
        _fill_floats(vllm_logprobs, r_off, lp_flat)
    else:
        r_len = np.zeros(0, dtype=np.int64)
    seq_len = q_len + r_len
    if n and int(seq_len.min()) < 1:
        raise ValueError("every sequence needs at least one token")
    total_tokens = int(seq_len.sum())
    if total_tokens > 0 and min_num_batches > 1:
        effective = min(total_tokens // min_num_batches, pack_length)
    else:
        effective = pack_length
    # greedy row assignment: O(n) scalar work
    row_first = [0] if n else []  # index of the first sequence of each row
    bases = []
    cur = 0
    for i, length in enumerate(seq_len.tolist()):
        if length + cur > effective and cur > 0:
            row_first.append(i)
            cur = 0
        bases.append(row_first[-1])
        cur += length
    dst = np.zeros(n + 1, dtype=np.int64)
    np.cumsum(seq_len, out=dst[1:])

    out_i64 = torch.empty(5, max(total_tokens, 1), dtype=torch.int64, device=dev)
    out_f32 = torch.empty(2, max(total_tokens, 1), dtype=torch.float32, device=dev)
    if with_adv:
        adv_np = np.asarray(advantages, dtype=np.float32).reshape(-1)
        if adv_np.shape[0] != n:
            raise ValueError(f"advantages has {adv_np.shape[0]} entries for {n} sequences")
    lens_dev = torch.zeros(2, 0, dtype=torch.int64, device=dev)
    if n:
        q_off_s[:], r_off_s[:], dst_s[:], mask_base[:] = q_off, r_off, dst[:-1], bases
        lens[:n], lens[n:] = r_len, seq_len
        if with_adv:
            adv_s[:] = adv_np
        ins = staging.upload(dev)
        q_p, r_p, tool_p, lp_p, qo_p, ro_p, dst_p, base_p, adv_p, _ = (ins.data_ptr() + at for at in staging.at)
        _lib.call(
            "oi_pack_sequences", q_p if n_q else None, qo_p, r_p if n_r else None, ro_p, tool_p if mask_tool_use else None,
            lp_p, adv_p if with_adv else None,
            dst_p, base_p, n, int(pad_token_id), int(bool(mask_tool_use)), out_i64[0].data_ptr(), out_i64[1].data_ptr(),
            out_i64[2].data_ptr(), out_i64[3].data_ptr(), out_i64[4].data_ptr(), out_f32[0].data_ptr(),
            out_f32[1].data_ptr() if with_adv else None, torch.cuda.current_stream(dev).cuda_stream,
        )  # fmt: skip
        # a tensor of their own: the caller keeps the lengths, not the inputs
        lens_dev = ins[staging.at[-1] : staging.at[-1] + 16 * n].view(torch.int64).view(2, n).clone()
    bounds = [int(dst[i]) for i in row_first] + [total_tokens]
    seq_bounds = row_first + [n]

    def rows(flat):
        return [flat[bounds[k] : bounds[k + 1]] for k in range(len(row_first))]

    def seq_rows(flat):
        return [flat[seq_bounds[k] : seq_bounds[k + 1]] for k in range(len(row_first))]

    return PackedSequences(
        query_responses=rows(out_i64[0]),
        attention_masks=rows(out_i64[1]),
        position_ids=rows(out_i64[2]),
        response_masks=rows(out_i64[3]),
        original_responses=responses,
        num_actions=seq_rows(lens_dev[0]),
        packed_seq_lens=seq_rows(lens_dev[1]),
        dones=rows(out_i64[4]),
        vllm_logprobs=rows(out_f32[0]),
        advantages=rows(out_f32[1]) if with_adv else None,
    )
