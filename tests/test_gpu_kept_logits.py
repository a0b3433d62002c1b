"""The backward that reads the forward's logits against the one that computes them again: the same products in
the same order, so both gradients must agree to the bit, at the edges of the tiles (rows and columns that are
no multiple of anything, a single row, masks that leave few rows or none)."""

import pytest
import torch

from open_instruct_amd import _lib, lm_head

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
