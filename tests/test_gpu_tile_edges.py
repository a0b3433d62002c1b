"""GPU parity of the tile kernels at the sizes where their work is divided differently: products cut along
the vocabulary, one vocabulary chunk or several, against fp32 autograd on the same bf16 inputs.

Gradients are held to 2 % of their norm and, per entry, to one bf16 rounding (2**-8) of the entry plus 2**-7
of the largest one: an entry is a sum of products with bf16 factors (dZ or the kept exponentials, 2**-9
each), rounded once to bf16.
"""

import types

import pytest
import torch

from open_instruct_amd import _lib, grpo_utils, lm_head

pytestmark = pytest.mark.gpu
DEV = "cuda:0"
TOL = 2e-3


def _inputs(n, h, v, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    hidden = torch.randn(n, h, generator=g, device=DEV).bfloat16()
    weight = (torch.randn(v, h, generator=g, device=DEV) * (2.0 / h**0.5)).bfloat16()
    labels = torch.randint(0, v, (n,), generator=g, device=DEV)
    mask = torch.rand(n, generator=g, device=DEV) < 0.8
    upstream = torch.randn(n, generator=g, device=DEV)
    return hidden, weight, labels, mask, upstream


def _reference(hidden, weight, labels, mask, upstream):
    """logprobs and both gradients in fp32, 2048 rows at a time."""
    h32, w32 = hidden.float(), weight.float()
    lp = torch.zeros(hidden.shape[0], device=DEV)
    dh, dw = torch.zeros_like(h32), torch.zeros_like(w32)
    for a in range(0, hidden.shape[0], 2048):
        rows = slice(a, a + 2048)
        z = h32[rows] @ w32.t()
        logp = z.log_softmax(1)
        lp[rows] = logp.gather(1, labels[rows, None])[:, 0] * mask[rows]
        dz = logp.exp_().neg_()
        dz[torch.arange(dz.shape[0], device=DEV), labels[rows]] += 1.0
        dz *= (upstream * mask)[rows, None]
        dh[rows] = dz @ w32
        dw += dz.t() @ h32[rows]
    return lp, dh, dw


def _close(got, exp, name):
    err = (got.float() - exp).abs()
    bound = TOL * exp.abs().max() + exp.abs() * 2**-8 + exp.abs().max() * 2**-7
    assert (err <= bound).all(), (name, err.max().item(), exp.abs().max().item())
    rel = ((got.float() - exp).norm() / exp.norm()).item()
    assert rel <= 2e-2, (name, rel)


@pytest.mark.parametrize(
    "n,h,v",
    [
        (70, 64, 1984),  # 31 k-tiles: too short to cut
        (70, 64, 2048),  # 32 k-tiles: the shortest product that is cut, in two
        (1, 64, 2049),  # one row, 33 k-tiles, the last of one vocabulary row
        (300, 320, 9001),  # two tiles (about 240 rows are selected) in eight pieces
        (600, 1088, 33000),  # ten tiles in 25 pieces, ragged last hidden tile
        (2100, 4096, 128256),  # 112 tiles in nine pieces: 1008, the most scratch there is
        (16500, 1088, 2300),  # a whole round of tiles and a cut rest
        (9000, 64, 120000),  # two vocabulary chunks
    ],
)
@pytest.mark.parametrize("route", ["d_weight", "d_hidden_in_forward", "slabs"])
def test_products_cut_along_the_vocabulary(n, h, v, route):
    print(f"case N={n} H={h} V={v} route={route}", flush=True)
    hidden, weight, labels, mask, upstream = _inputs(n, h, v, seed=n + v)
    mask[0] = True
    if route == "slabs":
        # the policy loss whose gradient to a logprob is -advantage / count: ratio 1, no KL term
        upstream = -upstream / mask.sum()
        adv = -upstream * mask.sum()
    lp, dh, dw = _reference(hidden, weight, labels, mask, upstream)
    hid, w = hidden.requires_grad_(True), weight.requires_grad_(route != "d_hidden_in_forward")
    if route == "slabs":
        cfg = types.SimpleNamespace(loss_fn="cispo", clip_lower=0.2, clip_higher=0.2, beta=0.0, kl_estimator=2)
        loss, _, out, _ = grpo_utils.grpo_loss_on_hidden(
            hid[None], w, labels[None], None, None, adv[None], mask[None], cfg, token_slabs=4096
        )
        loss.backward()
        out = out[0]
    else:
        out, _ = lm_head.fused_lm_head_logprobs(hid, w, labels, mask=mask)
        out.backward(upstream)
    assert (out.detach() - lp).abs().max().item() <= TOL
    _close(hid.grad, dh, "d_hidden")
    assert (hid.grad[~mask] == 0).all()
    if w.requires_grad:
        _close(w.grad, dw, "d_weight")


@pytest.mark.parametrize("n,h,v", [(70, 64, 301), (300, 320, 513), (16500, 64, 66000)])  # the last: three chunks
def test_gradients_off_16_byte_boundaries(n, h, v):
    """Gradients that lie on 4-byte boundaries only are stored by another route of the same epilogue."""
    print("case unaligned gradients", n, h, v, flush=True)
    g = torch.Generator().manual_seed(n)
    hidden = torch.randn(n, h, generator=g).bfloat16().to(DEV)
    weight = (torch.randn(v, h, generator=g) * 0.2).bfloat16().to(DEV)
    labels = torch.randint(0, v, (n,), generator=g).to(DEV)
    up = torch.rand(n, generator=g).to(DEV)
    lib = _lib.load()
    stream = torch.cuda.current_stream().cuda_stream
    lp, lse = torch.empty(n, device=DEV), torch.empty(n, device=DEV)
    ws_bytes = max(lib.oi_lmhead_fwd_workspace_bytes(n, h, v, 0), lib.oi_lmhead_bwd_workspace_bytes(n, h, v, 1, 0))
    ws = torch.empty(ws_bytes, dtype=torch.uint8, device=DEV)
    p = lambda t: t.data_ptr()  # noqa: E731
    assert lib.oi_lmhead_logp_fwd(p(hidden), p(weight), p(labels), None, n, h, v, 1.0, p(lp), None, p(lse), p(ws), ws_bytes, stream) == 0
    got = []
    for shift in (0, 2):
        dh = torch.full((n * h + 16,), 7.0, dtype=torch.bfloat16, device=DEV)
        dw = torch.full((v * h + 16,), 7.0, dtype=torch.bfloat16, device=DEV)
        rc = lib.oi_lmhead_logp_bwd(
            p(hidden), p(weight), p(labels), p(lse), p(up), None, 0, n, h, v, 1.0, p(lp), p(dh[shift:]), p(dw[shift:]),
            p(ws), ws_bytes, stream,
        )  # fmt: skip
        assert rc == 0
        for t, size in ((dh, n * h), (dw, v * h)):  # nothing written around them
            assert (t[:shift] == 7).all() and (t[shift + size :] == 7).all()
        got.append((dh[shift : shift + n * h], dw[shift : shift + v * h]))
    for a, b in zip(*got):
        assert a.float().abs().max() > 0 and torch.equal(a, b)


@pytest.mark.parametrize(
    "m,n,k,ldo,shift",
    [
        (257, 264, 64, 272, 0),  # whole 16-byte pieces
        (300, 260, 128, 260, 0),  # four columns at a time
        (64, 300, 192, 308, 4),  # the same, results off 16-byte boundaries
        (130, 258, 64, 262, 2),  # pairs of bf16
        (66, 517, 64, 518, 0),  # pairs and a last single column
        (5, 1001, 128, 1001, 0),  # one column at a time
        (513, 3, 64, 7, 0),
    ],
)
def test_products_of_any_pitch(m, n, k, ldo, shift):
    """Small whole numbers: every sum is exact in fp32 and is rounded once to bf16, so nothing may differ, and
    nothing may be written around the result."""
    print("case product", m, n, k, ldo, shift, flush=True)
    lib = _lib.load()
    stream = torch.cuda.current_stream().cuda_stream
    g = torch.Generator().manual_seed(m + n)
    a = torch.randint(-4, 5, (m, k), generator=g).bfloat16().to(DEV)
    b = torch.randint(-4, 5, (n, k), generator=g).bfloat16().to(DEV)
    exact = a.float() @ b.float().t()
    for dtype, accumulate in ((torch.float32, 0), (torch.float32, 1), (torch.bfloat16, 0)):
        out = torch.full((m * ldo + shift + 8,), 3.0, dtype=dtype, device=DEV)
        rows = out[shift : shift + m * ldo].view(m, ldo)
        o = rows.data_ptr()
        rc = lib.oi_gemm_bf16_tn(
            a.data_ptr(), k, m, b.data_ptr(), k, n, k, o if dtype == torch.float32 else None,
            o if dtype == torch.bfloat16 else None, ldo, accumulate, stream,
        )  # fmt: skip
        assert rc == 0
        assert torch.equal(rows[:, :n], (exact + 3.0 * accumulate).to(dtype)), (dtype, accumulate)
        assert (rows[:, n:] == 3).all() and (out[:shift] == 3).all() and (out[shift + m * ldo :] == 3).all()


# pitches past 24 and past 32 bits; one column tile and two
@pytest.mark.parametrize("m,n,ldo", [(3, 8, 1 << 24), (3, 264, (1 << 24) + 8), (2, 8, (1 << 32) + 8)])
def test_products_added_to_rows_far_apart(m, n, ldo):
    """Small whole numbers, exact in fp32."""
    k = 64
    print("case far rows", m, n, ldo, flush=True)
    g = torch.Generator().manual_seed(n)
    a = torch.randint(-4, 5, (m, k), generator=g).bfloat16().to(DEV)
    b = torch.randint(-4, 5, (n, k), generator=g).bfloat16().to(DEV)
    before = torch.randint(-9, 10, (m, n), generator=g).float().to(DEV)
    out = torch.empty((m - 1) * ldo + n, device=DEV)
    rows = out.as_strided((m, n), (ldo, 1))
    rows.copy_(before)
    rc = _lib.load().oi_gemm_bf16_tn(
        a.data_ptr(), k, m, b.data_ptr(), k, n, k, out.data_ptr(), None, ldo, 1, torch.cuda.current_stream().cuda_stream
    )
    assert rc == 0 and torch.equal(rows, before + a.float() @ b.float().t())


# operands of one row each (pitch 0), to and past the longest range that other operands have
@pytest.mark.parametrize("k", [1 << 22, (1 << 22) + 64])
@pytest.mark.parametrize("m,n", [(1, 1), (3, 264)])
def test_products_of_one_long_row(m, n, k):
    """Entries in -1 .. 1: every sum is a whole number below 2**24, so any order of the additions gives it."""
    print("case one row", m, n, k, flush=True)
    g = torch.Generator(device=DEV).manual_seed(n)
    a, b = (torch.randint(-1, 2, (k,), generator=g, device=DEV).bfloat16() for _ in range(2))
    exact = (a.float() * b.float()).double().sum().float()
    for dtype, accumulate in ((torch.float32, 0), (torch.float32, 1), (torch.bfloat16, 0)):
        out = torch.full((m, n), 3.0, dtype=dtype, device=DEV)
        o = out.data_ptr()
        rc = _lib.load().oi_gemm_bf16_tn(
            a.data_ptr(), 0, m, b.data_ptr(), 0, n, k, o if dtype == torch.float32 else None,
            o if dtype == torch.bfloat16 else None, n, accumulate, torch.cuda.current_stream().cuda_stream,
        )  # fmt: skip
        assert rc == 0 and (out == (exact + 3.0 * accumulate).to(dtype)).all(), (dtype, accumulate)


@pytest.mark.parametrize("n,h,v,flagged,slabs", [(1, 64, 300, 1, 4096), (300, 64, 301, 70, 4096), (600, 320, 513, 257, 256)])
def test_flagged_rows_are_added_to_d_weight(n, h, v, flagged, slabs):
    """Rows whose label lies more than 44 nats below the largest logit are recomputed and added to the bf16 d_weight
    of the others (which rounds its entries once more: within the bound of _close, half of which is one rounding)."""
    print("case flagged", n, h, v, flagged, slabs, flush=True)
    hidden, weight, labels, mask, upstream = _inputs(n, h, v, seed=n + v)
    labels = labels % (v - 1) + 1
    weight[0] = 0.5
    hidden[:flagged] = 1.5
    weight[labels[:flagged]] = -0.5
    mask[:flagged] = True
    upstream = -upstream / mask.sum()
    lp, dh, dw = _reference(hidden, weight, labels, mask, upstream)
    cfg = types.SimpleNamespace(loss_fn="cispo", clip_lower=0.2, clip_higher=0.2, beta=0.0, kl_estimator=2)
    hid, w = hidden.requires_grad_(True), weight.requires_grad_(True)
    adv = -upstream * mask.sum()
    loss, _, out, _ = grpo_utils.grpo_loss_on_hidden(
        hid[None], w, labels[None], None, None, adv[None], mask[None], cfg, token_slabs=slabs
    )
    loss.backward()
    assert lp[:flagged].max() < -44 and (out[0].detach() - lp).abs().max() <= 1e-5 * lp.abs().max() + TOL
    _close(hid.grad, dh, "d_hidden")
    _close(w.grad, dw, "d_weight")


@pytest.mark.parametrize("k_tiles", [1, 2, 3, 4, 5, 6, 11])  # around the ring of five slots, once and twice
@pytest.mark.parametrize("a_km,b_km", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_products_of_whole_numbers_are_exact(k_tiles, a_km, b_km):
    """Entries in -4 .. 4: every sum is a whole number below 2**24, so any order of the additions gives it."""
    for m, n in ((8, 8), (256, 264), (296, 520)):  # one fragment; one tile; ragged in both directions
        k = 64 * k_tiles
        print(f"case M={m} N={n} K={k} k-major {a_km} {b_km}", flush=True)
        g = torch.Generator(device=DEV).manual_seed(m + k)
        a = torch.randint(-4, 5, (m, k), generator=g, device=DEV).bfloat16()
        b = torch.randint(-4, 5, (n, k), generator=g, device=DEV).bfloat16()
        exp = (a.double() @ b.double().t()).float()
        at = a.t().contiguous() if a_km else a
        bt = b.t().contiguous() if b_km else b
        out = torch.full((m, n), -1.0, device=DEV)
        rc = _lib.load().oi_gemm_bf16_layouts(
            at.data_ptr(), m if a_km else k, a_km, bt.data_ptr(), n if b_km else k, b_km, m, n, k, out.data_ptr(), None,
            n, 0, torch.cuda.current_stream().cuda_stream,
        )  # fmt: skip
        assert rc == 0
        assert torch.equal(out, exp)


# last rows of each group of 64 token rows and the first of the next: the widths of the forward's last tile
@pytest.mark.parametrize("n", [64, 65, 128, 129, 192, 193, 256, 320, 321])
@pytest.mark.parametrize("keep_logits", [True, False])
def test_last_tile_of_token_rows(n, keep_logits):
    h, v = 192, 700  # three k-tiles; ragged vocabulary tile and d_hidden columns
    print(f"case N={n} keep_logits={keep_logits}", flush=True)
    hidden, weight, labels, _, upstream = _inputs(n, h, v, seed=n)
    lp, dh, dw = _reference(hidden, weight, labels, torch.ones_like(labels, dtype=torch.bool), upstream)
    for frozen in (False, True):  # logits or statistics alone; kept exponentials and their weighted sum
        hid, w = hidden.clone().requires_grad_(True), weight.clone().requires_grad_(not frozen)
        out = lm_head.fused_lm_head_logprobs(hid, w, labels, keep_logits=keep_logits)
        out = out[0] if isinstance(out, tuple) else out
        assert (out.detach() - lp).abs().max().item() <= TOL
        out.backward(upstream)
        _close(hid.grad, dh, "d_hidden")
        if not frozen:
            _close(w.grad, dw, "d_weight")


@pytest.mark.parametrize("n,h", [(1, 64), (256, 192), (100, 576), (257, 576)])  # k-tiles fewer than eighths, and not a multiple
def test_products_that_begin_at_another_k_tile(n, h):
    v = 8 * 32 * 256 + 300  # vocabulary tiles of every eighth and of the first once more
    print(f"case N={n} H={h}", flush=True)
    hidden, weight, labels, _, upstream = _inputs(n, h, v, seed=n + h)
    lp, dh, dw = _reference(hidden, weight, labels, torch.ones_like(labels, dtype=torch.bool), upstream)
    grads = []
    for keep_logits in (True, False):  # read back; computed again, by the same rule
        hid, w = hidden.clone().requires_grad_(True), weight.clone().requires_grad_(True)
        out = lm_head.fused_lm_head_logprobs(hid, w, labels, keep_logits=keep_logits)
        out = out[0] if isinstance(out, tuple) else out
        assert (out.detach() - lp).abs().max().item() <= TOL
        out.backward(upstream)
        _close(hid.grad, dh, "d_hidden")
        _close(w.grad, dw, "d_weight")
        grads.append(hid.grad)
    assert torch.equal(*grads)


# token counts in each width of the last tile; a narrow tile leaves the rows behind it as they were
@pytest.mark.parametrize("n", [1, 64, 65, 100, 130, 193, 300])
@pytest.mark.parametrize("masked", [False, True])
def test_old_contents_of_scratch_memory_do_not_matter(n, masked, monkeypatch):
    """Scratch memory full of NaN bits gives the results that other contents give, to the bit."""
    h, v = 192, 700
    hidden, weight, labels, mask, upstream = _inputs(n, h, v, seed=n)
    mask[0] = True  # an empty selection has no mean
    sel = mask if masked else None
    empty, empty_like = torch.empty, torch.empty_like

    def filled(t):
        t.untyped_storage().fill_(255)
        return t

    def results():
        out = []
        for keep_logits, frozen in ((True, False), (False, False), (False, True)):
            hid, w = hidden.clone().requires_grad_(True), weight.clone().requires_grad_(not frozen)
            lp = lm_head.fused_lm_head_logprobs(hid, w, labels, mask=sel, keep_logits=keep_logits)
            lp = lp[0] if isinstance(lp, tuple) else lp
            lp.backward(upstream)
            out += [lp.detach(), hid.grad] + ([] if frozen else [w.grad])
        hid, w = hidden.clone().requires_grad_(True), weight.clone().requires_grad_(True)
        y = labels.masked_fill(~mask, -100) if masked else labels
        loss = lm_head.fused_linear_cross_entropy(hid[None], w, shift_labels=y[None], token_slabs=True)
        loss.backward()
        return out + [loss.detach(), hid.grad, w.grad]

    print(f"case N={n} masked={masked}", flush=True)
    exp = results()
    monkeypatch.setattr(torch, "empty", lambda *a, **k: filled(empty(*a, **k)))
    monkeypatch.setattr(torch, "empty_like", lambda *a, **k: filled(empty_like(*a, **k)))
    got = results()
    monkeypatch.undo()
    for i, (a, b) in enumerate(zip(got, exp)):
        assert torch.equal(a, b), i
