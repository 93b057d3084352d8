"""The blocks' slot lists (mb_flash_ema_slot_lists) against the definition computed on the CPU,
and the attention over them (mb_flash_ema_fwd_lists / mb_flash_ema_bwd_lists) against the same
call over every slot: what the lists leave out is exactly zero, so outputs and gradients agree
to the rounding of reordered fp32 sums (the skipped slots' e^0 terms are added at once, and the
atomics' order is free): 1e-5 norm-wise.  dW_pe has a bound of its own: its product takes dpre
in bf16, and a last-bit difference of dpre can round it to the other neighbour, 2^-8 of that
term and so at most 2^-8 of the sum; in fp32 mode, with its second bf16 part, 2^-16.  The
default mode's gradients from stored scores are compared with the oracle instead, which takes the
same rounding: there a probability that rounds to either side of 2^-7 changes a whole slot's gate
arithmetic."""
import pytest
import torch

from tests.test_gpu_flash import (TOL_KERNEL_ROUNDING, case_rounding, make_case, norm_err, oracle_backward,
                                  oracle_forward)
from tests.test_gpu_fp32_mode import TOL_FP32

pytestmark = pytest.mark.gpu

TOL = 1e-5
TOL_DW = {"fp32": 2.0 ** -16, "bf16": 2.0 ** -8, "fp16": 2.0 ** -8}


def lists_of(c, dev):
    from mathbrain import _lib
    x, u, Cb = c["x"].to(dev), c["unique"].to(dev), c["Cb"].to(dev).float().contiguous()
    B, L = x.shape
    K, N = c["K"], c["rhos"].shape[0]
    buf = torch.full((_lib.lib().mb_flash_ema_slot_lists_bytes(B, L, K),), 255, dtype=torch.uint8, device=dev)
    _lib.call("mb_flash_ema_slot_lists", _lib.ptr(x), x.stride(0), x.stride(1), _lib.ptr(u), _lib.ptr(Cb), B, L, K,
              N, Cb.shape[3], Cb.shape[1], c["Br"], _lib.ptr(buf), _lib.stream(dev))
    return buf


def expected(c):
    """{(b, block): [k, ...]} of the active slots."""
    x, u, Cb, Br, N = c["x"], c["unique"], c["Cb"].cpu(), c["Br"], c["rhos"].shape[0]
    B, L = x.shape
    out = {}
    for b in range(B):
        for blk in range(-(-L // 32)):
            j = blk * 32 // Br
            seen = x[b, j * Br:min(blk * 32 + 31, L)]
            state = (Cb[b, j, :, :N] != 0).any(1)
            out[b, blk] = [k for k in range(c["K"]) if u[b, k] >= 0 and (state[k] or bool((seen == u[b, k]).any()))]
    return out


def call(c, dev, lists, absent_mass, use_silu, prec, table=False, workspace=False):
    """O, LSE, and the four gradients from the scores and without them, by the C entry points.
    ``table``: c's E_k / E_v are vocabulary tables.  ``workspace``: the backward gets its workspace,
    behind which nothing may be written."""
    from mathbrain import _lib
    from mathbrain.triton_flash_ema import _flash_flags, _prec
    B, H, L, hd = c["Q"].shape
    K, N, D = c["K"], c["rhos"].shape[0], H * hd
    size = _lib.lib().mb_flash_ema_bwd_lists_workspace(B, H, L, hd, K, N, _prec(prec)) if workspace else 0
    ws = torch.full((size + (1 << 22),), 0x5A, dtype=torch.uint8, device=dev)
    cu = lambda t: t.to(dev).float().contiguous()  # noqa: E731
    Q, Ek, Ev, W, rh, Cb = (cu(c[k]) for k in ("Q", "E_k", "E_v", "W", "rhos", "Cb"))
    x, u = c["x"].to(dev), c["unique"].to(dev)
    dO = torch.randn(B, H, L, hd, generator=torch.Generator().manual_seed(3)).to(dev)
    flags = _flash_flags(use_silu, absent_mass, table, _prec(prec))
    O, LSE, S2 = (torch.full(s, float("nan"), device=dev) for s in ((B, H, L, hd), (B, H, L), (B, H, K, L)))
    g = [torch.full(s, float("nan"), device=dev) for s in (Q.shape, Ek.shape, Ev.shape, (N, D))]
    p, st = _lib.ptr, _lib.stream(dev)
    common = (B, H, L, hd, K, N, Cb.shape[3], Cb.shape[1], c["Br"], c["V"], flags)
    _lib.call("mb_flash_ema_fwd_lists", p(Q), *Q.stride(), p(x), x.stride(0), x.stride(1), p(Ek), p(Ev), p(W), p(rh),
              p(u), p(Cb), *common, p(O), p(LSE), p(S2), None, 0, p(lists), st)
    outs = []
    for scores in (S2, None):
        _lib.call("mb_flash_ema_bwd_lists", p(Q), *Q.stride(), p(dO), p(x), x.stride(0), x.stride(1), p(Ek), p(Ev),
                  p(W), p(rh), p(u), p(Cb), p(O), p(LSE), *common, p(scores), *(p(t) for t in g), p(lists),
                  p(ws) if size else None, size, st)
        outs += [t.cpu() for t in g]
    assert bool((ws[size:] == 0x5A).all())
    return [O.cpu(), LSE.cpu()] + outs


@pytest.mark.parametrize("L, N, Br, warmup, pad_slots", [
    (64, 16, 64, 0, 0),        # no history: the first block sees only its own tokens
    (97, 33, 64, 40, 5),       # rows that are not float4s, a last block of one step
    (130, 64, 32, 30, 0),      # a chunk per block
    (70, 128, 24, 0, 0),       # chunks that do not end where blocks do; single fp16 products
    (1, 8, 64, 20, 0),         # one step
    (256, 16, 64, 900, 0),     # more than one round of 512 slots
])
@pytest.mark.parametrize("absent_mass", [True, False])
def test_lists_and_the_attention_over_them(L, N, Br, warmup, pad_slots, absent_mass):
    dev = torch.device("cuda", 0)
    c = make_case(2, L, 700, 4, 32, N, warmup=warmup, seed=L + N, qs=0.5, es=0.3, ws=0.2, Br=Br, pad_slots=pad_slots)
    B, K = c["unique"].shape
    buf = lists_of(c, dev)
    nblk = -(-L // 32)
    entries = buf[:B * nblk * K * 16].view(torch.int32).view(B, nblk, K, 4).cpu()
    counts = buf[B * nblk * K * 16:-B * nblk * 4].view(torch.int32).view(B, nblk, 2).cpu()
    order = buf[-B * nblk * 4:].view(torch.int32).cpu()
    for (b, blk), ks in expected(c).items():
        assert counts[b, blk].tolist() == [len(ks), int((c["unique"][b] >= 0).sum())]
        assert entries[b, blk, :len(ks), 3].tolist() == ks
        assert entries[b, blk, :len(ks), 2].tolist() == c["unique"][b, ks].tolist()
    # every block once, the longest lists first (to within a 1023rd of K)
    assert sorted(order.tolist()) == list(range(B * nblk))
    ordered = counts.view(-1, 2)[order.long(), 0]
    assert bool((ordered[1:] - ordered[:-1] <= K / 1023 + 1).all())
    for use_silu, prec in ((True, "bf16"), (False, "fp32" if N <= 64 else "fp16")):
        got = call(c, dev, buf, absent_mass, use_silu, prec)
        want = call(c, dev, None, absent_mass, use_silu, prec)
        for i, (a, w) in enumerate(zip(got, want)):
            assert torch.isfinite(a).all()
            if prec == "bf16" and 2 <= i <= 5:
                continue
            assert norm_err(a, w) < (TOL_DW[prec] if i in (5, 9) else TOL)


@pytest.mark.parametrize("B, L, H, hd, N", [
    (2, 97, 4, 32, 33),      # two slots per batch in fp32 mode
    (1, 130, 3, 64, 64),     # heads that a group of four does not fill
    (2, 64, 2, 128, 40),     # two 64-dim halves per head
    (3, 65, 2, 64, 128),     # the half-waves share the rate tiles
    (2, 40, 4, 32, 16),      # four slots per batch, more parts than some lists have batches
])
@pytest.mark.parametrize("table", [False, True])
def test_rows_and_workspace_over_lists(B, L, H, hd, N, table):
    """Gathered and vocabulary rows, with and without the dW_pe workspace: all over lists against
    every slot without it."""
    dev = torch.device("cuda", 0)
    c = make_case(B, L, 500, H, hd, N, warmup=25, seed=hd + N, qs=0.5, es=0.3, ws=0.2, pad_slots=3)
    if table:
        g = torch.Generator().manual_seed(5)
        c["E_k"], c["E_v"] = (torch.randn(c["V"], H * hd, generator=g) * 0.3 for _ in range(2))
    buf = lists_of(c, dev)
    assert sum(len(ks) for ks in expected(c).values()) < int((c["unique"] >= 0).sum()) * -(-L // 32)
    for prec in ("fp32" if N <= 64 and hd <= 64 else "fp16", "bf16"):
        want = call(c, dev, None, True, True, prec, table)
        for workspace in (False, True):
            got = call(c, dev, buf, True, True, prec, table, workspace)
            for i, (a, w) in enumerate(zip(got, want)):
                assert torch.isfinite(a).all()
                if prec == "bf16" and 2 <= i <= 5:
                    continue
                assert norm_err(a, w) < (TOL_DW[prec] if i in (5, 9) else TOL), (i, prec, workspace)


@pytest.mark.parametrize("L", [33, 160])
@pytest.mark.parametrize("H, hd, N, precision, table", [
    (4, 32, 16, "bf16", False), (8, 64, 64, "bf16", False), (3, 64, 33, "bf16", True), (2, 128, 64, "bf16", False),
    (2, 128, 128, "bf16", True), (4, 64, 80, "bf16", False), (6, 32, 33, "fp32", True), (8, 64, 64, "fp32", False),
    (8, 64, 64, "fp16", True)])
def test_kept_scores_over_lists_against_the_oracle(monkeypatch, L, H, hd, N, precision, table):
    """FlashEMAFunction as a training step calls it: the forward writes its scores over lists, the
    backward reads them.  Memory that the score tensor may land in holds NaN first, so a read of an
    entry that no list names shows."""
    from mathbrain import triton_flash_ema as tfe
    monkeypatch.setattr(tfe, "MIN_LISTED_SLOTS", 0)
    monkeypatch.setattr(tfe, "score_budget", tfe.ScoreBudget())
    c = make_case(2, L, 400, H, hd, N, warmup=30, seed=L + N, qs=0.5, es=0.3, ws=0.2, pad_slots=5)
    dO = torch.randn(c["Q"].shape, generator=torch.Generator().manual_seed(3))
    leaves = dict(c)
    if table:
        g = torch.Generator().manual_seed(5)
        leaves["E_k"], leaves["E_v"] = (torch.randn(c["V"], H * hd, generator=g) * 0.3 for _ in range(2))
        c["E_k"], c["E_v"] = (leaves[k][c["unique"].clamp(min=0)] for k in ("E_k", "E_v"))
    junk = torch.full((2 * H * c["K"] * L,), float("nan"), device="cuda")
    del junk
    got = autograd_grads(leaves, dO, precision)
    # the fp32 mode against the exact oracle at its own bound (the oracle's roundings include the
    # other modes' single bf16 operands of dW_pe, 2^-8)
    rounding, tol = (None, TOL_FP32) if precision == "fp32" else (case_rounding(c, precision), TOL_KERNEL_ROUNDING)
    want = [oracle_forward(c, gate_round=rounding)[0], *oracle_backward(c, dO, gate_round=rounding)]
    if table:  # a table row's gradient is the sum over the token's slots
        valid = (c["unique"] >= 0).reshape(-1)
        for i in (2, 3):
            rows = torch.zeros(c["V"], H * hd, dtype=torch.float64)
            want[i] = rows.index_add_(0, c["unique"].reshape(-1)[valid], want[i].double().reshape(-1, H * hd)[valid])
    for a, w in zip(got, want):
        assert torch.isfinite(a).all()
        assert norm_err(a, w) < tol


def autograd_grads(c, dO, precision="bf16"):
    """O and the gradients of FlashEMAFunction."""
    from mathbrain.triton_flash_ema import FlashEMAFunction
    leaves = [t.cuda().requires_grad_(True) for t in (c["Q"], c["E_k"], c["E_v"], c["W"])]
    O = FlashEMAFunction.apply(leaves[0], c["x"].cuda(), leaves[1], leaves[2], leaves[3], c["rhos"].cuda(), c["V"],
                               c["unique"].cuda(), c["K"], c["Cb"].cuda(), True, c["Br"], True, precision)
    return [t.cpu() for t in (O.detach(), *torch.autograd.grad(O, leaves, dO.cuda()))]


def test_lists_beyond_the_score_budget_are_made_again(monkeypatch):
    """With room for the scores and not for the lists, the backward lists the slots again, also where
    the rule for small calls would now say otherwise: the gradients stay finite (the scores of pairs
    outside the lists are never written) and are those with the lists kept."""
    from mathbrain import triton_flash_ema as tfe
    monkeypatch.setattr(tfe, "score_budget", tfe.ScoreBudget())
    monkeypatch.setattr(tfe, "MIN_LISTED_SLOTS", 0)
    c = make_case(2, 97, 700, 4, 32, 16, seed=4, qs=0.5, es=0.3, ws=0.2)
    dO = torch.randn(c["Q"].shape, generator=torch.Generator().manual_seed(3))
    want = autograd_grads(c, dO, "fp32")
    monkeypatch.setattr(tfe, "SAVE_SCORES_MAX_BYTES", 4 * 2 * 4 * c["K"] * 97)
    made = []
    real = tfe._slot_lists
    monkeypatch.setattr(tfe, "_slot_lists", lambda *a, **k: made.append(real(*a, **k)) or made[-1])
    junk = torch.full((4 * 2 * 4 * c["K"] * 97,), 255, dtype=torch.uint8, device="cuda")  # NaN where the scores go
    del junk
    got = autograd_grads(c, dO, "fp32")
    assert len(made) == 2 and all(m is not None for m in made)
    for i, (a, w) in enumerate(zip(got, want)):
        assert torch.isfinite(a).all() and norm_err(a, w) < (TOL_DW["fp32"] if i == 4 else TOL)
