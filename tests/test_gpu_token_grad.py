"""GPU parity of the loss forward that keeps the tokens' gradients (``siirl_actor_loss_fwd_grad``,
``siirl_token_grad_bwd``) against the backward that reads the operands again: every loss, aggregation and KL estimator (each
with its own and the straight-through gradient), with and without the other terms, at the edges of quads and of segments of
2048 tokens, rows and batches without a valid token, and through autograd.

Tolerance: both multiply the same per-token factors, in another order (g * c * (m * d) against g * ((m * c) * d)), so a
gradient differs by a few roundings (2^-24 each) of its largest term: 1e-6 of the row's largest gradient bounds it.
The result block of the two forwards: a segment's float32 sums are the same words in both; segments and rows add up in double,
rounded once to float32, so one unit in the last place."""

import ctypes
import itertools

import pytest
import torch

import siirl_amd.core_algos as CA
from siirl_amd import _lib

pytestmark = pytest.mark.gpu

MODES = ["vanilla", "gspo", "cpgd", "gpg", "geo_mean", "kl_cov", "clip_cov"]
# entropy, reference, drift, KL estimator, straight-through
TERMS = {"plain": (False, False, 0.0, 3, False), "all": (True, True, 0.05, 3, False), "k1": (False, True, 0.0, 0, False),
         "abs": (False, True, 0.0, 1, False), "k2": (False, True, 0.0, 2, False), "k1+": (False, True, 0.0, 0, True),
         "abs+": (False, True, 0.0, 1, True), "k2+": (False, True, 0.0, 2, True), "k3+": (True, True, 0.05, 3, True)}
SHAPES = [(1, 1), (3, 5), (2, 2044), (5, 2048), (2, 2049), (3, 4100), (8, 2048), (1, 16381), (9, 700), (130, 513), (1025, 6)]
NONE = ctypes.c_void_p(0)


def _mask(B, L, i, g, dev):
    mask = torch.rand(B, L, generator=g) < 0.7
    mask[:, 0] = True
    return mask.to([torch.bool, torch.int64, torch.float32, torch.bfloat16][i % 4]).to(dev)


def _buffers(B, L, dev, mask):
    f = lambda *s: torch.full(s, float("nan"), device=dev)  # noqa: E731  every word must be written
    nws = _lib.lib().siirl_loss_workspace_bytes(B, L)
    m = (_lib.ptr(mask), _lib.dtype_code(mask.dtype))
    return f(16), f(B), f(B), f(B, L), torch.empty(nws, dtype=torch.uint8, device=dev), nws, m


def _aux(mode, B, L, g, dev):
    """The covariance losses' token_aux: a few tokens' KL coefficients, or the tokens that are dropped."""
    if mode not in ("kl_cov", "clip_cov"):
        return None
    return ((torch.rand(B, L, generator=g) < 0.3) * (0.5 + torch.rand(B, L, generator=g))).to(dev)


def _compare(dev, mode, agg, terms, old, lp, adv, mask, isw, e, r, aux, bound):
    """Both routes on the same operands: (kept d log_prob, the other one's) after the checks of everything else."""
    ent, ref, drift, kl_mode, kl_st = TERMS[terms]
    B, L = lp.shape
    P, h, st = _lib.ptr, _lib.lib(), _lib.current_stream(dev)
    args = (CA._LOSS_CODES[mode], 0.2, 0.28, 3.0, 20.0, agg, 0.01 if ent else 0.0, kl_mode, kl_st, 0.1 if ref else 0.0, drift, 0.7)
    out16, msum, rs, tg, ws, nws, m = _buffers(B, L, dev, mask)
    rc = h.siirl_actor_loss_fwd_grad(P(old), P(lp), P(adv), *m, P(isw), P(e), P(r), P(aux) if aux is not None else NONE, B, L,
                                     *args, P(out16), P(msum), P(rs), P(tg), P(ws), nws, st)
    if mode == "geo_mean" or (mode == "gspo" and (ref or drift) and agg != 2):
        assert rc == -2 and b"row factor" in h.siirl_hip_last_error()
        return None
    assert rc == 0
    o_out16, o_msum, o_rs = torch.ops.siirl_hip.policy_loss_fwd(old, lp, adv, mask, isw, e, r, *args, aux)
    close = (out16 - o_out16).abs() <= 1.2e-7 * o_out16.abs()
    assert (close | (out16.isnan() & o_out16.isnan())).all() and torch.equal(msum, o_msum), (B, L)
    up = torch.tensor([1.7], device=dev)
    want, want_e = torch.ops.siirl_hip.policy_loss_bwd(up, old, lp, adv, mask, isw, e, r, *args, o_out16, o_msum, o_rs, aux)
    got, got_e = torch.full_like(lp, -77.0), torch.full_like(lp, -77.0)  # (a NaN may be right)
    kept = tg.clone()
    rc = h.siirl_token_grad_bwd(P(up), P(tg), *(m if ent else (NONE, 0)), B, L, 2 if mode == "gspo" else agg, agg, args[6],
                                args[-1], P(out16), P(msum), P(got), P(got_e) if ent else NONE, st)
    assert rc == 0 and torch.equal(tg, kept)
    same = (got - want).abs() <= bound * want.nan_to_num(0.0).abs().amax(1, keepdim=True)
    assert (same | (got.isnan() & want.isnan())).all(), (B, L)
    if ent:
        assert torch.equal(got_e, want_e) or torch.equal(got_e.nan_to_num(3.0), want_e.nan_to_num(3.0))
    return got, want


def _operands(mode, terms, B, L, i, g, dev):
    ent, ref = TERMS[terms][:2]
    f = lambda: torch.randn(B, L, generator=g).to(dev)  # noqa: E731
    lp, old = 0.3 * f() - 1.0, 0.3 * f() - 1.0
    adv, isw = f(), torch.rand(B, L, generator=g).to(dev) + 0.5
    e, r = (f().abs() if ent else None), (lp + 0.1 * f() if ref else None)
    return old, lp, adv, _mask(B, L, i, g, dev), isw, e, r, _aux(mode, B, L, g, dev)


@pytest.mark.parametrize("mode,agg,terms", list(itertools.product(MODES, range(4), TERMS)))
def test_kept_token_gradients(dev, mode, agg, terms):
    for i, (B, L) in enumerate(SHAPES):
        g = torch.Generator().manual_seed(1000 * agg + i)
        pair = _compare(dev, mode, agg, terms, *_operands(mode, terms, B, L, i, g, dev), 1e-6)
        assert pair is None or pair[0].isfinite().all()


@pytest.mark.parametrize("mode,agg", list(itertools.product([m for m in MODES if m != "geo_mean"], range(4))))
@pytest.mark.parametrize("empty", [slice(2, 3), slice(None)])
def test_kept_token_gradients_without_a_valid_token(dev, mode, agg, empty):
    """A row, or a whole batch, whose mask is zero: its gradient is zero, or NaN for the mean over the row's tokens (0 / 0), at
    the same tokens on both routes."""
    terms = "plain" if mode == "gspo" and agg != 2 else "all"
    for i, (B, L) in enumerate([(9, 700), (4, 2049), (3, 4100)]):
        g = torch.Generator().manual_seed(i)
        old, lp, adv, mask, *rest = _operands(mode, terms, B, L, i, g, dev)
        mask[empty] = 0
        got, want = _compare(dev, mode, agg, terms, old, lp, adv, mask, *rest, 1e-6)
        nan = agg == 2 or mode == "gspo"
        assert (got[empty].isnan() if nan else got[empty] == 0).all() and got.isnan().sum() == (got[empty].numel() if nan else 0)


def test_autograd_takes_the_kept_gradients(dev):
    """Above the rule's line: two backwards of one graph, the entropy's gradient, changed operands."""
    B, L = 1025, 2052
    f = lambda: torch.randn(B, L, device=dev)  # noqa: E731
    torch.manual_seed(3)
    lp, old, adv, ref, ent = 0.3 * f(), 0.3 * f(), f(), 0.3 * f(), f().abs()
    mask = (torch.rand(B, L, device=dev) < 0.7).long()
    args = (0, 0.2, 0.28, 3.0, 20.0, 0, 0.01, 3, False, 0.1, 0.0, 0.7)
    leaf, eleaf = lp.clone().requires_grad_(True), ent.clone().requires_grad_(True)
    outs = torch.ops.siirl_hip.actor_loss(leaf, eleaf, old, adv, mask, None, ref, *args, False, None)
    up = torch.tensor(1.7, device=dev)
    got, got_e = torch.autograd.grad(outs[0], [leaf, eleaf], up, retain_graph=True)
    (again,) = torch.autograd.grad(outs[0], leaf, 2 * up)
    fwd = torch.ops.siirl_hip.policy_loss_fwd(old, lp, adv, mask, None, ent, ref, *args)
    want, want_e = torch.ops.siirl_hip.policy_loss_bwd(up.reshape(1), old, lp, adv, mask, None, ent, ref, *args, *fwd)
    bound = 1e-6 * want.abs().amax(1, keepdim=True)
    assert not torch.equal(got, want)  # (the other order of the products: it is the kept gradients that were scaled)
    assert ((got - want).abs() <= bound).all() and ((again - 2 * want).abs() <= 2 * bound).all()
    assert torch.equal(got_e, want_e)
    outs = torch.ops.siirl_hip.actor_loss(leaf, None, old, adv, mask, None, ref, *args, False, None)
    old += 1.0  # a saved operand that changes before the backward is refused, though the backward would not read it
    with pytest.raises(RuntimeError, match="modified by an inplace operation"):
        torch.autograd.grad(outs[0], leaf)


@pytest.mark.parametrize("mode", ["kl_cov", "clip_cov"])
def test_autograd_takes_the_kept_gradients_of_the_covariance_losses(dev, mode):
    B, L = 1025, 2052
    g = torch.Generator().manual_seed(11)
    f = lambda: torch.randn(B, L, generator=g).to(dev)  # noqa: E731
    lp, old, adv, ref = 0.3 * f(), 0.3 * f(), f(), 0.3 * f()
    mask, aux = (torch.rand(B, L, generator=g) < 0.7).long().to(dev), _aux(mode, B, L, g, dev)
    args = (CA._LOSS_CODES[mode], 0.2, 0.28, 3.0, 20.0, 0, 0.0, 3, True, 0.1, 0.0, 0.7)
    leaf, up = lp.clone().requires_grad_(True), torch.tensor(1.7, device=dev)
    (got,) = torch.autograd.grad(torch.ops.siirl_hip.actor_loss(leaf, None, old, adv, mask, None, ref, *args, False, aux)[0],
                                 leaf, up)
    fwd = torch.ops.siirl_hip.policy_loss_fwd(old, lp, adv, mask, None, None, ref, *args, aux)
    want, _ = torch.ops.siirl_hip.policy_loss_bwd(up.reshape(1), old, lp, adv, mask, None, None, ref, *args, *fwd, aux)
    assert not torch.equal(got, want)
    assert ((got - want).abs() <= 1e-6 * want.abs().amax(1, keepdim=True)).all()


def test_no_gradient_is_kept_for_nothing(dev):
    """Without differentiation the forward allocates no [B, L] buffer."""
    lp, old, adv = (torch.randn(1025, 2052, device=dev) for _ in range(3))
    mask = torch.ones_like(lp, dtype=torch.bool)
    args = (0, 0.2, 0.2, 3.0, 20.0, 0, 0.0, 0, False, 0.0, 0.0, 1.0, False, None)
    torch.ops.siirl_hip.actor_loss(lp, None, old, adv, mask, None, None, *args)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    torch.ops.siirl_hip.actor_loss(lp, None, old, adv, mask, None, None, *args)
    assert torch.cuda.max_memory_allocated() - before < lp.numel()


def test_a_kept_gradient_keeps_no_copy_of_an_operand(dev):
    """Half-precision and strided operands are converted for the forward; with the tokens' gradients kept, the backward reads
    none of them, and the node holds the gradient and the result block (under a quarter of it here) alone."""
    B, L = 1025, 2052
    torch.manual_seed(5)
    lp, old, ref, ent = (torch.randn(B, L, device=dev, dtype=torch.bfloat16) for _ in range(4))
    adv, mask = torch.randn(L, B, device=dev).t(), (torch.rand(L, B, device=dev) < 0.7).double().t()
    args = (0, 0.2, 0.28, 3.0, 20.0, 0)
    tail = (3, False, 0.1, 0.0, 0.7, False, None)
    lp, ent = lp.requires_grad_(True), ent.requires_grad_(True)
    for with_ent in (False, True):
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        outs = torch.ops.siirl_hip.actor_loss(lp, ent if with_ent else None, old, adv, mask, None, ref, *args, 0.01, *tail)
        held = torch.cuda.memory_allocated() - before
        assert held < (2.25 if with_ent else 1.25) * 4 * B * L, held  # an entropy's gradient reads the (converted) mask
        got = torch.autograd.grad(outs[0], [lp, ent] if with_ent else [lp])
        leaf, eleaf = lp.detach().float().requires_grad_(True), ent.detach().float().requires_grad_(True)
        outs = torch.ops.siirl_hip.actor_loss(leaf, eleaf if with_ent else None, old.float(), adv.contiguous(),
                                              mask.float().contiguous(), None, ref.float(), *args, 0.01, *tail)
        want = torch.autograd.grad(outs[0], [leaf, eleaf] if with_ent else [leaf])
        for a, b in zip(got, want):
            assert torch.equal(a, b.to(torch.bfloat16))
        del outs, got, want
