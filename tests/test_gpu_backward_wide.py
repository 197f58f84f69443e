"""dK, dV and dS at head size 128 on wavefronts of 64 keys (key tiles with sixteen or 24 steps and more on average) against the form without dS in memory: rows and keys
around the tiles of 64 and 128 and their halves, a tile of rows that is the sequence's only one, wavefronts without keys or rows, more queries than keys
and the other way round, one to many steps, shares, fp32 gradients, several passes.  Every case says which kernel it is for, and how many shares it has; calls next
to them run on the other kernel.  Tolerance of test_gpu_backward.py: one rounding of the result over a tensor."""
import ctypes

import pytest
import torch

from mi355_attn import _lib, ops as inner
from test_gpu_backward import _both_forms, _packed_gradients, _same_gradients, check_grad, ops, rnd  # noqa: F401

ROLES, WIDE = 1, 2
# lens_q, lens_k (None: the same), query heads, kv heads, causal | kernel, shares
PACKED = [
    ([1, 900, 33, 0, 830, 64, 65], None, 8, 1, True, ROLES, 8), ([31, 32, 33, 1800, 97, 95, 96], None, 16, 2, True, ROLES, 8), ([1700, 1, 129, 1023], [1800, 300, 64, 900], 6, 2, True, ROLES, 8),
    ([800, 1, 63, 900], [129, 64, 1, 127], 3, 1, False, ROLES, 4), ([2100, 2000], [40, 2100], 4, 4, True, ROLES, 4), ([700, 900, 64], [66, 193, 32], 4, 2, False, ROLES, 2),
    ([2113] * 5, None, 12, 12, True, WIDE, 1), ([1, 900, 33, 0, 830, 64, 65], None, 96, 1, True, WIDE, 8), ([31, 32, 33, 700, 97, 95, 96], None, 160, 1, True, WIDE, 8),
    ([1700, 1, 129, 1023], [1800, 300, 64, 900], 144, 24, True, WIDE, 1), ([800, 1, 63, 900], [129, 64, 1, 127], 64, 2, False, WIDE, 8), ([2100, 2000], [40, 2100], 32, 32, True, WIDE, 1),
    ([700, 900, 64], [66, 193, 32], 96, 4, False, WIDE, 8), ([1025, 700, 33], [97, 161, 225], 128, 64, False, WIDE, 1)]
# batch, query heads, kv heads, queries, keys, causal, fp32 gradients | kernel, shares
DENSE = [
    (3, 16, 2, 289, 289, True, True, ROLES, 4), (1, 12, 12, 2625, 2625, True, False, ROLES, 2), (2, 24, 3, 600, 130, False, False, ROLES, 8), (5, 8, 8, 1700, 65, False, True, ROLES, 2),
    (9, 16, 1, 321, 500, True, False, ROLES, 4), (1, 32, 1, 1217, 1217, True, True, ROLES, 16), (1, 48, 1, 1217, 1217, True, True, WIDE, 16), (30, 96, 8, 289, 289, True, True, WIDE, 1), (1, 24, 24, 2625, 2625, True, False, WIDE, 1),
    (2, 64, 2, 600, 130, False, False, WIDE, 8), (64, 8, 8, 1025, 97, False, True, WIDE, 1), (64, 8, 8, 1025, 161, False, False, WIDE, 1), (17, 80, 4, 321, 500, True, False, WIDE, 2), (9, 160, 4, 321, 500, True, False, WIDE, 4), (3, 32, 8, 1600, 1600, True, False, WIDE, 2),
    (1, 16, 16, 2090, 2050, True, False, WIDE, 1)]
PASSES = [(1000, ROLES), (1600, WIDE)]
UNSEEN = [(2050, 2050), (2050, 2090), (2090, 2050)]


def _kernel(lens_q, lens_k, Hq, Hkv, causal, packed, promise_q=None, promise_k=None):
    shares = ctypes.c_int(0)
    kernel = _lib.load().mi355_prefill_bwd_ds_kernel(
        len(lens_q), Hq, Hkv, promise_q or max(lens_q), promise_k or max(lens_k), 128, _lib.MASK_CAUSAL if causal else _lib.MASK_NONE, packed, not packed or lens_q == lens_k,
        sum(lens_q) if packed else 0, sum(lens_k) if packed else 0, ctypes.byref(shares))
    return kernel, shares.value


def test_cases_run_on_the_kernel_that_they_are_for():
    """(host code: no GPU needed)"""
    for lens_q, lens_k, Hq, Hkv, causal, *want in PACKED:
        assert list(_kernel(lens_q, lens_k or lens_q, Hq, Hkv, causal, True)) == want, (lens_q, Hq, Hkv)
    for B, Hq, Hkv, Sq, Sk, causal, _, *want in DENSE:
        assert list(_kernel([Sq] * B, [Sk] * B, Hq, Hkv, causal, False)) == want, (B, Hq, Hkv, Sq, Sk)
    for n, want in PASSES:
        for packed in (True, False):
            assert _kernel([n] * 3, [n] * 3, 28, 14, True, packed) == (want, 1)
    for Sq, Sk in UNSEEN:
        assert _kernel([Sq], [Sk], 16, 16, True, False) == (WIDE, 1)
    assert {shares for *_, kernel, shares in PACKED + DENSE if kernel == WIDE} == {1, 2, 4, 8, 16}
    assert _kernel([4096], [4096], 32, 8, True, False)[0] == WIDE and _kernel([64], [64], 8, 8, True, False) == (0, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("lens_q,lens_k,Hq,Hkv,causal,kernel,shares", PACKED)
def test_wide_packed(ops, monkeypatch, lens_q, lens_k, Hq, Hkv, causal, kernel, shares):  # noqa: F811
    print(f"case: wide packed {lens_q} {lens_k} {Hq}/{Hkv} {causal} {kernel} {shares}", flush=True)
    _same_gradients(*_both_forms(ops, monkeypatch, lens_q, lens_k or lens_q, Hq, Hkv, causal, True))


@pytest.mark.gpu
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,causal,f32,kernel,shares", DENSE)
def test_wide_dense(ops, monkeypatch, B, Hq, Hkv, Sq, Sk, causal, f32, kernel, shares):  # noqa: F811
    """(strided queries and gradients; one key head and several shares of its row tiles; fp32 gradients)"""
    print(f"case: wide dense {B} {Hq}/{Hkv} {Sq} {Sk} {causal} {kernel} {shares}", flush=True)
    _same_gradients(*_both_forms(ops, monkeypatch, [Sq] * B, [Sk] * B, Hq, Hkv, causal, False, f32=f32))


@pytest.mark.gpu
@pytest.mark.parametrize("n,kernel", PASSES)
@pytest.mark.parametrize("packed", [True, False])
def test_wide_in_passes(ops, monkeypatch, packed, n, kernel):  # noqa: F811
    print(f"case: wide in passes {packed} {n} {kernel}", flush=True)
    _same_gradients(*_both_forms(ops, monkeypatch, [n] * 3, [n] * 3, 28, 14, True, packed, workspace_part=0.45))


@pytest.mark.gpu
def test_wide_sequences_beyond_the_promise(ops):  # noqa: F811
    """Up to the next multiple of 256: the gradients of the right promise, all rows of them."""
    lens, short = [2040] * 8 + [30], 1900
    print(f"case: wide, short promise {lens} {short}", flush=True)
    assert _kernel(lens, lens, 4, 2, False, True, short, short)[0] == _kernel(lens, lens, 4, 2, False, True)[0] == WIDE
    torch.full((1 << 28,), float("nan"), device="cuda")                  # (what is not written shows)
    got = _packed_gradients(ops, lens, None, short, short, False)
    _same_gradients(got, _packed_gradients(ops, lens, None, 2040, 2040, False))


@pytest.mark.gpu
@pytest.mark.parametrize("Sq,Sk", UNSEEN)
def test_wide_of_a_key_whose_dp_overflows_in_rows_that_do_not_see_it(ops, Sq, Sk):  # noqa: F811
    """dO . v of a key is beyond fp32 (1e15 * 1e25 * 128) in rows that do not see it: nothing that a row's dQ adds, and nothing of other keys' dK.  Keys that no row of a
    half tile sees have no dS written where the diagonal is no multiple of 64 off; the memory that they take is full of NaN beforehand."""
    print(f"case: wide, unseen overflow {Sq} {Sk}", flush=True)
    at, head, H = 150, 3, 16
    first = at - (Sk - Sq)                                               # the first row that sees the key
    q, dout = (rnd(1, H, Sq, 128, seed=s).cuda() for s in (440, 443))
    k, v = (rnd(1, H, Sk, 128, seed=s).cuda() for s in (441, 442))
    v[:, :, at] *= 1e25
    dout[:, :, :first] *= 1e15
    dout[:, :, first:] *= 1e-25
    leaves = [t.requires_grad_() for t in (q, k, v)]
    out = ops.flash_attn_prefill(*leaves, causal=True)
    torch.full((1 << 28,), float("nan"), device="cuda")
    grads = torch.autograd.grad(out, leaves, dout)
    wide = [t[0, head].detach().double().requires_grad_() for t in (q, k, v)]
    sees = torch.arange(Sk, device="cuda")[None] <= torch.arange(Sq, device="cuda")[:, None] + Sk - Sq
    none = ~sees.any(-1, keepdim=True)                                   # (rows without keys add nothing)
    p = torch.softmax((wide[0] @ wide[1].T / 128 ** 0.5).masked_fill(~(sees | none), -float("inf")), -1).masked_fill(none, 0.0)
    want = torch.autograd.grad(p @ wide[2], wide, dout[0, head].double())
    for name, cut, got, ref in zip(("dq", "dk", "dv"), (first, at, at), grads, want):
        got = got[0, head].double()
        for part in (slice(0, cut), slice(cut, cut + 1), slice(cut + 1, None)):                  # (sizes of their own)
            if name == "dk" and part.start == at:                        # (the key's own dK is NaN)
                continue
            assert bool(torch.isfinite(got[part]).all()), name
            size = ref[part].abs().max()
            check_grad(name, (got[part] / size).cpu(), (ref[part] / size).cpu())


@pytest.mark.gpu
@pytest.mark.parametrize("packed,lens,Hq,Hkv", [(True, [2113] * 5, 12, 12), (True, [300, 31, 1], 4, 2), (False, [200] * 3, 8, 2)])
def test_delta_is_what_the_header_says(ops, monkeypatch, packed, lens, Hq, Hkv):  # noqa: F811
    """rowsum(dout * out) in the caller's tensor, whichever kernel reads it: within the rounding of its fp32 sum of 128 products."""
    print(f"case: delta {packed} {lens} {Hq}/{Hkv}", flush=True)
    lib, seen = _lib.load(), []
    real, real_backward = lib.mi355_prefill_bwd_ds, inner._prefill_backward

    def backward(q, k, v, out, dout, lse, *rest, **kw):
        delta = torch.full_like(lse, float("nan"))
        monkeypatch.setattr(lib, "mi355_prefill_bwd_ds", lambda *a: real(*a[:6], delta.data_ptr(), *a[7:]))
        grads = real_backward(q, k, v, out, dout, lse, *rest, **kw)
        seen.append((delta, out, dout))
        return grads

    monkeypatch.setattr(inner, "_prefill_backward", backward)
    _both_forms(ops, monkeypatch, lens, lens, Hq, Hkv, True, packed)
    delta, out, dout = seen[0]                                           # (the first form is the one with dS in memory)
    products = out.double() * dout.double()
    want, size = products.sum(-1), products.abs().sum(-1)
    if packed:
        want, size = want.T, size.T
    assert bool(((delta.double() - want).abs() <= 128 * 2 ** -24 * size).all())
