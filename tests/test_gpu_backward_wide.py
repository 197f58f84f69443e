"""dK, dV and dS at head size 128 on wavefronts of 64 keys (key tiles with sixteen steps and more on average) against the form without dS in memory: rows and keys
around the tiles of 64 and 128 and their halves, a tile of rows that is the sequence's only one, wavefronts without keys or rows, more queries than keys
and the other way round, one to many steps, shares, fp32 gradients, several passes.  Tolerance of test_gpu_backward.py: one rounding of the result over a tensor."""
import pytest
import torch

from mi355_attn import ops as inner
from test_gpu_backward import _both_forms, _same_gradients, ops  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens_q,lens_k,Hq,Hkv,causal", [
    ([1, 900, 33, 0, 830, 64, 65], None, 8, 1, True), ([31, 32, 33, 1800, 97, 95, 96], None, 16, 2, True), ([1700, 1, 129, 1023], [1800, 300, 64, 900], 6, 2, True),
    ([800, 1, 63, 900], [129, 64, 1, 127], 3, 1, False), ([2100, 2000], [40, 2100], 4, 4, True), ([700, 900, 64], [66, 193, 32], 4, 2, False),
    ([2113] * 5, None, 12, 12, True)])
def test_wide_packed(ops, monkeypatch, lens_q, lens_k, Hq, Hkv, causal):  # noqa: F811
    print(f"case: wide packed {lens_q} {lens_k} {Hq}/{Hkv} {causal}", flush=True)
    _same_gradients(*_both_forms(ops, monkeypatch, lens_q, lens_k or lens_q, Hq, Hkv, causal, True))


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,causal,f32", [(3, 16, 2, 289, 289, True, True), (1, 12, 12, 2625, 2625, True, False), (2, 24, 3, 600, 130, False, False),
                                                       (5, 8, 8, 1700, 65, False, True), (9, 16, 1, 321, 500, True, False), (1, 32, 1, 1217, 1217, True, True)])
def test_wide_dense(ops, monkeypatch, B, Hq, Hkv, Sq, Sk, causal, f32):  # noqa: F811
    """(strided queries and gradients; one key head and several shares of its row tiles; fp32 gradients)"""
    print(f"case: wide dense {B} {Hq}/{Hkv} {Sq} {Sk} {causal}", flush=True)
    _same_gradients(*_both_forms(ops, monkeypatch, [Sq] * B, [Sk] * B, Hq, Hkv, causal, False, f32=f32))


@pytest.mark.parametrize("packed", [True, False])
def test_wide_in_passes(ops, monkeypatch, packed):  # noqa: F811
    print(f"case: wide in passes {packed}", flush=True)
    _same_gradients(*_both_forms(ops, monkeypatch, [1000] * 3, [1000] * 3, 28, 14, True, packed, workspace_part=0.45))


@pytest.mark.parametrize("packed,lens,Hq,Hkv", [(True, [2113] * 5, 12, 12), (True, [300, 31, 1], 4, 2), (False, [200] * 3, 8, 2)])
def test_delta_is_what_the_header_says(ops, monkeypatch, packed, lens, Hq, Hkv):  # noqa: F811
    """rowsum(dout * out) in the caller's tensor, whichever kernel reads it: within the rounding of its fp32 sum of 128 products."""
    from mi355_attn import _lib
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
