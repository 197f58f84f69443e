"""The prefill kernel that deals a query tile's keys to the wavefronts of a workgroup, at its edges: lengths around its 32 rows and
32 keys, wavefronts without keys, four and eight wavefronts, sequences longer than promised, more and fewer keys than queries,
block ids over more than one of the windows that a wavefront holds.  bf16 bound of test_gpu_parity.py, from the rounding of the
weights and of the result to 8 bits."""
import math

import pytest
import torch

from oracle import attention_oracle as orc
from test_gpu_parity import check, ops, rnd  # noqa: F401

pytestmark = pytest.mark.gpu


def _cu(lens):
    return torch.tensor([0] + list(torch.tensor(lens).cumsum(0)), dtype=torch.int32)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("Hq,Hkv", [(2, 2), (6, 2)])
@pytest.mark.parametrize("lens", [(1, 31, 32, 33, 0, 64, 127, 129, 300), (600, 5, 545), (512,), (511, 1)])
def test_packed_lengths(ops, D, Hq, Hkv, lens):  # noqa: F811
    """(512 keys and more with few workgroups: eight wavefronts, otherwise four)"""
    print(f"case: keys dealt D={D} {Hq}/{Hkv} {lens}", flush=True)
    T, cu = sum(lens), _cu(lens)
    q, k, v = rnd(T, Hq, D, seed=1), rnd(T, Hkv, D, seed=2), rnd(T, Hkv, D, seed=3)
    args = (q.cuda(), k.cuda(), v.cuda(), cu.cuda(), cu.cuda())
    for causal in (True, False):
        ref = orc.varlen_prefill_reference(q, k, v, cu, cu, causal=causal)
        check(ops.flash_attn_varlen_prefill(*args, max(lens), max(lens), causal=causal, kv_splits=1), ref, what=f"{causal}")
        check(ops.flash_attn_varlen_prefill(*args, max(1, max(lens) // 3), max(1, max(lens) // 3), causal=causal, kv_splits=1), ref,
              what=f"{causal}, promise too small")


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("Sq,Sk", [(40, 333), (333, 40), (1, 700), (33, 31), (290, 1)])
def test_dense_rows_and_keys(ops, D, Sq, Sk):  # noqa: F811
    """Strided rows (views of a (batch, seq, heads, d) projection), other numbers of keys than queries; queries without a key are NaN."""
    print(f"case: keys dealt, dense D={D} {Sq} {Sk}", flush=True)
    q, k, v = (rnd(2, n, 3, D, seed=10 + i).permute(0, 2, 1, 3) for i, n in enumerate((Sq, Sk, Sk)))
    for causal in (True, False):
        ref = orc.prefill_reference(q, k, v, causal=causal)
        got = ops.flash_attn_prefill(q.cuda(), k.cuda(), v.cuda(), causal=causal, kv_splits=1).cpu()
        none = max(0, Sq - Sk) if causal else 0
        assert torch.isnan(got[:, :, :none]).all()
        check(got[:, :, none:], ref[:, :, none:], what=f"{causal}")


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("Hq,rows,ctx", [(2, (40, 3), (9000, 70)), (16, (544,), (4200,)), (4, (17, 100, 1), (33, 100, 16)), (1, (300,), (305,))])
def test_block_tables(ops, D, Hq, rows, ctx):  # noqa: F811
    """9000 keys: two windows of ids with eight wavefronts; 4200 keys with more than 256 workgroups: two with four."""
    print(f"case: keys dealt, paged D={D} {Hq} {rows} {ctx}", flush=True)
    _, kc, vc, bt, cl = orc.make_paged_case(batch=len(ctx), n_q_heads=Hq, n_kv_heads=Hq, head_dim=D, block_size=16, context_lens=list(ctx), seed=5,
                                            dtype=torch.bfloat16)
    q, cu = rnd(sum(rows), Hq, D, seed=6), _cu(rows)
    ref = orc.paged_prefill_reference(q, kc, vc, cu, bt, cl)
    got = ops.flash_attn_paged_prefill(q.cuda(), kc.cuda(), vc.cuda(), cu.cuda(), bt.cuda(), cl.cuda(), max(rows), max_context=max(ctx), kv_splits=1)
    check(got, ref, what="paged")


@pytest.mark.parametrize("D", [32, 64, 128])
def test_scores_of_any_size_and_their_sums(ops, D):  # noqa: F811
    """Rows whose scores are all far below or above zero, of which one wavefront sees the largest, and gradients, which take the log-sum-exps from here
    (their bound: what rounding P and dS to 8 bits leaves, as in test_gpu_backward.py)."""
    print(f"case: keys dealt, scores D={D}", flush=True)
    q, k, v = rnd(1, 2, 200, D, seed=20), rnd(1, 2, 200, D, seed=21), rnd(1, 2, 200, D, seed=22)
    for shift in (-300.0, 300.0):
        k2 = k.clone()
        k2[..., 0] = shift
        q2 = q.clone()
        q2[..., 0] = math.sqrt(D)                                 # every score moves by shift
        k2[:, :, 37] += 0.25
        check(ops.flash_attn_prefill(q2.cuda(), k2.cuda(), v.cuda(), kv_splits=1), orc.prefill_reference(q2, k2, v), what=f"{shift}")
    mine = [t.cuda().requires_grad_() for t in (q, k, v)]
    want = [t.float().requires_grad_() for t in (q, k, v)]
    dout = rnd(1, 2, 200, D, seed=23)
    got = torch.autograd.grad(ops.flash_attn_prefill(*mine), mine, dout.cuda())
    s = (want[0] @ want[1].transpose(-1, -2) / math.sqrt(D)).masked_fill(~torch.ones(200, 200).tril().bool(), -math.inf)
    for g, w in zip(got, torch.autograd.grad(torch.softmax(s, -1) @ want[2], want, dout.float())):
        check(g, w, atol=2e-2 * float(w.abs().max()), rtol=2e-2, what="gradient")


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("S", [40, 300])
def test_means_of_the_largest_and_of_tiny_values(ops, D, S):  # noqa: F811
    """Rows are means of values: finite for the largest finite ones, and of the values' own size for tiny ones (300 keys: eight wavefronts).  Within a column values
    are equal, so a row is the column's value: rounding of the result to 8 bits."""
    from mi355_attn import _lib
    lib = _lib.load()
    assert lib.mi355_prefill_kernel(1, 2, 2, D, S, S, 1, 1, 0, 0, 1, 0, 0, None) == 4
    print(f"case: keys dealt, values D={D} {S}", flush=True)
    q, k, cu = rnd(S, 2, D, seed=30), rnd(S, 2, D, seed=31), _cu([S])
    for size in (torch.finfo(torch.bfloat16).max, 2.0 ** -100):
        v = (torch.linspace(-1, 1, D) * size).to(torch.bfloat16).repeat(S, 2, 1)
        got = ops.flash_attn_varlen_prefill(q.cuda(), k.cuda(), v.cuda(), cu.cuda(), cu.cuda(), S, S, kv_splits=1).double().cpu()
        assert bool(((got - v.double()).abs() <= 2.0 ** -8 * v.double().abs()).all()), size
