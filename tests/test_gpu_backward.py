"""GPU parity of the prefill backward (dq, dk, dv) and of the forward's log-sum-exp against the
CPU oracle, through the C ABI (ops -> ctypes -> mi355_prefill_fwd_lse / mi355_prefill_bwd).

Tolerance: the kernels recompute P from bf16 inputs, round P and dS to bf16 for the second MFMA and
round the results to bf16; against the fp32 oracle on the same bf16 inputs a gradient element is
accepted within 1e-4 + 2e-2 * max|grad of that tensor| + 2e-2 |ref| (gradients of long sequences sum many
terms, so the absolute part scales with the tensor), and the relative RMS error must stay below 1.5 %.
lse: |got - ref| <= 3e-3 + 1e-3 |ref| (the kernels sum the weights as rounded to bf16 -- exactly what multiplies V --
so a row whose weights all round the same way is off by up to 2^-9 = 0.002 in its log-sum-exp).
"""
import pytest
import torch

from oracle import attention_oracle as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    import mi355_attn
    mi355_attn.load()
    return mi355_attn


def rnd(*shape, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(torch.bfloat16)


def check_grad(name, got, ref):
    got = got.float().cpu()
    err = (got - ref).abs()
    bound = 1e-4 + 2e-2 * float(ref.abs().max()) + 2e-2 * ref.abs()
    rms = float((got - ref).pow(2).mean().sqrt() / ref.pow(2).mean().sqrt().clamp_min(1e-3))
    assert bool((err <= bound).all()), f"{name}: max err {float(err.max()):.4g} (ref max {float(ref.abs().max()):.4g})"
    assert rms < 1.5e-2, f"{name}: relative rms error {rms:.4f}"


def run_dense(ops, B, Hq, Hkv, Sq, Sk, D, causal, seed, scale=None):
    q, k, v = rnd(B, Hq, Sq, D, seed=seed), rnd(B, Hkv, Sk, D, seed=seed + 1), rnd(B, Hkv, Sk, D, seed=seed + 2)
    dout = rnd(B, Hq, Sq, D, seed=seed + 3)
    qg, kg, vg = (t.cuda().requires_grad_() for t in (q, k, v))
    out = ops.flash_attn_prefill(qg, kg, vg, causal=causal, softmax_scale=scale)
    out.backward(dout.cuda())
    torch.cuda.synchronize()
    dq, dk, dv, _ = orc.prefill_backward_reference(q, k, v, dout, causal=causal, softmax_scale=scale)
    ref_out = orc.prefill_reference(q, k, v, causal=causal, softmax_scale=scale)
    torch.testing.assert_close(out.detach().float().cpu(), ref_out, atol=2e-2, rtol=1e-2)
    check_grad("dq", qg.grad, dq)
    check_grad("dk", kg.grad, dk)
    check_grad("dv", vg.grad, dv)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("causal", [True, False])
def test_backward_square(ops, D, causal):
    print(f"case: backward square D={D} causal={causal}", flush=True)
    run_dense(ops, 2, 4, 4, 256, 256, D, causal, seed=10 + D)


@pytest.mark.parametrize("Sq,Sk", [(1, 1), (7, 7), (65, 65), (129, 129), (200, 333), (128, 64 + 128), (33, 500)])
def test_backward_ragged_and_rectangular(ops, Sq, Sk):
    print(f"case: backward ragged Sq={Sq} Sk={Sk}", flush=True)
    run_dense(ops, 1, 2, 2, Sq, Sk, 64, True, seed=Sq + Sk)
    run_dense(ops, 1, 2, 2, Sq, Sk, 128, False, seed=Sq + Sk + 1)


def test_backward_gqa_and_custom_scale(ops):
    print("case: backward GQA", flush=True)
    run_dense(ops, 2, 8, 2, 192, 192, 128, True, seed=40)
    run_dense(ops, 1, 6, 1, 100, 100, 64, True, seed=41, scale=0.2)


def test_backward_config1_shape_with_reference_layouts(ops):
    """configs[1] (B4, H16, S1024, D64, causal) with the reference's tensor layouts: contiguous Q/K, V as the
    strided view of the (B, S, H*D) projection (model.py:367-370); dV must come back in V's layout."""
    print("case: backward config1 layouts", flush=True)
    B, H, S, D = 4, 16, 1024, 64
    q, k = rnd(B, H, S, D, seed=50, scale=0.5), rnd(B, H, S, D, seed=51, scale=0.5)
    vproj = rnd(B, S, H * D, seed=52, scale=0.5)
    dout = rnd(B, H, S, D, seed=53)
    qg, kg = q.cuda().requires_grad_(), k.cuda().requires_grad_()
    vp = vproj.cuda().requires_grad_()
    vview = vp.view(B, S, H, D).permute(0, 2, 1, 3)
    out = ops.sdpa_slot(qg, kg, vview, is_causal=True)
    out.backward(dout.cuda())
    torch.cuda.synchronize()
    v = vproj.view(B, S, H, D).permute(0, 2, 1, 3)
    dq, dk, dv, _ = orc.prefill_backward_reference(q, k, v, dout, causal=True)
    check_grad("dq", qg.grad, dq)
    check_grad("dk", kg.grad, dk)
    check_grad("dv", vp.grad.view(B, S, H, D).permute(0, 2, 1, 3), dv)


def test_backward_varlen_equals_per_sequence(ops):
    print("case: backward varlen", flush=True)
    lens = [37, 128, 1, 200, 64]
    Hq, Hkv, D = 4, 2, 128
    T = sum(lens)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    q, k, v, dout = rnd(T, Hq, D, seed=60), rnd(T, Hkv, D, seed=61), rnd(T, Hkv, D, seed=62), rnd(T, Hq, D, seed=63)
    qg, kg, vg = (t.cuda().requires_grad_() for t in (q, k, v))
    out = ops.flash_attn_varlen_prefill(qg, kg, vg, cu.cuda(), cu.cuda(), max(lens), max(lens), causal=True)
    out.backward(dout.cuda())
    torch.cuda.synchronize()
    dq_ref, dk_ref, dv_ref = torch.zeros(T, Hq, D), torch.zeros(T, Hkv, D), torch.zeros(T, Hkv, D)
    for b, n in enumerate(lens):
        sl = slice(int(cu[b]), int(cu[b + 1]))
        args = [t[sl].transpose(0, 1)[None] for t in (q, k, v, dout)]
        a, bb, c, _ = orc.prefill_backward_reference(*args, causal=True)
        dq_ref[sl], dk_ref[sl], dv_ref[sl] = a[0].transpose(0, 1), bb[0].transpose(0, 1), c[0].transpose(0, 1)
    check_grad("dq", qg.grad, dq_ref)
    check_grad("dk", kg.grad, dk_ref)
    check_grad("dv", vg.grad, dv_ref)


@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("seed", [0, 1])
def test_backward_packed_sequences_of_very_different_lengths(ops, D, seed):
    """Packed sequences from one token to several query tiles, 8 query heads on 2 kv heads: the grids of the two
    backward kernels then hold several chunks of workgroup ids per XCD, whole rounds of eight chunks and a partial
    one, and many workgroups of short sequences that have nothing to do."""
    g = torch.Generator().manual_seed(7000 + seed)
    n_seq = int(torch.randint(6, 10, (1,), generator=g))
    lens = [int(x) for x in torch.randint(1, 900, (n_seq,), generator=g)]
    lens[int(torch.randint(0, n_seq, (1,), generator=g))] = 1
    print(f"case: backward packed D={D} seed={seed} lens={lens}", flush=True)
    Hq, Hkv = 8, 2
    T = sum(lens)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32)
    q, k, v, dout = (rnd(T, Hq, D, seed=7100 + seed), rnd(T, Hkv, D, seed=7200 + seed), rnd(T, Hkv, D, seed=7300 + seed),
                     rnd(T, Hq, D, seed=7400 + seed))
    qg, kg, vg = (t.cuda().requires_grad_() for t in (q, k, v))
    out = ops.flash_attn_varlen_prefill(qg, kg, vg, cu.cuda(), cu.cuda(), max(lens), max(lens), causal=True)
    out.backward(dout.cuda())
    torch.cuda.synchronize()
    dq_ref, dk_ref, dv_ref = torch.zeros(T, Hq, D), torch.zeros(T, Hkv, D), torch.zeros(T, Hkv, D)
    for b in range(n_seq):
        sl = slice(int(cu[b]), int(cu[b + 1]))
        args = [t[sl].transpose(0, 1)[None] for t in (q, k, v, dout)]
        a, bb, c, _ = orc.prefill_backward_reference(*args, causal=True)
        dq_ref[sl], dk_ref[sl], dv_ref[sl] = a[0].transpose(0, 1), bb[0].transpose(0, 1), c[0].transpose(0, 1)
    check_grad("dq", qg.grad, dq_ref)
    check_grad("dk", kg.grad, dk_ref)
    check_grad("dv", vg.grad, dv_ref)


@pytest.mark.parametrize("D", [64, 128])
def test_forward_lse_matches_oracle(ops, D):
    """The log-sum-exp that comes from row sums and the exponent reference that went into them (as the sizes choose; each
    kernel by name in test_gpu_prefill_kernels.py) -- also after that reference has moved (keys with runaway scores),
    for ragged packed sequences, and for rows past the end of a partial query tile."""
    print(f"case: forward lse D={D}", flush=True)
    from mi355_attn import ops as raw
    B, Hq, Hkv, S = 2, 4, 2, 300
    q, k, v = rnd(B, Hq, S, D, seed=70, scale=2.0), rnd(B, Hkv, S, D, seed=71), rnd(B, Hkv, S, D, seed=72)
    out, lse = raw._dense(q.cuda(), k.cuda(), v.cuda(), None, 1, None, want_lse=True)
    torch.cuda.synchronize()
    _, _, _, lse_ref = orc.prefill_backward_reference(q, k, v, torch.zeros(B, Hq, S, D), causal=True)
    torch.testing.assert_close(lse.cpu(), lse_ref, atol=3e-3, rtol=1e-3)
    # the output is unchanged by asking for lse
    assert torch.equal(out, ops.flash_attn_prefill(q.cuda(), k.cuda(), v.cuda(), causal=True, kv_splits=1))
    # runaway keys, no mask, more keys than queries
    Sq, Sk = 200, 1100
    q, k, v = rnd(1, Hq, Sq, D, seed=73), rnd(1, Hkv, Sk, D, seed=74).float(), rnd(1, Hkv, Sk, D, seed=75)
    k[:, :, 500:520] *= 25.0
    k[:, :, 900] *= -40.0
    k = k.to(torch.bfloat16)
    out, lse = raw._dense(q.cuda(), k.cuda(), v.cuda(), None, 0, None, want_lse=True)
    _, _, _, lse_ref = orc.prefill_backward_reference(q, k, v, torch.zeros(1, Hq, Sq, D), causal=False)
    torch.testing.assert_close(lse.cpu(), lse_ref, atol=3e-3, rtol=1e-3)


def test_backward_is_deterministic_and_linear_in_dout(ops):
    print("case: backward determinism / linearity", flush=True)
    B, H, S, D = 1, 4, 384, 128
    q, k, v = rnd(B, H, S, D, seed=80).cuda(), rnd(B, H, S, D, seed=81).cuda(), rnd(B, H, S, D, seed=82).cuda()
    d1 = rnd(B, H, S, D, seed=83).cuda()

    def grads(dout):
        qg, kg, vg = (t.clone().requires_grad_() for t in (q, k, v))
        ops.flash_attn_prefill(qg, kg, vg, causal=True).backward(dout)
        return qg.grad, kg.grad, vg.grad

    a, b = grads(d1), grads(d1)
    for x, y in zip(a, b):
        assert torch.equal(x, y)
    c = grads(2 * d1)                               # exact in bf16: every product and sum doubles
    for x, y in zip(a, c):
        assert torch.equal((2 * x.float()).to(torch.bfloat16), y)


def test_no_grad_path_and_errors(ops):
    print("case: backward misc", flush=True)
    q = rnd(1, 2, 64, 64, seed=90).cuda().requires_grad_()
    k, v = rnd(1, 2, 64, 64, seed=91).cuda(), rnd(1, 2, 64, 64, seed=92).cuda()
    with torch.no_grad():
        out = ops.flash_attn_prefill(q, k, v)
    assert not out.requires_grad
    out = ops.flash_attn_prefill(q, k, v)
    assert out.requires_grad
    out.sum().backward()
    assert q.grad is not None and k.grad is None


def test_backward_rows_without_keys_and_empty_sequences(ops):
    """Causal with more queries than keys: the first Sq - Sk rows see no key (forward: NaN rows, like the
    reference softmax of an all-masked row); they must get dq = 0 and leave dk, dv untouched, i.e. the
    gradients equal those of the problem restricted to the rows that do see keys.  Packed batch with a
    sequence that has keys but no queries, and one with queries but no keys: every gradient row is
    written (zeros where nothing contributes)."""
    print("case: backward rows without keys / empty sequences", flush=True)
    B, Hq, Hkv, Sq, Sk, D = 1, 4, 2, 200, 130, 64
    q, k, v, dout = rnd(B, Hq, Sq, D, seed=90), rnd(B, Hkv, Sk, D, seed=91), rnd(B, Hkv, Sk, D, seed=92), rnd(B, Hq, Sq, D, seed=93)
    qg, kg, vg = (t.cuda().requires_grad_() for t in (q, k, v))
    out = ops.flash_attn_prefill(qg, kg, vg, causal=True)
    out.backward(dout.cuda())
    torch.cuda.synchronize()
    dead = Sq - Sk
    assert bool(torch.isnan(out[:, :, :dead].float()).all()) and bool(torch.isfinite(out[:, :, dead:].float()).all())
    dq_ref, dk_ref, dv_ref, _ = orc.prefill_backward_reference(q[:, :, dead:], k, v, dout[:, :, dead:], causal=True)
    assert bool((qg.grad[:, :, :dead] == 0).all())
    check_grad("dq", qg.grad[:, :, dead:], dq_ref)
    check_grad("dk", kg.grad, dk_ref)
    check_grad("dv", vg.grad, dv_ref)

    lens_q, lens_k = [70, 0, 33, 40], [70, 50, 33, 0]
    Hq, Hkv, D = 4, 2, 128
    cu_q = torch.tensor([0] + torch.tensor(lens_q).cumsum(0).tolist(), dtype=torch.int32)
    cu_k = torch.tensor([0] + torch.tensor(lens_k).cumsum(0).tolist(), dtype=torch.int32)
    Tq, Tk = sum(lens_q), sum(lens_k)
    q, k, v, dout = rnd(Tq, Hq, D, seed=94), rnd(Tk, Hkv, D, seed=95), rnd(Tk, Hkv, D, seed=96), rnd(Tq, Hq, D, seed=97)
    qg, kg, vg = (t.cuda().requires_grad_() for t in (q, k, v))
    out = ops.flash_attn_varlen_prefill(qg, kg, vg, cu_q.cuda(), cu_k.cuda(), max(lens_q), max(lens_k), causal=False)
    out.backward(dout.cuda())
    torch.cuda.synchronize()
    dq_ref, dk_ref, dv_ref = torch.zeros(Tq, Hq, D), torch.zeros(Tk, Hkv, D), torch.zeros(Tk, Hkv, D)
    for b in range(len(lens_q)):
        sq, sk = slice(int(cu_q[b]), int(cu_q[b + 1])), slice(int(cu_k[b]), int(cu_k[b + 1]))
        if lens_q[b] == 0 or lens_k[b] == 0:
            continue                                                   # nothing attends / nothing to attend: zero gradients
        args = [q[sq].transpose(0, 1)[None], k[sk].transpose(0, 1)[None], v[sk].transpose(0, 1)[None], dout[sq].transpose(0, 1)[None]]
        a, bb, c, _ = orc.prefill_backward_reference(*args, causal=False)
        dq_ref[sq], dk_ref[sk], dv_ref[sk] = a[0].transpose(0, 1), bb[0].transpose(0, 1), c[0].transpose(0, 1)
    assert bool(torch.isnan(out[int(cu_q[3]):].float()).all())        # queries without keys: NaN rows, as for any row that keeps no key
    check_grad("dq", qg.grad, dq_ref)
    check_grad("dk", kg.grad, dk_ref)
    check_grad("dv", vg.grad, dv_ref)


def oracle_masked_grads(q, k, v, mask, dout):
    """autograd through the oracle's restatement of model.py:308-325 in fp32: what the reference's own training step
    derives behind its non-flash branch."""
    qq, kk, vv = (t.float().requires_grad_() for t in (q, k, v))
    out = orc.scaled_dot_product_attention(qq, kk, vv, mask)
    out.backward(dout.float())
    return out.detach(), qq.grad, kk.grad, vv.grad


@pytest.mark.parametrize("S,D", [(256, 32), (200, 64), (131, 128), (384, 128)])
def test_masked_sdpa_trains_like_the_reference_non_flash_branch(ops, S, D):
    """llm-core/llm_core/model.py:384-385 as the reference runs it under autograd: the tril keep-mask rebuilt per call,
    handed to scaled_dot_product_attention with inputs that require grad.  Outputs and gradients against the oracle's
    causal backward (S = 131: rows that are no multiple of 4 bytes go through the padded copy of the mask)."""
    print(f"case: sdpa(Q, K, V, tril mask) under autograd S={S} D={D}", flush=True)
    B, H = 2, 4
    q, k, v, dout = (rnd(B, H, S, D, seed=300 + i + S) for i in range(4))
    qg, kg, vg = (t.cuda().requires_grad_() for t in (q, k, v))
    causal_mask = torch.tril(torch.ones(S, S, dtype=torch.bool, device="cuda"))          # model.py:384
    out = ops.scaled_dot_product_attention(qg, kg, vg, causal_mask)                        # model.py:385
    out.backward(dout.cuda())
    torch.cuda.synchronize()
    dq, dk, dv, _ = orc.prefill_backward_reference(q, k, v, dout, causal=True)
    torch.testing.assert_close(out.detach().float().cpu(), orc.prefill_reference(q, k, v, causal=True), atol=2e-2, rtol=1e-2)
    check_grad("dq", qg.grad, dq)
    check_grad("dk", kg.grad, dk)
    check_grad("dv", vg.grad, dv)


@pytest.mark.parametrize("mask_lead", ["none", "batch", "full"])
def test_masked_sdpa_backward_with_an_arbitrary_mask(ops, mask_lead):
    """A random keep-mask (no row fully masked), more keys than queries, the mask broadcast over heads and/or batch:
    gradients against autograd through the oracle's scaled_dot_product_attention."""
    print(f"case: sdpa backward, random mask, lead={mask_lead}", flush=True)
    B, H, Sq, Sk, D = 2, 3, 150, 212, 64
    q, k, v, dout = rnd(B, H, Sq, D, seed=400), rnd(B, H, Sk, D, seed=401), rnd(B, H, Sk, D, seed=402), rnd(B, H, Sq, D, seed=403)
    g = torch.Generator().manual_seed(404)
    lead = {"none": (), "batch": (B, 1), "full": (B, H)}[mask_lead]
    mask = torch.rand(*lead, Sq, Sk, generator=g) < 0.6
    mask[..., torch.arange(Sq), torch.arange(Sq)] = True
    qg, kg, vg = (t.cuda().requires_grad_() for t in (q, k, v))
    out = ops.scaled_dot_product_attention(qg, kg, vg, mask.cuda())
    out.backward(dout.cuda())
    torch.cuda.synchronize()
    ref, dq, dk, dv = oracle_masked_grads(q, k, v, mask, dout)
    torch.testing.assert_close(out.detach().float().cpu(), ref, atol=2e-2, rtol=1e-2)
    check_grad("dq", qg.grad, dq)
    check_grad("dk", kg.grad, dk)
    check_grad("dv", vg.grad, dv)


def test_masked_sdpa_backward_of_a_fully_masked_row(ops):
    """A query row whose keys are all masked: NaN output row like the reference softmax; its gradients are zero here
    (the reference propagates the NaN) and every other row's gradients are those of the problem without that row."""
    print("case: sdpa backward, one fully masked row", flush=True)
    B, H, S, D = 1, 2, 96, 64
    q, k, v, dout = (rnd(B, H, S, D, seed=500 + i) for i in range(4))
    mask = torch.tril(torch.ones(S, S, dtype=torch.bool))
    mask[17] = False
    qg, kg, vg = (t.cuda().requires_grad_() for t in (q, k, v))
    out = ops.scaled_dot_product_attention(qg, kg, vg, mask.cuda())
    out.backward(dout.cuda())
    torch.cuda.synchronize()
    assert bool(torch.isnan(out[:, :, 17].float()).all())
    keep = [i for i in range(S) if i != 17]
    _, dq, dk, dv = oracle_masked_grads(q[:, :, keep], k, v, mask[keep], dout[:, :, keep])
    assert bool((qg.grad[:, :, 17] == 0).all())
    check_grad("dq", qg.grad[:, :, keep], dq)
    check_grad("dk", kg.grad, dk)
    check_grad("dv", vg.grad, dv)


@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("Sq,Sk,causal", [(1, 1, True), (33, 33, True), (64, 129, True), (130, 130, False), (257, 300, True)])
def test_backward_of_many_short_heads(ops, D, Sq, Sk, causal):
    """More than 256 workgroups: the kernel with both roles in a wavefront; edges of the 32 keys of a wavefront, of the 64-row tiles
    and of the 128-key workgroups, pairs of key tiles and a middle one, two query heads per key head."""
    print(f"case: backward many heads D={D} {Sq} {Sk} {causal}", flush=True)
    run_dense(ops, 65, 8, 4, Sq, Sk, D, causal, seed=D + Sq)


@pytest.mark.parametrize("D", [32, 64])
def test_backward_of_many_packed_sequences_and_masks(ops, D):
    """The same kernel on packed sequences (some empty) against its dense runs, and under a mask of every element kept against no mask."""
    lens = [0, 1, 200, 17, 128, 0, 129] * 10
    H, G = 8, 4
    T = sum(lens)
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    q, k, v, do = (rnd(T, h, D, seed=s).cuda() for s, h in ((1, H), (2, G), (3, G), (4, H)))
    leaves = [t.requires_grad_() for t in (q, k, v)]
    grads = torch.autograd.grad(ops.flash_attn_varlen_prefill(q, k, v, cu, cu, 200, 200), leaves, do)
    at = 0
    for n in lens[:7]:
        if n:
            part = [t.detach()[at:at + n].transpose(0, 1)[None] for t in (q, k, v)]
            dq, dk, dv, _ = orc.prefill_backward_reference(*(t.cpu() for t in part), do[at:at + n].transpose(0, 1)[None].cpu(), causal=True)
            for name, got, ref in (("dq", grads[0], dq), ("dk", grads[1], dk), ("dv", grads[2], dv)):
                check_grad(name, got[at:at + n].transpose(0, 1)[None], ref)
        at += n
    B, S = 65, 100
    q, k, v, do = (rnd(B, 4, S, D, seed=s).cuda() for s in (5, 6, 7, 8))
    leaves = [t.requires_grad_() for t in (q, k, v)]
    keep = torch.ones(S, S, dtype=torch.bool, device="cuda")
    masked = torch.autograd.grad(ops.scaled_dot_product_attention(q, k, v, keep), leaves, do)
    plain = torch.autograd.grad(ops.scaled_dot_product_attention(q, k, v), leaves, do)
    for a, b in zip(masked, plain):          # (the two forwards differ in their exponent reference, so in the log-sum-exp's last bits)
        assert float((a.float() - b.float()).norm()) <= 2 ** -8 * float(b.float().norm())


@pytest.mark.parametrize("D,B", [(32, 65), (64, 65), (64, 1), (128, 1)])
def test_gradients_of_float32_inputs(ops, D, B):
    """float32 inputs are rounded to bf16 and get the float32 gradients that the bf16 ones are the rounding of."""
    H, S = 4, 70
    q, k = (torch.randn(B, H, S, D, generator=torch.Generator().manual_seed(s)).cuda() for s in (1, 2))
    v, do = rnd(B, S, H, D, seed=3).cuda().permute(0, 2, 1, 3), rnd(B, H, S, D, seed=4).cuda()
    mixed = [t.detach().clone().requires_grad_() for t in (q, k, v)]
    out = ops.sdpa_slot(*mixed)
    grads = torch.autograd.grad(out, mixed, do)
    half = [t.detach().to(torch.bfloat16).requires_grad_() for t in (q, k, v)]
    ref = ops.sdpa_slot(*half)
    want = torch.autograd.grad(ref, half, do)
    assert out.dtype == torch.bfloat16 and torch.equal(out, ref)
    assert [g.dtype for g in grads] == [torch.float32, torch.float32, torch.bfloat16] and grads[2].stride() == v.stride()
    for g, w in zip(grads, want):
        assert torch.equal(g.to(torch.bfloat16), w)


@pytest.mark.parametrize("lead", ["none", "batch", "full"])
@pytest.mark.parametrize("D,Sq,Sk", [(32, 77, 301), (64, 130, 212), (64, 67, 33)])
def test_masked_backward_of_many_short_heads(ops, D, Sq, Sk, lead):
    """Above 256 workgroups at head sizes 32 and 64: random keep-masks whose rows, columns, heads and sequences all differ (or are broadcast),
    odd sizes, a query row and a key that the mask leaves out altogether; against autograd through the oracle."""
    print(f"case: masked backward many heads D={D} {Sq} {Sk} {lead}", flush=True)
    B, H = 65, 4
    q, k, v, dout = (rnd(B, H, n, D, seed=600 + i + Sq) for i, n in enumerate((Sq, Sk, Sk, Sq)))
    mask = torch.rand(*{"none": (), "batch": (B, 1), "full": (B, H)}[lead], Sq, Sk, generator=torch.Generator().manual_seed(604)) < 0.6
    rows = torch.arange(Sq)
    mask[..., rows, rows % (Sk - 1)] = True
    mask[..., Sk - 1] = False                                             # nobody sees the last key
    mask[..., 17, :] = False                                              # a row that sees nothing
    leaves = [t.cuda().requires_grad_() for t in (q, k, v)]
    out = ops.scaled_dot_product_attention(*leaves, mask.cuda())
    dq, dk, dv = torch.autograd.grad(out, leaves, dout.cuda())
    assert bool(torch.isnan(out[:, :, 17].float()).all()) and bool((dq[:, :, 17] == 0).all())
    assert bool((dk[:, :, Sk - 1] == 0).all()) and bool((dv[:, :, Sk - 1] == 0).all())
    keep = [i for i in range(Sq) if i != 17]
    ref, rq, rk, rv = oracle_masked_grads(q[:, :, keep], k, v, mask[..., keep, :], dout[:, :, keep])
    torch.testing.assert_close(out.detach()[:, :, keep].float().cpu(), ref, atol=2e-2, rtol=1e-2)
    check_grad("dq", dq[:, :, keep], rq)
    check_grad("dk", dk, rk)
    check_grad("dv", dv, rv)


@pytest.mark.parametrize("D,copies", [(32, 1), (64, 1), (64, 33), (128, 1)])
def test_gradients_of_float32_inputs_packed_and_masked(ops, D, copies):
    """All three inputs float32, packed sequences (one of them empty) and explicit masks, fewer and more than 256 workgroups: the float32
    gradients are those that the bf16 inputs' gradients are the rounding of."""
    print(f"case: fp32 gradients packed and masked D={D} x{copies}", flush=True)
    lens = [70, 0, 33, 1, 130] * copies
    T, H, G = sum(lens), 4, 2
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()

    def both(call, q, k, v, do):
        full = [t.cuda().requires_grad_() for t in (q, k, v)]
        half = [t.detach().to(torch.bfloat16).requires_grad_() for t in full]
        out, ref = call(*full), call(*half)
        assert out.dtype == torch.float32 and torch.equal(out, ref.float())
        got, want = torch.autograd.grad(out, full, do.float().cuda()), torch.autograd.grad(ref, half, do.cuda())
        for name, g, w in zip(("dq", "dk", "dv"), got, want):
            assert g.dtype == torch.float32 and w.dtype == torch.bfloat16 and bool(torch.isfinite(g).all()), name
            assert torch.equal(g.to(torch.bfloat16), w), name
            assert not torch.equal(g, w.float()), name                    # (not rounded on the way)

    g = torch.Generator().manual_seed(D)
    q, k, v = (torch.randn(T, h, D, generator=g) for h in (H, G, G))
    both(lambda *t: ops.flash_attn_varlen_prefill(*t, cu, cu, 130, 130), q, k, v, rnd(T, H, D, seed=5))
    B, Sq, Sk = 3 * copies, 45, 67
    mask = (torch.rand(B, 1, Sq, Sk, generator=g) < 0.7).cuda()
    mask[..., 0] = True
    q, k, v = (torch.randn(B, H, n, D, generator=g) for n in (Sq, Sk, Sk))
    both(lambda *t: ops.scaled_dot_product_attention(*t, mask), q, k, v, rnd(B, H, Sq, D, seed=6))


def test_gradients_of_broadcast_float32_inputs(ops):
    """One float32 key and value head behind several query heads, as views: the gradients of what is shared are the sums over who shares it."""
    print("case: fp32 broadcast gradients", flush=True)
    B, H, S, D = 2, 4, 50, 64
    g = torch.Generator().manual_seed(9)
    q, k, v = torch.randn(B, H, S, D, generator=g), torch.randn(B, 1, S, D, generator=g), torch.randn(1, 1, S, D, generator=g)
    do = rnd(B, H, S, D, seed=4)
    leaves = [t.cuda().requires_grad_() for t in (q, k, v)]
    dq, dk, dv = torch.autograd.grad(ops.scaled_dot_product_attention(*leaves), leaves, do.float().cuda())
    b = [t.to(torch.bfloat16).float().requires_grad_() for t in (q, k, v)]
    ref = torch.autograd.grad(torch.softmax(b[0] @ b[1].transpose(-1, -2) / D ** 0.5, -1) @ b[2], b, do.float())
    assert dk.shape == k.shape and dv.shape == v.shape
    for name, got, want in zip(("dq", "dk", "dv"), (dq, dk, dv), ref):
        check_grad(name, got, want)


def _both_forms(ops, monkeypatch, lens_q, lens_k, Hq, Hkv, causal, packed, f32=False, workspace_part=1.0, D=128, spare=0):
    """Gradients with dS in memory and with S and dP computed again, of one forward pass."""
    from mi355_attn import _lib, ops as inner
    lib = _lib.load()
    real = lib.mi355_prefill_bwd_ds_workspace
    dt = torch.float32 if f32 else torch.bfloat16
    mode = _lib.MASK_CAUSAL if causal else _lib.MASK_NONE
    if packed:
        cu_q, cu_k = (torch.tensor([0] + torch.tensor(n).cumsum(0).tolist(), dtype=torch.int32).cuda() for n in (lens_q, lens_k))
        if lens_q == lens_k:
            cu_k = cu_q
        Tq, Tk, Sq, Sk = sum(lens_q), sum(lens_k), max(lens_q) + spare, max(lens_k) + spare
        qkv = rnd(max(Tq, Tk), Hq + 2 * Hkv, D, seed=400, scale=0.5).cuda()
        q, k, v, dout = qkv[:Tq, :Hq], qkv[:Tk, Hq:Hq + Hkv], qkv[:Tk, Hq + Hkv:], rnd(Tq, Hq, D, seed=401, scale=0.5).cuda()
        out, lse = inner._varlen(q, k, v, cu_q, cu_k, Sq, Sk, causal, None, want_lse=True)
    else:
        B, Sq, Sk = len(lens_q), lens_q[0], lens_k[0]
        cu_q = cu_k = None
        q, dout = (rnd(B, Sq, Hq, D, seed=s, scale=0.5).cuda().permute(0, 2, 1, 3) for s in (402, 403))
        k, v = (rnd(B, Hkv, Sk, D, seed=s, scale=0.5).cuda() for s in (404, 405))
        out, lse = inner._dense(q, k, v, None, mode, None, want_lse=True)
    asked = []

    def workspace(*a):
        asked.append(real(*a))
        return int(asked[-1] * workspace_part) // 4096 * 4096

    grads = []
    for fn in (workspace, lambda *a: 0):
        monkeypatch.setattr(lib, "mi355_prefill_bwd_ds_workspace", fn)
        grads.append(inner._prefill_backward(q, k, v, out, dout, lse, cu_q, cu_k, Sq, Sk, D ** -0.5, mode, dtypes=(dt,) * 3))
    torch.cuda.synchronize()
    assert asked and asked[0] > 0
    return grads


def _same_gradients(with_ds, without):
    # Both round P and dS to bf16 and sum the same products in fp32; delta is summed in another order, which moves single roundings of dS: less
    # than one rounding of the result (2^-9) over a tensor.
    for name, a, b in zip(("dq", "dk", "dv"), with_ds, without):
        a, b = a.float(), b.float()
        assert bool(torch.isfinite(a).all()), name
        assert float((a - b).norm()) <= 2 ** -9 * float(b.norm()), f"{name}: {float((a - b).norm() / b.norm()):.3g}"


@pytest.mark.parametrize("lens_q,lens_k,Hq,Hkv,causal", [
    ([129], [129], 3, 1, True), ([1, 64, 65, 200, 0, 333], None, 6, 2, True), ([300, 31, 1], [130, 64, 200], 4, 4, True),
    ([100, 257, 64, 0], [333, 33, 64, 70], 4, 2, False), ([1500, 40, 700], None, 8, 1, True), ([30 + i for i in range(130)], None, 2, 2, True)])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_backward_with_ds_in_memory_packed(ops, monkeypatch, D, lens_q, lens_k, Hq, Hkv, causal):
    """Packed: ragged row and key tiles, sequences without queries or keys, more queries than keys and the other way round, more sequences
    than lanes, few key tiles (dealt to several workgroups)."""
    _same_gradients(*_both_forms(ops, monkeypatch, lens_q, lens_k or lens_q, Hq, Hkv, causal, True, D=D, spare=5 if D == 128 else 40))


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,causal,f32", [(1, 2, 2, 130, 130, True, True), (3, 8, 2, 200, 333, True, False),
                                                       (2, 4, 4, 257, 96, False, False), (40, 8, 8, 190, 190, True, True), (1, 5, 1, 1025, 1025, False, False)])
@pytest.mark.parametrize("D", [32, 64, 128])
def test_backward_with_ds_in_memory_dense(ops, monkeypatch, D, B, Hq, Hkv, Sq, Sk, causal, f32):
    B = min(B, 12 if D == 32 else 19 if D == 64 else B)               # (what the form is chosen for)
    Sq, Sk = (Sq + 130, Sk + 130) if D < 128 and Hq == Hkv and max(Sq, Sk) <= 256 else (Sq, Sk)
    _same_gradients(*_both_forms(ops, monkeypatch, [Sq] * B, [Sk] * B, Hq, Hkv, causal, False, f32=f32, D=D))


@pytest.mark.parametrize("packed", [True, False])
def test_backward_with_ds_in_memory_in_passes(ops, monkeypatch, packed):
    """A workspace for a part of the kv heads: several passes over it, the last one smaller."""
    _same_gradients(*_both_forms(ops, monkeypatch, [420] * 3, [420] * 3, 28, 14, True, packed, workspace_part=0.45))


@pytest.mark.parametrize("D,B,H,S", [(128, 2, 3, 200), (64, 2, 3, 300), (32, 2, 3, 300), (64, 26, 16, 200), (32, 1, 3, 200)])
def test_backward_of_a_key_whose_dp_overflows_in_rows_that_do_not_see_it(ops, D, B, H, S):
    """dO . v of a key behind the diagonal is beyond fp32 (1e15 * 1e25 * D): nothing that a row's dQ adds.  With dS in memory and in
    the kernel of short heads (200 tokens), where dK has nothing of it either."""
    print(f"case: unseen overflow D={D} {B}x{H} {S}", flush=True)
    at = 150
    q, k, v, dout = (rnd(B, H, S, D, seed=440 + i) for i in range(4))
    v[:, :, at] *= 1e25
    dout[:, :, :at] *= 1e15
    dout[:, :, at:] *= 1e-25
    leaves = [t.cuda().requires_grad_() for t in (q, k, v)]
    grads = torch.autograd.grad(ops.flash_attn_prefill(*leaves, causal=True), leaves, dout.cuda())
    wide = [t[:1].double().requires_grad_() for t in (q, k, v)]
    scores = (wide[0] @ wide[1].transpose(-1, -2) / D ** 0.5).masked_fill(~torch.ones(S, S, dtype=torch.bool).tril(), -float("inf"))
    want = torch.autograd.grad(torch.softmax(scores, -1) @ wide[2], wide, dout[:1].double())
    for name, got, ref in zip(("dq", "dk", "dv"), grads, want):
        if name == "dk" and (D == 128 or S > 256):                  # (there such a key's dK is NaN)
            continue
        assert bool(torch.isfinite(got).all()), name
        for part in (slice(0, at), slice(at, at + 1), slice(at + 1, S)):                    # (sizes of their own)
            size = ref[:, :, part].abs().max()
            check_grad(name, got[:1, :, part].double().cpu() / size, ref[:, :, part] / size)


def _packed_gradients(ops, lens_q, lens_k, max_q, max_k, causal):
    cu_q = torch.tensor([0] + torch.tensor(lens_q).cumsum(0).tolist(), dtype=torch.int32).cuda()
    cu_k = cu_q if lens_k is None else torch.tensor([0] + torch.tensor(lens_k).cumsum(0).tolist(), dtype=torch.int32).cuda()
    Tq, Tk = sum(lens_q), sum(lens_k or lens_q)
    leaves = [rnd(T, H, 128, seed=430 + i, scale=0.5).cuda().requires_grad_() for i, (T, H) in enumerate(((Tq, 4), (Tk, 2), (Tk, 2)))]
    out = ops.flash_attn_varlen_prefill(*leaves, cu_q, cu_k, max_q, max_k, causal=causal)
    return torch.autograd.grad(out, leaves, rnd(Tq, 4, 128, seed=433, scale=0.5).cuda())


@pytest.mark.parametrize("lens_q,lens_k,max_q,max_k,causal", [
    ([420, 100], None, 320, 420, True), ([420, 100], None, 420, 300, True), ([420, 100], None, 260, 257, False), ([512, 512, 512], None, 257, 257, True),
    ([300, 200], [500, 333], 260, 500, True), ([300, 200], [500, 333], 300, 460, False)])
def test_backward_with_ds_in_memory_promises_that_are_too_small(ops, lens_q, lens_k, max_q, max_k, causal):
    """Sequences longer than max_seqlen_*, up to its next multiple of 256: the gradients of the right promise, all rows of them."""
    print(f"case: short promises {lens_q} {lens_k} {max_q} {max_k} {causal}", flush=True)
    torch.full((1 << 26,), float("nan"), device="cuda")              # (what is not written shows)
    short = _packed_gradients(ops, lens_q, lens_k, max_q, max_k, causal)
    _same_gradients(short, _packed_gradients(ops, lens_q, lens_k, max(lens_q), max(lens_k or lens_q), causal))


def test_backward_with_ds_in_memory_of_sequences_far_beyond_the_promise(ops):
    """A sequence that dS has no room for gets gradients of zero; one beyond the promise that fits, and those that keep it, get theirs."""
    lens = [700, 30, 500, 200]
    torch.full((1 << 26,), float("nan"), device="cuda")
    got = _packed_gradients(ops, lens, None, 256, 256, True)
    want = [t.clone() for t in _packed_gradients(ops, lens, None, 700, 700, True)]
    for t in want:
        t[:700] = 0
    _same_gradients(got, want)
    assert all(bool((t[:700] == 0).all()) for t in got)


@pytest.mark.parametrize("Sq,Sk", [(1, 1), (31, 33), (64, 64), (65, 40), (128, 129), (129, 256), (256, 255), (256, 256)])
@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("causal", [True, False])
def test_backward_of_short_heads(ops, D, Sq, Sk, causal):
    """Many heads of up to 256 queries and keys, one workgroup each: edges of its blocks of 32 and of its sizes (64, 128, 256 rows), more queries than
    keys (rows without keys add nothing under a causal mask) and the other way round, mixed types, gradients in the layout of their input."""
    print(f"case: backward of short heads {D} {Sq} {Sk} {causal}", flush=True)
    B, H = 13, 16                                                    # (208 heads of up to two key tiles: not a launch of few)
    q, k, dout = rnd(B, H, Sq, D, seed=1), rnd(B, H, Sk, D, seed=2), rnd(B, H, Sq, D, seed=4)
    v = rnd(B, Sk, H, D, seed=3).permute(0, 2, 1, 3)
    first = max(0, Sq - Sk) if causal else 0                        # the first row with a key
    leaves = [q.float().cuda().requires_grad_(), k.cuda().requires_grad_(), v.cuda().requires_grad_()]
    out = ops.flash_attn_prefill(*leaves, causal=causal)
    dq, dk, dv = torch.autograd.grad(out, leaves, dout.cuda())
    assert dq.dtype == torch.float32 and dk.dtype == dv.dtype == torch.bfloat16 and dv.stride() == v.stride()
    for b in (0, B - 1):                                              # (every head is the same work: two sequences of the reference's are enough)
        want = orc.prefill_backward_reference(q[b:b + 1, :, first:], k[b:b + 1], v[b:b + 1], dout[b:b + 1, :, first:], causal=causal)
        check_grad("dq", dq[b:b + 1, :, first:], want[0])
        check_grad("dk", dk[b:b + 1], want[1])
        check_grad("dv", dv[b:b + 1], want[2])
    assert bool((dq[:, :, :first] == 0).all()) and all(bool(torch.isfinite(t).all()) for t in (dq, dk, dv))


@pytest.mark.parametrize("D,B,H,S,causal", [(32, 1, 1, 256, True), (32, 2, 4, 161, True), (64, 1, 3, 200, False), (64, 12, 16, 161, True)])
def test_backward_of_few_short_heads(ops, D, B, H, S, causal):
    """Launches of few workgroups are the short kernel's as well: one sequence and one head, up to one round of the chip."""
    print(f"case: backward of few short heads {D} {B}x{H} {S} {causal}", flush=True)
    run_dense(ops, B, H, H, S, S, D, causal, seed=60 + D)
