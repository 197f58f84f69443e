"""The operators' native calls (csrc/calls.cpp) against ops.py alone: the same arguments have to reach the same kernels, so results are
equal bit for bit.  Every case runs with the native module and without it; `taken` says whether the native call is meant to do it."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF, F32 = torch.bfloat16, torch.float32


@pytest.fixture(scope="module")
def ma():
    import mi355_attn
    mi355_attn.load()
    return mi355_attn


class _Seen:
    """The native module, noting which calls it did."""

    def __init__(self, module):
        self.module, self.done = module, []

    def __getattr__(self, name):
        def call(*a):
            out = getattr(self.module, name)(*a)
            self.done.append(out is not None)
            return out
        return call


def rnd(*shape, seed, dtype=BF, std=0.5):
    return (torch.randn(*shape, generator=torch.Generator().manual_seed(seed)) * std).to(dtype).cuda()


def flat(x):
    if isinstance(x, torch.Tensor):
        return [x.detach()]
    return [] if x is None else [t for y in x for t in flat(y)]


def both(monkeypatch, fn, taken, what):
    """fn() with the native module and without it, and whether the first call in it was native."""
    from mi355_attn import ops
    print(f"case: {what}", flush=True)
    seen = _Seen(ops._native)
    assert seen.module is not None, "the native module is not built"
    monkeypatch.setattr(ops, "_native", seen)
    a = flat(fn())
    assert seen.done[0] == taken, what
    monkeypatch.setattr(ops, "_native", None)
    b = flat(fn())
    torch.cuda.synchronize()
    monkeypatch.undo()
    assert len(a) == len(b)
    for i, (x, y) in enumerate(zip(a, b)):
        assert x.shape == y.shape and x.dtype == y.dtype and x.stride() == y.stride(), (what, i)
        assert torch.equal(x.reshape(-1).contiguous().view(torch.uint8), y.reshape(-1).contiguous().view(torch.uint8)), (what, i)


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,D,types,grad,causal", [
    (2, 4, 2, 50, 50, 64, (BF, BF, BF), False, True), (2, 4, 4, 300, 300, 32, (F32, F32, BF), True, True), (1, 3, 1, 65, 130, 128, (BF, F32, BF), True, False),
    (1, 2, 2, 7, 2100, 128, (BF, BF, BF), False, True), (2, 2, 2, 129, 129, 128, (BF, BF, BF), True, True), (3, 4, 4, 200, 200, 32, (F32, F32, BF), True, True),
    (2, 3, 3, 65, 256, 64, (BF, F32, BF), True, True), (2, 2, 2, 256, 33, 32, (F32, BF, F32), True, False), (1, 2, 2, 1, 1, 64, (F32, F32, BF), True, True),
    (1, 2, 1, 40, 40, 64, (F32, F32, F32), True, True)])
def test_dense(ma, monkeypatch, B, Hq, Hkv, Sq, Sk, D, types, grad, causal):
    q, k = rnd(B, Hq, Sq, D, seed=1, dtype=types[0]), rnd(B, Hkv, Sk, D, seed=2, dtype=types[1])
    for form in ("rows of a projection", "contiguous", "misaligned", "broadcast"):
        v = rnd(B, Sk, Hkv, D, seed=3, dtype=types[2]).permute(0, 2, 1, 3)
        if form == "contiguous":
            v = v.contiguous()
        elif form == "misaligned":
            v = rnd(B, Hkv, Sk, D + 1, seed=3, dtype=types[2])[..., 1:]
        kk = k[:, :1].expand(k.shape) if form == "broadcast" else k
        dout = rnd(B, Hq, Sq, D, seed=4)

        def call():
            ins = [t.detach().requires_grad_(grad) for t in (q, kk, v)]
            out = ma.flash_attn_prefill(*ins, causal=causal)
            return (out, *torch.autograd.grad(out, ins, dout.to(out.dtype))) if grad else out
        both(monkeypatch, call, types != (F32,) * 3 and not (form == "broadcast" and types[1] == F32 and Hkv > 1), f"{form} {B} {Hq} {Sq} {Sk} {D} {types}")


@pytest.mark.parametrize("which", [0, 1, 2])
def test_dense_float32_rows_far_apart(ma, which):
    """Rows of 2^24 elements and more: the rounding forward does not take them, the conversion in front of the general one brings them together."""
    t = [rnd(1, 2, 3, 32, seed=50 + i, dtype=F32 if i == which else BF) for i in range(3)]
    far = torch.empty_strided((1, 2, 3, 32), (64, 32, 1 << 24, 1), dtype=F32, device="cuda")
    far.copy_(t[which])
    g = rnd(1, 2, 3, 32, seed=54)

    def run(x):
        leaves = [t[i] if i != which else x for i in range(3)]
        leaves = [y.detach().requires_grad_() for y in leaves]
        out = ma.flash_attn_prefill(*leaves, causal=True)
        return [out, *torch.autograd.grad(out, leaves, g)]

    for a, b in zip(run(far), run(t[which])):
        assert torch.equal(a, b)


@pytest.mark.parametrize("lens,Hq,Hkv,D,grad,causal,window", [
    ([1, 64, 0, 200], 4, 2, 64, False, True, 0), ([300, 31, 1], 4, 4, 128, True, True, 0), ([130, 40], 2, 1, 32, True, False, 0), ([70, 900], 2, 1, 128, False, True, 64)])
def test_packed(ma, monkeypatch, lens, Hq, Hkv, D, grad, causal, window):
    T = sum(lens)
    qkv = rnd(T, Hq + 2 * Hkv, D, seed=1)
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32).cuda()
    dout = rnd(T, Hq, D, seed=4)

    def call(**kw):
        ins = [t.detach().requires_grad_(grad) for t in (qkv[:, :Hq], qkv[:, Hq:Hq + Hkv], qkv[:, Hq + Hkv:])]
        out = ma.flash_attn_varlen_prefill(*ins, cu, kw.pop("cu_k", cu), max(lens), max(lens), causal=causal, window=window, keep_first=4 if window else 0, **kw)
        return (out, *torch.autograd.grad(out, ins, dout)) if grad else out
    both(monkeypatch, call, True, f"packed {lens}")
    both(monkeypatch, lambda: call(cu_k=cu.clone()), True, f"packed, two arrays {lens}")


def test_autograd_sees_what_it_saw(ma, monkeypatch):
    """Saved-tensor hooks, an input changed behind the forward, a second backward, a graph of the backward, another stream, no_grad."""
    q, k, v, dout = (rnd(1, 2, 70, 64, seed=i) for i in range(4))
    leaves = [t.requires_grad_() for t in (q, k, v)]

    def hooked():
        packed = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(t.detach().clone()) or t.cpu(), lambda t: t.cuda()):
            out = ma.sdpa_slot(*leaves)
        return (*packed, *torch.autograd.grad(out, leaves, dout))
    both(monkeypatch, hooked, True, "saved-tensor hooks")

    def with_graph():
        out = ma.sdpa_slot(*leaves)
        g = torch.autograd.grad(out, leaves, dout.clone().requires_grad_(), create_graph=True)
        return out, *g
    both(monkeypatch, with_graph, True, "create_graph")

    def streamed():
        s = torch.cuda.Stream()
        s.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(s):
            out = ma.sdpa_slot(*leaves)
        torch.cuda.current_stream().wait_stream(s)
        g = torch.autograd.grad(out, leaves, dout)
        torch.cuda.synchronize()
        return out, *g
    both(monkeypatch, streamed, True, "another stream")
    with torch.no_grad():
        both(monkeypatch, lambda: ma.sdpa_slot(*leaves), True, "no_grad")
    from mi355_attn import ops
    for native in (ops._native, None):
        monkeypatch.setattr(ops, "_native", native)
        out = ma.sdpa_slot(*leaves)
        torch.autograd.grad(out, leaves, dout)
        with pytest.raises(RuntimeError, match="second time"):
            torch.autograd.grad(out, leaves, dout)
        with torch.no_grad():
            w = leaves[0].clone()
        out = ma.sdpa_slot(w.requires_grad_(), *leaves[1:])
        with torch.no_grad():
            w.add_(1)
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            out.backward(dout)
        import torch.autograd.forward_ad as fwad
        with fwad.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
            ma.sdpa_slot(fwad.make_dual(leaves[0], dout), *leaves[1:])
        with pytest.raises(RuntimeError):
            torch.func.vmap(lambda a: ma.sdpa_slot(a, *leaves[1:]))(leaves[0][None])
        monkeypatch.undo()


@pytest.mark.filterwarnings("ignore")
def test_a_trace_records_the_call(ma):
    """What torch.jit.trace records is called again with other inputs: its results are theirs, not the traced ones."""
    q, k, v = (rnd(1, 2, 70, 64, seed=i).requires_grad_() for i in range(3))
    traced = torch.jit.trace(lambda a, b, c: ma.sdpa_slot(a, b, c), (q, k, v), check_trace=False)
    for seed in (3, 4):
        other = [rnd(1, 2, 70, 64, seed=seed + i).requires_grad_() for i in range(3)]
        assert torch.equal(traced(*other), ma.sdpa_slot(*other)), seed


def test_forms_that_are_left_to_python(ma, monkeypatch):
    """A tensor subclass, a mode that sees operators, wrong arguments: the same result or the same error as without the native module."""
    from mi355_attn import ops
    from torch.utils._python_dispatch import TorchDispatchMode

    class Sub(torch.Tensor):
        pass

    class Watch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))
    q = rnd(1, 2, 40, 64, seed=1)
    both(monkeypatch, lambda: ma.sdpa_slot(q.as_subclass(Sub), q, q).as_subclass(torch.Tensor), False, "subclass")
    with Watch():
        both(monkeypatch, lambda: ma.sdpa_slot(q, q, q), False, "dispatch mode")
    cu = torch.tensor([0, 40], dtype=torch.int32).cuda()
    p = q[0].transpose(0, 1).contiguous()
    kc = rnd(4, 2, 16, 64, seed=2)
    bt, cl = torch.zeros(1, 4, dtype=torch.int32).cuda(), torch.full((1,), 20, dtype=torch.int32).cuda()
    wrong = [
        lambda: ma.sdpa_slot(q, q[..., :32], q), lambda: ma.sdpa_slot(q.half(), q, q), lambda: ma.sdpa_slot(q.cpu(), q, q), lambda: ma.sdpa_slot(q[0], q, q),
        lambda: ma.sdpa_slot(rnd(1, 2, 40, 48, seed=1), *[rnd(1, 2, 40, 48, seed=1)] * 2), lambda: ma.sdpa_slot(q, q[:, :1], q),
        lambda: ma.flash_attn_varlen_prefill(p, p, p, cu.long(), cu, 40, 40), lambda: ma.flash_attn_varlen_prefill(p, p, p, cu, cu, 0, 40),
        lambda: ma.flash_attn_varlen_prefill(p, p, p, cu, cu, 40, 40, causal=False, window=8),
        lambda: ma.paged_attention_decode(p[:1], kc, kc, bt, cl, max_context=100), lambda: ma.paged_attention_decode(p[:1], kc, kc, bt.long(), cl),
        lambda: ma.paged_attention_decode(p[:1], kc, kc, bt, cl, k_scale=torch.ones(4, 2).cuda()),
        lambda: ma.paged_attention_decode(p[:1], kc, kc, bt, cl, workspace=torch.empty(16, dtype=torch.uint8).cuda(), softmax_scale="x"),
        lambda: ma.flash_attn_paged_prefill(p, kc, kc, cu, bt, cl, 0), lambda: ma.flash_attn_paged_prefill(p, kc[:, :0], kc[:, :0], cu, bt, cl, 40),
        lambda: ma.moe_route(p[:, 0], p[:, 0], torch.zeros(40).cuda(), 41),
        lambda: ma.moe_route(p[:, 0, :60], p[:3, 0, :60], torch.zeros(3).cuda(), 2), lambda: ma.gated_norm(p[:, 0], p[:, 0], torch.ones(64).cuda(), 3, 1e-6)]
    for i, f in enumerate(wrong):
        print(f"case: wrong {i}", flush=True)
        errors = []
        for native in (ops._native, None):
            monkeypatch.setattr(ops, "_native", native)
            with pytest.raises(Exception) as e:
                f()
            errors.append((type(e.value), str(e.value)))
            monkeypatch.undo()
        assert errors[0] == errors[1], i


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("Hq,Hkv,D", [(4, 2, 64), (8, 1, 128)])
def test_paged(ma, monkeypatch, Hq, Hkv, D, fp8):
    """Rotation and cache write, portions over the cache, decode steps; with and without a window, a workspace, bounds."""
    B, n, before = 3, 33, [16, 64, 0]
    total = [b + n for b in before]
    tables = torch.arange(B * 7, dtype=torch.int32).view(B, 7).cuda()
    slots = torch.cat([int(tables[i, 0]) * 16 + torch.arange(b, b + n) for i, b in enumerate(before)]).cuda()
    pos = torch.cat([torch.arange(b, b + n) for b in before]).int().cuda()
    lens, cu = torch.tensor(total, dtype=torch.int32).cuda(), (torch.arange(B + 1) * n).int().cuda()
    cu_k = torch.tensor([0] + torch.tensor(total).cumsum(0).tolist(), dtype=torch.int32).cuda()
    qkv = rnd(B * n, Hq + 2 * Hkv, D, seed=1)
    q, k, v = qkv[:, :Hq], qkv[:, Hq:Hq + Hkv], qkv[:, Hq + Hkv:]
    freq = ma.build_rope_cache(128, D, device="cuda:0")

    def pools():
        if not fp8:
            return [rnd(B * 7, Hkv, 16, D, seed=s) for s in (2, 3)], [None, None]
        return [torch.randint(0, 100, (B * 7, Hkv, 16, D), generator=torch.Generator().manual_seed(s)).to(torch.uint8).cuda() for s in (2, 3)], \
            [rnd(B * 7, Hkv, seed=s, dtype=F32).abs() + 0.1 for s in (4, 5)]

    def write(**kw):
        (kc, vc), (ks, vs) = pools()
        got = ma.rope_and_cache_fp8(q, k, v, pos, freq, kc, vc, ks, vs, slots, **kw) if fp8 else ma.rope_and_cache(q, k, v, pos, freq, kc, vc, slots, **kw)
        return got, kc, vc, ks, vs
    both(monkeypatch, write, True, "write")
    both(monkeypatch, lambda: write(k_out=True), True, "write, k_out")
    _, kc, vc, ks, vs = write()
    kw = dict(k_scale=ks, v_scale=vs)

    def portion(**more):
        return ma.flash_attn_paged_prefill(q, kc, vc, cu, tables, lens, n, **kw, **more)
    both(monkeypatch, lambda: portion(max_context=max(total), total_context=sum(total), cu_seqlens_k=cu_k), True, "portion")
    both(monkeypatch, lambda: portion(max_context=max(total), total_context=sum(total), cu_seqlens_k=cu_k, softmax_scale=0.3), True, "portion, scale")
    both(monkeypatch, portion, not fp8, "portion without bounds")
    step = rnd(B, Hq, D, seed=7)
    for more, taken in ((dict(), True), (dict(window=32, keep_first=4), True), (dict(max_context=max(total), softmax_scale=0.2), True),
                        (dict(workspace=ma.paged_decode_workspace(B, Hq, D, 128, step.device)), True)):
        both(monkeypatch, lambda: ma.paged_attention_decode(step, kc, vc, tables, lens, **kw, **more), taken, f"decode {more.keys()}")
    wide = rnd(B, Hq + 1, D, seed=8)[:, 1:]
    both(monkeypatch, lambda: ma.paged_attention_decode(wide, kc, vc, tables, lens, **kw), False, "decode, rows of a wider matrix")


@pytest.mark.parametrize("T,E,top,k,ff,n", [(3, 8, 2, 64, 64, 40), (300, 4, 2, 128, 192, 72)])
def test_experts_and_norms(ma, monkeypatch, T, E, top, k, ff, n):
    h, w, bias = rnd(T, k + 8, seed=1)[:, :k], rnd(E, k, seed=2), rnd(E, seed=3, dtype=F32)
    both(monkeypatch, lambda: ma.moe_route(h, w, bias, top), True, "route")
    ids, wt, _ = ma.moe_route(h, w, bias, top)
    gu, dn = rnd(E, 2 * ff, k, seed=4, std=k ** -0.5), rnd(E, n, ff, seed=5, std=ff ** -0.5)
    both(monkeypatch, lambda: ma.moe_experts(h, ids, wt, gu, dn), True, "experts")
    routed, sub, weight = ma.moe_experts(h, ids, wt, gu, dn), rnd(T, n, seed=6), rnd(n, seed=7, dtype=F32)
    resid = rnd(T, n, seed=8, dtype=F32)
    both(monkeypatch, lambda: ma.residual_rms(resid.clone(), weight, sub=sub, routed=routed, top=top, weight_offset=1.0), True, "sum and norm")
    both(monkeypatch, lambda: ma.residual_rms(None, weight, sub=sub), True, "norm of one")
    x = resid.clone()
    assert ma.residual_rms(x, weight, sub=sub)[0] is x
    z = rnd(T, n + 8, seed=9)[:, :n]
    both(monkeypatch, lambda: ma.gated_norm(sub, z, weight, 2, 1e-6), True, "gated norm")
    y = sub.clone()
    assert ma.gated_norm(y, z, weight, 1, 1e-6, out=y) is y
    both(monkeypatch, lambda: ma.gated_norm(sub.clone(), z, None, 1, 1e-6), False, "gated norm without a weight")


@pytest.mark.parametrize("lens,state,groups", [([5, 70], 64, 1), ([2000], 128, 2), ([1, 9, 3], 20, 1)])
def test_mixer(ma, monkeypatch, lens, state, groups):
    H, P, T, B = 4, 64, sum(lens), len(lens)
    inner, channels = H * P, H * P + 2 * groups * state
    proj = rnd(T, inner + channels + H, seed=1)
    params = dict(conv=rnd(4, channels, seed=2, dtype=F32), conv_b=rnd(channels, seed=3, dtype=F32), dt_bias=rnd(H, seed=4, dtype=F32) - 3,
                  neg_a=-rnd(H, seed=5, dtype=F32).exp(), d_skip=rnd(H, seed=6, dtype=F32))
    cu = torch.tensor([0] + torch.tensor(lens).cumsum(0).tolist(), dtype=torch.int32).cuda()
    pos = torch.cat([torch.arange(m) for m in lens]).int().cuda()
    slots = torch.arange(B).int().cuda()

    def call():
        conv, ssm = torch.zeros(B, 4, channels, dtype=BF).cuda(), torch.zeros(B, H, state, P).cuda()
        y = ma.ssm_mix(proj, inner, inner + channels, params, conv, ssm, slots, pos, cu, heads=H, vdim=P, state=state, groups=groups)
        return y, conv, ssm
    both(monkeypatch, call, True, f"mixer {lens}")


@pytest.mark.parametrize("T", [1, 17, 40])
def test_rows(ma, monkeypatch, T):
    k, n, H, D = 72, 96, 2, 32
    x, w, norm = rnd(50, k + 8, seed=1)[:, :k], rnd(n, k, seed=2, std=k ** -0.5), rnd(k, seed=3, dtype=F32)
    ids, pick = (torch.randint(0, 50, (T,), generator=torch.Generator().manual_seed(s)).cuda() for s in (4, 5))
    for kw in (dict(), dict(norm=norm, out_dtype=F32), dict(resid=rnd(50, n, seed=6), resid_rows=pick), dict(norm=norm, eps=1e-6, gate_up=True),
               dict(resid=rnd(T, n, seed=7))):
        both(monkeypatch, lambda: ma.rows_linear(x, w, x_rows=ids, prompt=T > 32, **kw), True, f"rows_linear {list(kw)}")
    if T > 32:
        return
    freq, slots, pos = ma.build_rope_cache(64, D, device="cuda:0"), torch.arange(T).cuda(), torch.arange(T).int().cuda()
    wq = rnd(3 * H * D, k, seed=8)

    def qkv():
        kc, vc = torch.zeros(4, H, 16, D, dtype=BF).cuda(), torch.zeros(4, H, 16, D, dtype=BF).cuda()
        return ma.rows_qkv(x, wq, pos, freq, kc, vc, slots, H, norm=norm, x_rows=ids), kc, vc
    both(monkeypatch, qkv, True, "rows_qkv")
