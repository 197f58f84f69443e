"""Forward tiles of four and of eight wavefronts at the edges of their tiles and of their launches' orders, against fp32 on the host."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ma():
    import mi355_attn
    return mi355_attn


def reference(q, k, v, window, keep):
    """q (n, H, D), k, v (n, Hkv, D), one sequence, causal."""
    n, H, D = q.shape
    k, v = (x.double().repeat_interleave(H // k.shape[1], 1) for x in (k, v))
    s = torch.einsum("qhd,khd->hqk", q.double(), k) * D ** -0.5
    i, j = torch.arange(n)[:, None], torch.arange(n)[None]
    seen = j <= i
    if window:
        seen &= (i - j < window) | (j < keep)
    return torch.einsum("hqk,khd->qhd", torch.softmax(s.masked_fill(~seen, float("-inf")), -1), v)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("H,Hkv,lens,promised", [
    (3, 1, [127, 1, 128, 129], 129),                # fewer than eight kv heads: all of them in front
    (8, 8, [255, 256, 257, 63, 65], 257),
    (4, 2, [33] * 9 + [300, 513], 513),             # whole rounds and some in front
    (16, 4, [700, 31, 385], 300),                   # longer than promised
    (2, 2, [96] * 40 + [1030], 1030)])
@pytest.mark.parametrize("window,keep", [(0, 0), (100, 3), (5000, 0)])
def test_tiles_and_orders(ma, D, H, Hkv, lens, promised, window, keep):
    """Each output is a convex mean of bf16 values: rounding of the weights, in the products and in their sum, and of the result, up to 2^-8 of themselves and half of it on
    average.  As outputs are well below the largest value, 3 * 2^-9 of that holds, with a little for fp32 sums."""
    print(f"case: units {D} {H} {Hkv} {lens} {window}", flush=True)
    g = torch.Generator().manual_seed(D + H)
    T = sum(lens)
    q, k, v = (torch.randn(T, h, D, generator=g).bfloat16() for h in (H, Hkv, Hkv))
    cu = torch.tensor([0] + lens).cumsum(0).int()
    got = ma.flash_attn_varlen_prefill(q.cuda(), k.cuda(), v.cuda(), cu.cuda(), cu.cuda(), promised, promised, window=window, keep_first=keep).cpu()
    for a, n in zip(cu.tolist(), lens):
        ref = reference(q[a:a + n], k[a:a + n], v[a:a + n], window, keep)
        bound = 3.1 * 2 ** -9 * float(v[a:a + n].float().abs().max())
        assert float((got[a:a + n].double() - ref).abs().max()) <= bound, (a, n)


@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("B,H,S,causal", [(1, 3, 700, False), (2, 9, 130, False), (1, 17, 1025, True), (260, 16, 384, True), (1, 1100, 640, True)])
def test_dense_launches_of_every_size(ma, D, B, H, S, causal):
    """All workgroups resident at once, more of them, and the pairs of launches beyond four rounds of the chip; a few heads are looked at (eight wavefronts and each kernel by
    name: test_gpu_prefill_kernels.py)."""
    print(f"case: dense units {D} {B} {H} {S}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(S)
    q, k, v = (torch.randn(B, H, S, D, generator=g, device="cuda", dtype=torch.bfloat16) for _ in range(3))
    out = ma.flash_attn_prefill(q, k, v, causal=causal)
    assert bool(torch.isfinite(out).all())
    for b, h in {(0, 0), (B - 1, H - 1), (B // 2, H // 2), (0, H - 1), (B - 1, 0)}:
        s = q[b, h].double() @ k[b, h].double().T * D ** -0.5
        if causal:
            s = s.masked_fill(torch.ones(S, S, device="cuda", dtype=torch.bool).triu(1), float("-inf"))
        ref = torch.softmax(s, -1) @ v[b, h].double()
        assert float((out[b, h].double() - ref).abs().max()) <= 3.1 * 2 ** -9 * float(v[b, h].float().abs().max()), (b, h)


@pytest.mark.parametrize("D", [32, 64])
@pytest.mark.parametrize("H,Hkv,lens,promised", [
    (9, 9, [127, 300, 129, 1, 513, 64] * 5, 513),   # more than one round of single tiles, some in front
    (2, 1, [700, 31] * 9, 700),
    (6, 3, [385, 1030, 255, 257, 1500] * 8, 1500),
    (40, 40, [640], 640), (600, 600, [512], 512),   # equal pairs
    (12, 12, [900, 200, 130, 600] * 4, 700)])       # longer than promised
def test_gradients_of_dealt_tiles(ma, monkeypatch, D, H, Hkv, lens, promised):
    """Without dS in memory.  Rounding of P, dS and the results to bf16 moves each gradient by up to 2^-9 of its terms three times; over a tensor these average, and
    2^-7 of its norm leaves room for sums that cancel."""
    from mi355_attn import _lib, ops
    print(f"case: dealt gradients {D} {H} {Hkv} {lens[:6]} x{len(lens)}", flush=True)
    monkeypatch.setattr(_lib.load(), "mi355_prefill_bwd_ds_workspace", lambda *a: 0)
    g = torch.Generator(device="cuda").manual_seed(D + H)
    T = sum(lens)
    q, k, v, dout = (torch.randn(T, h, D, generator=g, device="cuda", dtype=torch.bfloat16) * 0.5 for h in (H, Hkv, Hkv, H))
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    out, lse = ops._varlen(q, k, v, cu, cu, promised, promised, True, None, want_lse=True)
    got = ops._prefill_backward(q, k, v, out, dout, lse, cu, cu, promised, promised, D ** -0.5, _lib.MASK_CAUSAL)
    torch.cuda.synchronize()
    a = 0
    for n in lens[:6]:
        for h in {0, H // 2, H - 1} if H == Hkv else {0, H - H // Hkv}:
            hk, G = h // (H // Hkv), H // Hkv
            heads = range(hk * G, hk * G + G)
            leaves = [t[a:a + n, i].double().cpu().requires_grad_() for t, i in [(q, j) for j in heads] + [(k, hk), (v, hk)]]
            loss = 0.0
            for qh, i in zip(leaves[:-2], heads):
                sc = (qh @ leaves[-2].T * D ** -0.5).masked_fill(torch.ones(n, n, dtype=torch.bool).triu(1), float("-inf"))
                loss = loss + (torch.softmax(sc, -1) @ leaves[-1] * dout[a:a + n, i].double().cpu()).sum()
            want = torch.autograd.grad(loss, leaves)
            mine = [got[0][a:a + n, i] for i in heads] + [got[1][a:a + n, hk], got[2][a:a + n, hk]]
            for x, y in zip(mine, want):
                # (a single key has no gradient but what rounding leaves)
                assert float((x.double().cpu() - y).norm()) <= 2 ** -7 * float(y.norm()) + (1e-2 if n == 1 else 0.0), (a, n, h)
        a += n


@pytest.mark.parametrize("window", [0, 150])
@pytest.mark.parametrize("S", [64, 300, 700])
def test_values_beyond_2_to_the_94_under_high_scores(ma, S, window):
    """Heads of 128 on four wavefronts, every weight 2^24 times that of a score of 0: rows stay the means of their values, of which each column has equal
    ones (S of 64: inside the last three key tiles, whose references follow the scores; 300 and 700: in front of them too)."""
    import ctypes
    from mi355_attn import _lib
    D, H, B, waves = 128, 4, {64: 200, 300: 60, 700: 20}[S], ctypes.c_int(0)
    kernel = _lib.load().mi355_prefill_kernel(B, H, H, D, S, S, 1, window, 0, 0, 1, window, 0, ctypes.byref(waves))
    assert (kernel, waves.value) == (1, 4)
    print(f"case: values of 2^120 {S} {window}", flush=True)
    q = torch.zeros(B, H, S, D, device="cuda", dtype=torch.bfloat16)
    k = torch.randn(B, H, S, D, device="cuda", generator=torch.Generator(device="cuda").manual_seed(S)).bfloat16()
    q[..., 0], k[..., 0] = 13.75, 13.6875                 # 24 = 13.75 * 13.6875 / sqrt(128) * log2(e)
    v = (torch.linspace(-1, 1, D, device="cuda") * 2.0 ** 120).bfloat16().expand(B, H, S, D).contiguous()
    cu = (torch.arange(B + 1, device="cuda") * S).int()
    rows = [x.transpose(1, 2).reshape(B * S, H, D) for x in (q, k, v)]
    outs = [ma.flash_attn_varlen_prefill(*rows, cu, cu, S, S, window=window).view(B, S, H, D).transpose(1, 2)] if window else [ma.flash_attn_prefill(q, k, v, causal=True)]
    for got in outs:
        assert bool(((got.double() - v.double()).abs() <= 2.0 ** -8 * v.double().abs()).all())
