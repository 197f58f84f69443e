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
    """Each output is a convex mean of bf16 values: rounding of the weights (2^-9 each, both in the products and in their sum) and of the result 2^-9 of the largest value, so
    3 * 2^-9 of it together, and a little for fp32 sums."""
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
    """All workgroups resident at once, more of them, and the pairs of launches beyond four rounds of the chip; a few heads are looked at."""
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
