"""Short heads of 32, whose workgroups are dealt to the XCDs eight heads at a time: numbers of heads that are no multiple of eight or of eight times eight, grouped heads, several
query tiles, fp32 queries and keys.  Against float64 attention of the bf16 operands: the weights and the result are rounded to bf16, gradients after one product more."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Hkv,Sq,Sk,train,f32", [(1, 1, 1, 33, 33, True, False), (9, 15, 15, 130, 130, True, True), (11, 12, 4, 100, 100, False, False), (4, 16, 16, 256, 256, True, True),
                                                     (3, 24, 24, 64, 64, True, False), (5, 26, 13, 300, 200, False, False)])
def test_short_heads(B, H, Hkv, Sq, Sk, train, f32):
    import mi355_attn as ma
    print(f"case: short heads {B} {H}/{Hkv} {Sq} {Sk} {train} {f32}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(B * H)
    q, k = (torch.randn(B, h, s, 32, generator=g, device="cuda").mul_(0.5).bfloat16() for h, s in ((H, Sq), (Hkv, Sk)))
    v = torch.randn(B, Sk, Hkv, 32, generator=g, device="cuda").mul_(0.5).bfloat16().permute(0, 2, 1, 3)
    dout = torch.randn(B, Sq, H, 32, generator=g, device="cuda").mul_(0.5).bfloat16().permute(0, 2, 1, 3)
    mine = [t.float() if f32 and t is not v else t.detach() for t in (q, k, v)]
    ref = [t.double() for t in (q, k, v)]
    causal = Sq == Sk
    for t in (*mine, *ref):
        t.requires_grad_(train)
    out = ma.flash_attn_prefill(*mine, causal=causal)
    kr, vr = (t.repeat_interleave(H // Hkv, 1) for t in ref[1:])
    s = ref[0] @ kr.transpose(-1, -2) / 32 ** 0.5
    if causal:
        s = s.masked_fill(torch.ones(Sq, Sk, dtype=torch.bool, device="cuda").triu(1), -float("inf"))
    want = torch.softmax(s, -1) @ vr

    def close(got, ref, roundings):
        assert bool(torch.isfinite(got).all())
        assert float((got.double() - ref).norm()) <= roundings * 2 ** -8 * float(ref.norm())

    close(out, want, 2)
    if train:
        for got, ref in zip(torch.autograd.grad(out, mine, dout), torch.autograd.grad(want, ref, dout.double())):
            close(got, ref, 4)
