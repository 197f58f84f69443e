"""fp32 operands of a prefill: rounded in one launch (sizes that are no multiple of eight, one to three of them, strided views, views that are not aligned or have gaps), and read as
they are by the kernel of short heads.  Rounding is torch's own, so results are those of the rounded operands."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [(1, 0, 0), (7, 8, 9), (0, 2049, 0), (2048, 0, 5), (100003, 64, 100001)])
def test_round_operands(sizes):
    import mi355_attn as ma
    print(f"case: round operands {sizes}", flush=True)
    lib = ma.load()
    x = [torch.randn(max(n, 8), device="cuda") * 3 for n in sizes]
    for t in x:
        t[0], t[-1] = float("inf"), 1e-40
    out = [torch.full((max(n, 8) + 8,), -1.0, dtype=torch.bfloat16, device="cuda") for n in sizes]
    in_p = (ctypes.c_void_p * 3)(*[t.data_ptr() if n else None for t, n in zip(x, sizes)])
    out_p = (ctypes.c_void_p * 3)(*[t.data_ptr() if n else None for t, n in zip(out, sizes)])
    assert lib.mi355_round_operands(in_p, out_p, (ctypes.c_int64 * 3)(*sizes), torch.cuda.current_stream().cuda_stream) == 0
    for t, o, n in zip(x, out, sizes):
        assert torch.equal(o[:n], t[:n].bfloat16()) and bool((o[n:] == -1).all())
    assert lib.mi355_round_operands(in_p, out_p, (ctypes.c_int64 * 3)(-1, -1, -1), None) < 0


@pytest.mark.parametrize("B,H,Hkv,S,D,f32", [(2, 3, 3, 33, 32, "qk"), (9, 8, 8, 256, 32, "kv"), (3, 4, 4, 100, 64, "qk"), (2, 4, 2, 100, 64, "qk"), (2, 6, 6, 300, 64, "q"), (1, 4, 4, 177, 128, "qk"),
                                             (1, 2, 2, 70, 128, "kv"), (4, 8, 8, 128, 64, "qk"), (4, 8, 8, 129, 64, "kv"), (3, 11, 11, 256, 64, "qk"), (1, 1, 1, 177, 32, "qk")])
@pytest.mark.parametrize("layout", ["whole", "heads apart", "gap", "odd"])
@pytest.mark.parametrize("train", [False, True])
def test_mixed_operands(B, H, Hkv, S, D, f32, layout, train):
    """Against the same call with operands that torch has rounded; they may take another kernel, so within two roundings of the result."""
    import mi355_attn as ma
    print(f"case: mixed {B} {H}/{Hkv} {S} {D} {f32} {layout} {train}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(S)

    def make(h):
        if layout == "heads apart":
            return torch.randn(B, S, h, D, generator=g, device="cuda").permute(0, 2, 1, 3)
        if layout == "gap":
            return torch.randn(B, h, S, D + 8, generator=g, device="cuda")[..., :D]
        if layout == "odd":                                              # (4 bytes off)
            return torch.randn(B * h * S * D + 1, generator=g, device="cuda")[1:].view(B, h, S, D)
        return torch.randn(B, h, S, D, generator=g, device="cuda")

    q, k, v = make(H), make(Hkv), make(Hkv)
    mixed = [t if name in f32 else t.bfloat16() for name, t in zip("qkv", (q, k, v))]
    ref = [t.bfloat16() for t in mixed]
    for t in (*mixed, *ref):
        t.requires_grad_(train)
    got, want = ma.flash_attn_prefill(*mixed, causal=True), ma.flash_attn_prefill(*ref, causal=True)
    assert got.dtype == torch.bfloat16

    def close(a, b):
        assert float((a.double() - b.double()).norm()) <= 2 * 2 ** -8 * float(b.double().norm())

    close(got, want)
    if train:
        dout = torch.randn(got.shape, generator=g, device="cuda").bfloat16()
        for a, b, t in zip(torch.autograd.grad(got, mixed, dout), torch.autograd.grad(want, ref, dout), mixed):
            assert a.dtype == t.dtype
            close(a, b)


@pytest.mark.parametrize("lens,H,Hkv,D,f32", [([33, 1, 200], 4, 2, 128, "qk"), ([100, 64], 3, 3, 64, "q"), ([257, 30], 2, 1, 32, "kv")])
@pytest.mark.parametrize("layout", ["whole", "sliced"])
@pytest.mark.parametrize("train", [False, True])
def test_mixed_packed_operands(lens, H, Hkv, D, f32, layout, train):
    """Packed sequences, operands of their own or slices of one projection (not whole memory: torch's conversion): the kernels of the rounded operands, so the same bits."""
    import mi355_attn as ma
    print(f"case: mixed packed {lens} {H}/{Hkv} {D} {f32} {layout} {train}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(sum(lens))
    T, cu = sum(lens), torch.tensor([0, *torch.tensor(lens).cumsum(0).tolist()], dtype=torch.int32, device="cuda")
    if layout == "sliced":
        x = torch.randn(T, H + 2 * Hkv, D, generator=g, device="cuda")
        q, k, v = x[:, :H], x[:, H:H + Hkv], x[:, H + Hkv:]
    else:
        q, k, v = (torch.randn(T, h, D, generator=g, device="cuda") for h in (H, Hkv, Hkv))
    mixed = [t.detach() if name in f32 else t.bfloat16() for name, t in zip("qkv", (q, k, v))]
    ref = [t.bfloat16() for t in mixed]
    for t in (*mixed, *ref):
        t.requires_grad_(train)
    got, want = (ma.flash_attn_varlen_prefill(*t, cu, cu, max(lens), max(lens)) for t in (mixed, ref))
    assert torch.equal(got, want)
    if train:
        dout = torch.randn(got.shape, generator=g, device="cuda").bfloat16()
        for a, b, t in zip(torch.autograd.grad(got, mixed, dout), torch.autograd.grad(want, ref, dout), mixed):
            assert a.dtype == t.dtype and torch.equal(a.bfloat16(), b)
