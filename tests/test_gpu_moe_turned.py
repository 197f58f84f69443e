"""Experts' products without an order, of few pairs and over rows of whole 4096 bytes: steps of k that begin elsewhere in every workgroup, few and many pairs per expert (the line between the
two rings on either side, one and two row tiles, more than one pass over the weights), columns that are no whole tile, experts without pairs.  Against float64 products of
the bf16 operands; one rounding of the activation and one of the result, 2^-8 of the norm each at most."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,top,k,ff,n", [(1, 8, 1, 2048, 64, 2048), (5, 8, 2, 2048, 1024, 72), (47, 4, 1, 2048, 192, 2048), (48, 4, 1, 2048, 192, 100), (50, 3, 3, 4096, 128, 36),
                                            (96, 4, 1, 2048, 2048, 2048), (97, 4, 1, 2048, 2048, 40), (300, 6, 2, 2048, 64, 64), (33, 4, 2, 1536, 2048, 96), (127, 8, 1, 1536, 1088, 64),
                                            (128, 8, 1, 1536, 1088, 64)])
def test_direct_products_of_whole_pages(T, E, top, k, ff, n):
    _products(T, E, top, k, ff, n, "direct")


@pytest.mark.parametrize("T,E,top,k,ff,n", [(1, 2, 1, 64, 64, 40), (7, 32, 4, 2048, 128, 64), (16, 80, 4, 128, 64, 36), (21, 80, 3, 512, 192, 2048), (13, 80, 5, 128, 64, 64),
                                            (63, 64, 1, 256, 64, 72), (64, 64, 1, 256, 64, 72)])
def test_fewer_pairs_than_experts(T, E, top, k, ff, n):
    """(workgroups per pair: experts that several pairs name, most of them, up to 64 pairs and fewer than experts, and one more of each)"""
    _products(T, E, top, k, ff, n, "direct")


@pytest.mark.parametrize("T,E,top,k,ff,n", [(1, 2, 1, 2048, 64, 2048), (130, 3, 1, 2048, 2048, 136), (200, 8, 2, 4096, 192, 2048), (513, 2, 1, 2048, 128, 128), (512, 2, 1, 2048, 2048, 96), (192, 2, 1, 4096, 128, 72),
                                            (193, 2, 1, 4096, 128, 72)])
def test_large_tiles_of_whole_pages(T, E, top, k, ff, n):
    """(128 x 128 tiles, up to 256 pairs an expert and one more, 96 with longer rows)"""
    _products(T, E, top, k, ff, n, "large")


@pytest.mark.parametrize("tiling,T,E,top,k,ff,n", [("direct", 32, 33, 1, 2048, 960, 72), ("direct", 15, 40, 2, 64, 2048, 2000), ("direct", 70, 4, 2, 2048, 192, 72), ("large", 400, 2, 1, 2048, 2048, 136),
                                                   ("large", 700, 3, 1, 4096, 192, 2048)])
def test_a_tokens_result_does_not_depend_on_its_place(tiling, T, E, top, k, ff, n):
    """The same tokens in another order, so that a token's pair, row tile and workgroup are others: the same bits."""
    import mi355_attn as ma
    print(f"case: place {tiling} {T} {E} {top} {k} {ff} {n}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T)

    def t(*shape, std=1.0):
        return (torch.randn(*shape, generator=g, device="cuda") * std).bfloat16()

    h, up, down = t(T, k), t(E, 2 * ff, k, std=k ** -0.5), t(E, n, ff, std=ff ** -0.5)
    ids = torch.rand(T, E, generator=g, device="cuda").argsort(-1)[:, :top].to(torch.int32).contiguous()
    weights, perm = torch.rand(T, top, generator=g, device="cuda"), torch.randperm(T, generator=g, device="cuda")
    here = ma.moe_experts(h, ids, weights, up, down, tiling=tiling).view(T, top, n)
    there = ma.moe_experts(h[perm], ids[perm], weights[perm], up, down, tiling=tiling).view(T, top, n)
    assert torch.equal(there, here[perm])


def _products(T, E, top, k, ff, n, tiling):
    import mi355_attn as ma
    print(f"case: {tiling} {T} {E} {top} {k} {ff} {n}", flush=True)
    g = torch.Generator().manual_seed(T + E)

    def t(*shape, std=1.0):
        return (torch.randn(*shape, generator=g) * std).to(torch.bfloat16).cuda()

    h, up, down = t(T, k), t(E, 2 * ff, k, std=k ** -0.5), t(E, n, ff, std=ff ** -0.5)
    ids = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(T)]).to(torch.int32).cuda()
    if T > 40:
        ids[:30] = torch.arange(top, dtype=torch.int32)                  # (more rows than one pass takes)
    weights = torch.rand(T, top, generator=g).cuda()
    got = ma.moe_experts(h, ids, weights, up, down, tiling=tiling)
    ref = torch.zeros(T, top, n, dtype=torch.float64, device="cuda")
    for e in range(E):
        t_at, c_at = (ids == e).nonzero(as_tuple=True)
        x = h[t_at].double() @ up[e].double().T
        act = torch.nn.functional.silu(x[:, :ff]) * x[:, ff:]
        ref[t_at, c_at] = weights[t_at, c_at].double()[:, None] * (act @ down[e].double().T)
    got = got.double().view(T, top, n)
    assert bool(torch.isfinite(got).all())
    assert float((got - ref).norm()) <= 2 * 2 ** -8 * float(ref.norm())
