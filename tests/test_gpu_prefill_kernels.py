"""Every kernel of a prefill call by its name.  Which one runs is chosen by the sizes that a call promises, so that small sequences under a larger promise
reach each of them: drawn lengths (empty ones, single tokens), heads, more keys than queries, windows, keys whose scores run away by tens to hundreds of
binary orders in both directions, and the log-sum-exp.

Bounds, against 64 bits.  Scores are sums of D fp32 products, off by up to D 2^-24 of the sum of their parts' sizes; weights are off by that and by the 2^-8 of
rounding to bf16, an output so by as much of the weighted mean of |value - output|, and by 2^-8 of itself.  The log-sum-exp is of weights rounded to bf16: 2^-8
and the scores' error.  1e-5 of the largest value for fp32 sums."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
TILES, W64, SHORT, KEYS = 1, 2, 3, 4
NAMES = {TILES: "tiles", W64: "w64", SHORT: "short", KEYS: "keys"}
KERNELS = [(D, kernel, waves) for D in (32, 64, 128) for kernel, waves in ((TILES, 4), (W64, 4), (KEYS, 4), (KEYS, 8)) if D == 128 or kernel != W64]


@pytest.fixture(scope="module")
def ma():
    import mi355_attn
    return mi355_attn


def named(B, Hq, Hkv, D, Sq, Sk, mask, packed=0, blocks=0, lse=0, window=0, n_cu=0):
    from mi355_attn import _lib
    waves = ctypes.c_int(0)
    return _lib.load().mi355_prefill_kernel(B, Hq, Hkv, D, Sq, Sk, mask, packed, blocks, lse, 1, window, n_cu, ctypes.byref(waves)), waves.value


def promise(want, B, Hq, Hkv, D, rows, keys, mask, window=0, n_cu=0):
    """The smallest lengths promised to a packed call, beside the real ones or above, that its kernel takes"""
    for more in (1, 1.5, 2, 3, 5, 8, 12, 20, 40, 80, 160, 0.3):
        for of_keys in (1, 4, 0.25):
            sq, sk = max(1, int(rows * more)), max(1, int(keys * more * of_keys))
            if all(named(B, Hq, Hkv, D, sq, sk, mask, 1, 0, lse, window, n_cu) == want for lse in (0, 1)):
                return sq, sk


def taken(draw, reach):
    """The first drawn shape for which there is a promise, and that"""
    for _ in range(100):
        shape = draw()
        most = reach(*shape)
        if most:
            return shape, most
    raise AssertionError("no drawn shape reaches the kernel")


def number(g, low, high):
    return int(torch.randint(low, high + 1, (1,), generator=g))


def one_of(g, values):
    return values[number(g, 0, len(values) - 1)]


def run_away(k, g, at_most=5):
    """k (keys, ...): runs of keys whose scores leave the others far behind, in either direction"""
    for _ in range(number(g, 1, at_most)):
        j = number(g, 0, k.shape[0] - 1)
        k[j:j + number(g, 1, 70)] *= one_of(g, [6.0, 20.0, -15.0, 45.0])


def look(what, got, lse, q, k, v, causal, window=0, keep=0):
    """got (n, H, D), lse (H, n) or None; q (n, H, D); k, v (m, Hkv, D): the queries are the last n of the m positions"""
    (n, H, D), m, G = q.shape, k.shape[0], q.shape[1] // k.shape[1]
    i, j = torch.arange(n, device=q.device)[:, None] + (m - n), torch.arange(m, device=q.device)[None]
    seen = torch.ones(n, m, dtype=torch.bool, device=q.device)
    if causal:
        seen = j <= i
    if window:
        seen &= (i - j < window) | (j < keep)
    for h in range(H):
        qh, kh, vh = q[:, h].double(), k[:, h // G].double(), v[:, h // G].double()
        s = (qh @ kh.T * D ** -0.5).masked_fill(~seen, -float("inf"))
        size = (qh.abs() @ kh.abs().T * D ** -0.5).masked_fill(~seen, 0.0).amax(-1)
        off = D * 2.0 ** -24 * size
        p = torch.softmax(s, -1)
        want = p @ vh
        bound = 2.0 ** -8 * want.abs() + (2.0 ** -8 + 2 * off[:, None]) * (p @ vh.abs() + want.abs()) + 1e-5 * vh.abs().max()
        err = (got[:, h].double() - want).abs()
        assert bool((err <= bound).all()), (what, h, float((err - bound).max()))
        if lse is not None:
            assert bool(((lse[h].double() - torch.logsumexp(s, -1)).abs() <= 2.0 ** -8 + 1e-5 + off).all()), (what, h, "lse")


def packed_shape(g, longer):
    lens = [number(g, 1, 600) for _ in range(number(g, 1, 6))] + [1, 0]
    Hkv = number(g, 1, 4)
    return lens, [n + (number(g, 0, longer) if n else 0) for n in lens], Hkv * one_of(g, [1, 2, 3, 4, 8]), Hkv


@pytest.mark.parametrize("D,kernel,waves", KERNELS, ids=lambda x: str(x))
@pytest.mark.parametrize("seed", [0, 1, 2])
def test_packed_calls(ma, D, kernel, waves, seed):
    from mi355_attn import _lib, ops
    g = torch.Generator().manual_seed(100 * D + 10 * kernel + seed)
    for case in range(4):
        causal = case != 2
        mask = _lib.MASK_CAUSAL if causal else _lib.MASK_NONE
        window, keep = (number(g, 1, 400), number(g, 0, 5)) if kernel == TILES and case == 3 else (0, 0)
        (rows, keys, Hq, Hkv), most = taken(lambda: packed_shape(g, 0 if case % 2 else 300), lambda rows, keys, Hq, Hkv: promise(
            (kernel, waves), len(rows), Hq, Hkv, D, max(rows), max(keys), mask, window))
        print(f"case: {NAMES[kernel]} {waves} D={D} #{case} {Hq}/{Hkv} {rows} {keys} {causal} {window} promised {most}", flush=True)
        q, k, v = (torch.randn(n, h, D, generator=g) for n, h in ((sum(rows), Hq), (sum(keys), Hkv), (sum(keys), Hkv)))
        if case:
            run_away(k, g)
        q, k, v = (x.bfloat16().cuda() for x in (q, k, v))
        cq, ck = (torch.tensor([0] + n).cumsum(0).int() for n in (rows, keys))
        given = (q, k, v, cq.cuda(), ck.cuda(), *most)
        got = ma.flash_attn_varlen_prefill(*given, causal=causal, kv_splits=1, window=window, keep_first=keep)
        lse = None
        if not window:
            again, lse = ops._varlen(*given, causal, None, want_lse=True)
            assert torch.equal(again, got)
        for a, n, b, m in zip(cq.tolist(), rows, ck.tolist(), keys):
            if n:
                look((case, n, m), got[a:a + n], None if lse is None else lse[:, a:a + n], q[a:a + n], k[b:b + m], v[b:b + m], causal, window, keep)


@pytest.mark.parametrize("D,kernel,waves", KERNELS + [(32, TILES, 8), (64, TILES, 8)], ids=lambda x: str(x))
@pytest.mark.parametrize("seed", [0, 1])
def test_paged_calls(ma, D, kernel, waves, seed):
    """Block tables wider than any context are what is promised here; behind the contexts they hold ids of no block, and the blocks behind the contexts NaN."""
    g = torch.Generator().manual_seed(100 * D + 10 * kernel + waves + seed)
    for case in range(3):
        longer = 9000 if case == 2 and (kernel, waves) != (TILES, 4) else 900             # (several windows of block ids, where the kernel takes such)
        (rows, keys, Hq, Hkv), (width, most) = taken(lambda: packed_shape(g, longer), lambda rows, keys, Hq, Hkv: paged_promise(
            (kernel, waves), len(rows), Hq, Hkv, D, max(rows), (max(keys) + 15) // 16))
        keys = [max(1, m) for m in keys]
        blocks = [(m + 15) // 16 for m in keys]
        print(f"case: paged {NAMES[kernel]} {waves} D={D} #{case} {Hq}/{Hkv} {rows} {keys} promised {most}, {width} blocks", flush=True)
        q = torch.randn(sum(rows), Hq, D, generator=g).bfloat16().cuda()
        pool = sum(blocks) + 3
        kc, vc = (torch.full((pool, Hkv, 16, D), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
        table, ids = torch.full((len(rows), width), 2 ** 30, dtype=torch.int32), torch.randperm(pool, generator=g)
        held = []
        for b, m in enumerate(keys):
            k, v = (torch.randn(m, Hkv, D, generator=g) for _ in range(2))
            if case:
                run_away(k, g)
            own, ids = ids[:blocks[b]], ids[blocks[b]:]
            table[b, :blocks[b]] = own.int()
            held.append([x.bfloat16().cuda() for x in (k, v)])
            for cache, x in zip((kc, vc), held[-1]):
                full = torch.full((blocks[b] * 16, Hkv, D), float("nan"), dtype=torch.bfloat16, device="cuda")
                full[:m] = x
                cache[own.cuda()] = full.view(-1, 16, Hkv, D).transpose(1, 2)
        cu = torch.tensor([0] + rows).cumsum(0).int()
        got = ma.flash_attn_paged_prefill(q, kc, vc, cu.cuda(), table.cuda(), torch.tensor(keys).int().cuda(), most, kv_splits=1)
        for a, n, (k, v) in zip(cu.tolist(), rows, held):
            if n:
                look((case, n, len(k)), got[a:a + n], None, q[a:a + n], k, v, True)


def paged_promise(want, B, Hq, Hkv, D, rows, blocks, n_cu=0):
    for width in (blocks, 128, 129, 2 * blocks, 200, 4 * blocks, 500):
        for more in (1, 2, 4, 8, 16, 40, 100, 0.3):
            most = max(1, int(rows * more))
            if width >= blocks and named(B, Hq, Hkv, D, most, 0, 1, blocks=width, n_cu=n_cu) == want:
                return width, most


DENSE = [
    # eight wavefronts without split keys: pairs of tiles of long sequences that go over the chip more than four times, and calls without a mask
    (32, TILES, 8, 1, 130, 130, 4033, True), (64, TILES, 8, 1, 130, 65, 4033, True), (64, TILES, 8, 3, 16, 4, 933, False), (32, TILES, 8, 8, 8, 4, 2769, False),
    (64, TILES, 8, 128, 1, 1, 970, False),
    (32, TILES, 4, 24, 4, 4, 1309, False), (64, TILES, 4, 1, 32, 4, 2658, False), (64, TILES, 4, 16, 16, 16, 305, True), (128, TILES, 4, 60, 4, 4, 300, True),
    (128, W64, 4, 17, 16, 16, 1024, True), (128, W64, 4, 9, 16, 4, 1000, True), (128, W64, 4, 8, 32, 32, 960, False)]
DENSE += [(D, SHORT, 4, B, 16, hk, S, causal) for D in (32, 64) for B, hk, S, causal in (
    (64, 16, 17, True), (64, 4, 32, True), (64, 16, 33, False), (64, 4, 64, True), (64, 16, 127, True), (64, 4, 160, False), (64, 16, 193, True), (64, 8, 224, False),
    (64, 16, 256, True))]


@pytest.mark.parametrize("D,kernel,waves,B,Hq,Hkv,S,causal", DENSE)
def test_dense_calls(ma, D, kernel, waves, B, Hq, Hkv, S, causal):
    """A few heads are looked at, one of each with keys that run away, and one whose scores are all far below zero."""
    from mi355_attn import _lib, ops
    mask = _lib.MASK_CAUSAL if causal else _lib.MASK_NONE
    print(f"case: dense {NAMES[kernel]} {waves} D={D} {B} x {Hq}/{Hkv} {S} {causal}", flush=True)
    assert named(B, Hq, Hkv, D, S, S, mask) == named(B, Hq, Hkv, D, S, S, mask, lse=1) == (kernel, waves)
    g, G = torch.Generator(device="cuda").manual_seed(S + D), Hq // Hkv
    q, k, v = (torch.randn(B, h, S, D, generator=g, device="cuda") for h in (Hq, Hkv, Hkv))
    at = sorted({(0, 0), (B - 1, Hkv - 1), (B // 2, Hkv // 2), (0, Hkv - 1), (B - 1, 0)})
    draw = torch.Generator().manual_seed(S)
    for b, h in at[1:]:
        run_away(k[b, h], draw)
    b, h = at[-1]
    k[b, h], q[b, h * G] = k[b, h].abs() * 4.0, -q[b, h * G].abs() * 2.0
    q, k, v = (x.bfloat16() for x in (q, k, v))
    got, lse = ops._dense(q, k, v, None, mask, None, want_lse=True)
    assert torch.equal(ma.flash_attn_prefill(q, k, v, causal=causal, kv_splits=1), got) and bool(torch.isfinite(got).all())
    for b, h in at:
        heads = slice(h * G, h * G + G)
        look((b, h), got[b, heads].transpose(0, 1), lse[b, heads], q[b, heads].transpose(0, 1), k[b, h][:, None], v[b, h][:, None], causal)


@pytest.mark.parametrize("B,kernel", [(4096, W64), (4097, TILES)])
def test_as_many_sequences_as_the_wide_kernel_counts_and_one_more(ma, B, kernel):
    """It keeps one number per sequence, 4096 at most: packed sequences of one to three tokens, and the same over block tables."""
    print(f"case: {B} sequences, {NAMES[kernel]}", flush=True)
    g, D, Hq, Hkv = torch.Generator().manual_seed(B), 128, 2, 1
    rows = torch.randint(1, 4, (B,), generator=g).tolist()
    cu = torch.tensor([0] + rows).cumsum(0).int()
    q, k, v = (torch.randn(sum(rows), h, D, generator=g).bfloat16().cuda() for h in (Hq, Hkv, Hkv))
    most = promise((kernel, 4), 4096, Hq, Hkv, D, 800, 800, 1) if kernel == W64 else (1024, 1024)
    assert named(B, Hq, Hkv, D, *most, 1, 1) == (kernel, 4)
    got = ma.flash_attn_varlen_prefill(q, k, v, cu.cuda(), cu.cuda(), *most, causal=True, kv_splits=1)
    width, rows_most = paged_promise((kernel, 4), B, Hq, Hkv, D, 800, 100)
    table = torch.full((B, width), 2 ** 30, dtype=torch.int32)
    table[:, 0] = torch.randperm(B, generator=g)
    starts = cu[:-1].long().repeat_interleave(torch.tensor(rows))
    block, place = table[:, 0].long().repeat_interleave(torch.tensor(rows)).cuda(), (torch.arange(sum(rows)) - starts).cuda()
    caches = [torch.full((B, Hkv, 16, D), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    for cache, x in zip(caches, (k, v)):
        cache[block, 0, place] = x[:, 0]
    paged = ma.flash_attn_paged_prefill(q, *caches, cu.cuda(), table.cuda(), torch.tensor(rows).int().cuda(), rows_most, kv_splits=1)
    # rows of up to three positions, all sequences at once: position of each row in its sequence, and the two rows in front
    at = torch.stack([(torch.arange(sum(rows)) - d).clamp(min=0) for d in range(3)], 1).cuda()
    sees = torch.arange(3, device="cuda")[None] <= place[:, None]
    qd, kd, vd = q.double(), k.double()[:, 0][at], v.double()[:, 0][at]                                   # (T, Hq, D), (T, 3, D)
    s = (qd @ kd.transpose(1, 2) * D ** -0.5).masked_fill(~sees[:, None], -float("inf"))
    want = torch.softmax(s, -1) @ vd
    for out in (got, paged):
        assert bool(((out.double() - want).abs() <= 2.0 ** -8 * (2 * want.abs() + torch.softmax(s, -1) @ vd.abs()) + 1e-5).all())
