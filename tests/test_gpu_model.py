"""GPU parity of the operators around attention (RMSNorm, silu*up) and of the KV-cached decoder
(`CachedTransformerLM`) against the CPU oracle of the reference model.

Tolerances.  rms_norm / silu_mul: fp32 math with one rounding to bf16, so within one bf16 ulp of the
oracle's bf16 result: |got - ref| <= 2^-7 |ref| + 1e-3.  Decoder logits: the product path keeps weights,
activations and the residual stream in bf16 while the oracle computes in fp32 on the same bf16-rounded
weights; on the test models (2-3 layers, |logits| up to about 4) the observed error is below 0.03 and the
bound asserted is |got - ref| <= 8e-2 + 3e-2 |ref|.  Cached decode against a full forward of the same
path (same arithmetic, different kernels for attention): <= 3e-2 + 2e-2 |ref|.  Greedy tokens are checked
through the oracle's own logits: a generated token must be within 0.15 of the oracle's maximum at that step.
"""
import json

import pytest
import torch

from oracle import model_oracle as mo

pytestmark = pytest.mark.gpu

CFG = dict(vocab_size=211, context_length=64, d_model=128, num_layers=2, num_heads=4, d_ff=352, rope_theta=10000.0)


@pytest.fixture(scope="module")
def ops():
    import mi355_attn
    mi355_attn.load()
    return mi355_attn


def rnd(*shape, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(*shape, generator=g) * scale).to(torch.bfloat16)


def close_bf16(got, ref):
    torch.testing.assert_close(got.float().cpu(), ref.float(), atol=1e-3, rtol=2 ** -7)


@pytest.mark.parametrize("n_cols", [64, 512, 1000, 1024, 2048, 4096, 8192, 8200, 33])
@pytest.mark.parametrize("wdtype", [torch.float32, torch.bfloat16])
def test_rms_norm_matches_oracle(ops, n_cols, wdtype):
    print(f"case: rms_norm n_cols={n_cols} weight={wdtype}", flush=True)
    x = rnd(3, 7, n_cols, seed=n_cols, scale=2.5)
    w = (1.0 + 0.2 * torch.randn(n_cols, generator=torch.Generator().manual_seed(1))).to(wdtype)
    ref = mo.rms_norm_reference(x, w, 1e-5)
    y, rstd = ops.rms_norm(x.cuda(), w.cuda(), 1e-5, return_rstd=True)
    torch.cuda.synchronize()
    assert y.shape == x.shape and y.dtype == torch.bfloat16
    close_bf16(y, ref)
    want_rstd = torch.rsqrt(x.float().pow(2).mean(-1) + 1e-5)
    torch.testing.assert_close(rstd.cpu(), want_rstd, atol=1e-6, rtol=1e-5)


@pytest.mark.parametrize("n_cols", [128, 1536, 40])
def test_rms_norm_with_fused_residual(ops, n_cols):
    print(f"case: rms_norm residual n_cols={n_cols}", flush=True)
    x, r = rnd(19, n_cols, seed=2), rnd(19, n_cols, seed=3, scale=3.0)
    w = 1.0 + 0.2 * torch.randn(n_cols, generator=torch.Generator().manual_seed(4))
    h_ref = (x.float() + r.float()).to(torch.bfloat16)               # the bf16 add in front of the norm
    y, h = ops.rms_norm(x.cuda(), w.cuda(), 1e-5, residual=r.cuda(), return_sum=True)
    torch.cuda.synchronize()
    assert torch.equal(h.cpu(), h_ref)
    close_bf16(y, mo.rms_norm_reference(h_ref, w, 1e-5))
    # fused == unfused, bit for bit
    assert torch.equal(y, ops.rms_norm(h, w.cuda(), 1e-5))


def test_rms_norm_strided_rows_and_errors(ops):
    print("case: rms_norm strided / errors", flush=True)
    wide = rnd(11, 3 * 256, seed=5).cuda()
    w = torch.ones(256, device="cuda")
    x = wide[:, 256:512]                                              # row stride 768
    assert torch.equal(ops.rms_norm(x, w), ops.rms_norm(x.contiguous(), w))
    assert ops.rms_norm(torch.empty(0, 256, dtype=torch.bfloat16, device="cuda"), w).shape == (0, 256)
    with pytest.raises(ValueError):
        ops.rms_norm(x, torch.ones(255, device="cuda"))
    with pytest.raises(TypeError):
        ops.rms_norm(x.float(), w)
    with pytest.raises(TypeError):
        ops.rms_norm(x, w.half())
    with pytest.raises(ValueError):
        ops.rms_norm(x.cpu(), w)
    with pytest.raises(ValueError):
        ops.rms_norm(x, w, return_sum=True)


@pytest.mark.parametrize("n_cols", [352, 1024, 37])
def test_silu_mul_matches_oracle(ops, n_cols):
    print(f"case: silu_mul n_cols={n_cols}", flush=True)
    g, u = rnd(4, 9, n_cols, seed=6, scale=3.0), rnd(4, 9, n_cols, seed=7)
    ref = mo.silu_mul_reference(g, u)
    out = ops.silu_mul(g.cuda(), u.cuda())
    torch.cuda.synchronize()
    close_bf16(out, ref)
    # exp/sigmoid differ from torch's by an fp32 ulp at most: almost every element is bit-identical
    assert (out.cpu() == ref).float().mean() > 0.99
    # the two halves of one merged projection output, read in place
    gu = torch.cat((g, u), dim=-1).cuda()
    assert torch.equal(ops.silu_mul(gu[..., :n_cols], gu[..., n_cols:]), out)
    with pytest.raises(ValueError):
        ops.silu_mul(g.cuda(), u.cuda()[..., :-1])


def _bf16_params(cfg, seed, fused=False):
    return {k: v.to(torch.bfloat16) for k, v in mo.random_lm_params(cfg, seed, fused_ffn=fused).items()}


def _logit_close(got, ref, atol=8e-2, rtol=3e-2):
    err = (got.float().cpu() - ref).abs()
    bound = atol + rtol * ref.abs()
    assert bool((err <= bound).all()), f"max err {float(err.max()):.4f}, worst excess {float((err - bound).max()):.4f}"


@pytest.mark.parametrize("fused", [False, True])
def test_decoder_forward_matches_oracle(ops, fused):
    print(f"case: decoder forward fused_ffn={fused}", flush=True)
    params = _bf16_params(CFG, seed=11, fused=fused)
    model = ops.CachedTransformerLM(CFG, params, max_batch=8)
    ids = torch.randint(0, CFG["vocab_size"], (3, 41), generator=torch.Generator().manual_seed(12))
    got = model.forward(ids)
    ref = mo.transformer_lm_reference(params, CFG, ids)
    assert got.shape == ref.shape
    _logit_close(got, ref)
    assert model.engine.allocator.num_free == model.engine.allocator.num_blocks


def test_cached_decode_equals_full_forward_and_oracle(ops):
    print("case: cached decode vs full forward", flush=True)
    cfg = dict(CFG, num_layers=3, num_heads=2, d_model=128)          # d_head 64
    params = _bf16_params(cfg, seed=13)
    model = ops.CachedTransformerLM(cfg, params, max_batch=4)
    g = torch.Generator().manual_seed(14)
    seqs = [torch.randint(0, cfg["vocab_size"], (n,), generator=g) for n in (50, 33)]
    n_prompt = [17, 30]
    sids = [model.new_sequence() for _ in seqs]
    logits = model.prefill(sids, [s[:n] for s, n in zip(seqs, n_prompt)])
    per_seq = [[logits[i]] for i in range(2)]
    live = [0, 1]
    pos = list(n_prompt)
    while live:
        lg = model.decode([sids[i] for i in live], [int(seqs[i][pos[i]]) for i in live])
        for j, i in enumerate(live):
            per_seq[i].append(lg[j])
            pos[i] += 1
        live = [i for i in live if pos[i] < len(seqs[i])]
    for i, s in enumerate(seqs):
        got = torch.stack(per_seq[i])                                  # logits after tokens n_prompt-1 .. len-1
        full = model.forward(s)[0, n_prompt[i] - 1:]
        err = (got - full).abs()
        assert bool((err <= 3e-2 + 2e-2 * full.abs()).all()), float(err.max())
        _logit_close(got, mo.transformer_lm_reference(params, cfg, s[None])[0, n_prompt[i] - 1:])
    for s in sids:
        model.free_sequence(s)
    assert model.engine.allocator.num_free == model.engine.allocator.num_blocks


def test_cached_decode_with_fp8_kv_cache_tracks_the_oracle(ops):
    """The same decode loop over an fp8 KV pool (fused quantising cache write + fp8 decode kernel).
    e4m3 keeps 4 significant bits, so the logits carry quantisation noise on top of the bf16 path's: the
    bound asserted is 0.15 + 5e-2 |ref| against the fp32 oracle (observed 0.07), and the mean absolute
    error must stay below 0.03."""
    print("case: cached decode, fp8 KV", flush=True)
    cfg = dict(CFG, num_layers=3, num_heads=2, d_model=128)          # d_head 64
    params = _bf16_params(cfg, seed=13)
    model = ops.CachedTransformerLM(cfg, params, max_batch=4, kv_dtype="fp8")
    assert model.engine.k_caches[0].dtype == torch.uint8
    g = torch.Generator().manual_seed(14)
    seqs = [torch.randint(0, cfg["vocab_size"], (n,), generator=g) for n in (50, 33)]
    n_prompt = [17, 30]
    sids = [model.new_sequence() for _ in seqs]
    logits = model.prefill(sids, [s[:n] for s, n in zip(seqs, n_prompt)])
    per_seq = [[logits[i]] for i in range(2)]
    live, pos = [0, 1], list(n_prompt)
    while live:
        lg = model.decode([sids[i] for i in live], [int(seqs[i][pos[i]]) for i in live])
        for j, i in enumerate(live):
            per_seq[i].append(lg[j])
            pos[i] += 1
        live = [i for i in live if pos[i] < len(seqs[i])]
    for i, s in enumerate(seqs):
        got = torch.stack(per_seq[i]).float().cpu()
        ref = mo.transformer_lm_reference(params, cfg, s[None])[0, n_prompt[i] - 1:]
        err = (got - ref).abs()
        print(f"fp8 KV logits: max err {float(err.max()):.4f} mean {float(err.mean()):.4f}", flush=True)
        assert bool((err <= 0.15 + 5e-2 * ref.abs()).all()), float(err.max())
        assert float(err.mean()) < 0.03
    for s in sids:
        model.free_sequence(s)
    assert model.engine.allocator.num_free == model.engine.allocator.num_blocks


@pytest.mark.parametrize("kv_dtype", ["bf16", "fp8"])
def test_decode_steps_replayed_from_a_hip_graph_equal_eager_steps(ops, kv_dtype):
    """decode_graphs=True: the first step of a batch size runs eagerly and is captured, later steps are
    replays.  Every step of a graphed model is compared with the same step of an eager twin (whose own
    launches and synchronisations sit between the replays); sequences cross block boundaries, one leaves
    (a second batch size, a second graph) and a new one joins."""
    print(f"case: decode graphs, {kv_dtype} KV", flush=True)
    cfg = dict(CFG, num_layers=3, num_heads=2, d_model=128)          # d_head 64
    params = _bf16_params(cfg, seed=21)
    eager = ops.CachedTransformerLM(cfg, params, max_batch=4, kv_dtype=kv_dtype)
    graphed = ops.CachedTransformerLM(cfg, params, max_batch=4, kv_dtype=kv_dtype, decode_graphs=True)
    g = torch.Generator().manual_seed(22)
    prompts = [torch.randint(0, cfg["vocab_size"], (n,), generator=g) for n in (13, 30)]
    stream = torch.randint(0, cfg["vocab_size"], (40, 2), generator=g)
    se = [eager.new_sequence() for _ in prompts]
    sg = [graphed.new_sequence() for _ in prompts]
    torch.testing.assert_close(graphed.prefill(sg, prompts), eager.prefill(se, prompts))

    def step(ids_e, ids_g, toks):
        a = eager.decode(ids_e, toks)
        torch.cuda.synchronize()
        b = graphed.decode(ids_g, toks)
        torch.cuda.synchronize()
        err = (a - b).abs()
        assert bool((err <= 2e-2 + 2e-2 * a.abs()).all()), float(err.max())     # same kernels; the attention chunking differs
        return b

    for t in range(20):                                               # 13 -> 33 and 30 -> 50 tokens: new blocks on the way
        step(se, sg, stream[t].tolist())
    assert set(graphed._graphs) == {2} and graphed._graphs[2][1] is not None
    eager.free_sequence(se[0])
    graphed.free_sequence(sg[0])
    for t in range(20, 26):                                           # one sequence left: batch size 1
        step(se[1:], sg[1:], stream[t, 1:].tolist())
    ne, ng = eager.new_sequence(), graphed.new_sequence()             # a newcomer: back to batch size 2, its graph is reused
    p3 = torch.randint(0, cfg["vocab_size"], (5,), generator=g)
    torch.testing.assert_close(graphed.prefill([ng], [p3]), eager.prefill([ne], [p3]))
    for t in range(26, 34):
        last = step([se[1], ne], [sg[1], ng], stream[t].tolist())
    assert set(graphed._graphs) == {1, 2}
    # and against the oracle: the last step of the long sequence
    hist = torch.cat([prompts[1], stream[:26, 1], stream[26:34, 0]])    # what that sequence was fed
    ref = mo.transformer_lm_reference(params, cfg, hist[None])[0, -1]
    err = (last[0].float().cpu() - ref).abs()
    assert bool((err <= (0.15 if kv_dtype == "fp8" else 8e-2) + 5e-2 * ref.abs()).all()), float(err.max())


@pytest.mark.parametrize("name", ["_forward", "_forward_rows"])
def test_decode_graphs_of_a_subclass_hold_its_own_forward(ops, name):
    """A step's first run is eager and the others are replayed: both are what the subclass makes of it."""
    print(f"case: decode graphs of a subclass, {name}", flush=True)
    doubled = type("Doubled", (ops.CachedTransformerLM,), {
        name: lambda self, *a, **kw: getattr(super(type(self), self), name)(*a, **kw) * 2})
    cfg = dict(CFG, num_layers=2, num_heads=2, d_model=128)
    params, ids = _bf16_params(cfg, seed=51), [[3, 1, 4], [1, 5]]
    models = [ops.CachedTransformerLM(cfg, params, max_batch=2), doubled(cfg, params, max_batch=2, decode_graphs=True)]
    sids = [[m.new_sequence() for _ in ids] for m in models]
    for m, s in zip(models, sids):
        m.prefill(s, ids)
    for t in range(5):
        plain, twice = (m.decode(s, [t, 2 * t]) for m, s in zip(models, sids))
        torch.cuda.synchronize()
        _logit_close(twice / 2, plain.cpu())


@pytest.mark.parametrize("B", [1, 32, 33])
def test_replayed_logits_are_the_callers_own(ops, B):
    """On either side of the rows whose head may run behind the graph: what one step returned stays when later steps are replayed, and is an eager twin's."""
    print(f"case: replayed logits, {B} rows", flush=True)
    cfg = dict(CFG, num_layers=3, num_heads=2, d_model=128)
    params = _bf16_params(cfg, seed=61)
    models = [ops.CachedTransformerLM(cfg, params, max_batch=B, decode_graphs=g) for g in (False, True)]
    tokens = torch.randint(0, cfg["vocab_size"], (B, 8), generator=torch.Generator().manual_seed(62))
    sids = [[m.new_sequence() for _ in range(B)] for m in models]
    for m, s in zip(models, sids):
        m.prefill(s, list(tokens[:, :3]))
    got = [[m.decode(s, tokens[:, t].tolist()) for t in range(3, 8)] for m, s in zip(models, sids)]
    torch.cuda.synchronize()
    assert len({t.data_ptr() for t in got[1]}) == 5
    for a, b in zip(*got):
        _logit_close(b[None], a[None].cpu())


def test_decode_steps_ask_the_attention_they_are_given(ops):
    """An engine whose attend_decode is replaced (to look at queries and keys, say) is asked in every layer of a decode step."""
    print("case: replaced attend_decode", flush=True)
    params = _bf16_params(CFG, seed=3)
    model = ops.CachedTransformerLM(CFG, params, max_batch=2)
    twin = ops.CachedTransformerLM(CFG, params, max_batch=2)
    seen, attend = [], model.engine.attend_decode
    model.engine.attend_decode = lambda layer, plan, q, k, v: seen.append((layer, q.shape, k.shape)) or attend(layer, plan, q, k, v)
    for m in (model, twin):
        m.sids = [m.new_sequence()]
        m.prefill(m.sids, [torch.arange(5)])
    got, ref = model.decode(model.sids, [7]), twin.decode(twin.sids, [7])
    assert seen == [(i, (1, 4, 32), (1, 4, 32)) for i in range(CFG["num_layers"])]
    assert bool(((got - ref).abs() <= 3e-2 + 2e-2 * ref.abs()).all())               # (queries and keys are rounded once more in front of the rotation)


def _check_greedy(params, cfg, prompt, toks, margin=0.15):
    """Every generated token must be (nearly) the oracle's argmax given the tokens before it, with the
    reference's sliding window (model.py:215)."""
    ids = [int(t) for t in prompt]
    for t in toks:
        ctx = torch.tensor(ids[-cfg["context_length"]:])[None]
        lg = mo.transformer_lm_reference(params, cfg, ctx)[0, -1]
        assert float(lg.max() - lg[t]) <= margin, (len(ids), t, int(lg.argmax()))
        ids.append(int(t))


def test_generate_greedy_follows_oracle_including_window_slide(ops):
    print("case: generate greedy", flush=True)
    params = _bf16_params(CFG, seed=15)
    model = ops.CachedTransformerLM(CFG, params, max_batch=4)
    prompt = torch.randint(0, CFG["vocab_size"], (1, 9), generator=torch.Generator().manual_seed(16))
    out = model.generate(prompt, 12, temperature=0)
    assert out.shape == (1, 12) and out.dtype == torch.int64
    _check_greedy(params, CFG, prompt[0].tolist(), out[0].tolist())
    # eos: generation stops before the eos token (model.py:229-230)
    out2 = model.generate(prompt[0], 12, temperature=0, eos_token_id=int(out[0, 4]))
    first = out[0].tolist().index(int(out[0, 4]))
    assert out2[0].tolist() == out[0].tolist()[:first]
    # prompt close to the context length: the window slides and positions restart (model.py:215)
    long_prompt = torch.randint(0, CFG["vocab_size"], (60,), generator=torch.Generator().manual_seed(17))
    out3 = model.generate(long_prompt, 9, temperature=0)
    _check_greedy(params, CFG, long_prompt.tolist(), out3[0].tolist())
    # a prompt longer than the context is truncated to its last context_length tokens
    over = torch.randint(0, CFG["vocab_size"], (80,), generator=torch.Generator().manual_seed(18))
    out4 = model.generate(over, 3, temperature=0)
    _check_greedy(params, CFG, over.tolist(), out4[0].tolist())
    assert model.engine.allocator.num_free == model.engine.allocator.num_blocks


def test_generate_sampling_and_top_k(ops):
    print("case: generate sampling", flush=True)
    params = _bf16_params(CFG, seed=19)
    model = ops.CachedTransformerLM(CFG, params, max_batch=4)
    prompt = torch.tensor([5, 6, 7, 8])
    g = torch.Generator(device="cuda").manual_seed(1)
    a = model.generate(prompt, 8, temperature=0.8, top_k=5, generator=g)
    g.manual_seed(1)
    b = model.generate(prompt, 8, temperature=0.8, top_k=5, generator=g)
    assert torch.equal(a, b) and a.shape == (1, 8)
    # top_k=1 is greedy whatever the temperature
    assert torch.equal(model.generate(prompt, 6, temperature=1.3, top_k=1), model.generate(prompt, 6, temperature=0))
    # with top_k = 5 every sampled token is among the oracle's 5 best (up to near-ties)
    ids = prompt.tolist()
    for t in a[0].tolist():
        lg = mo.transformer_lm_reference(params, CFG, torch.tensor(ids)[None])[0, -1]
        assert float(torch.topk(lg, 5).values[-1] - lg[t]) <= 0.15
        ids.append(t)


def test_generate_batch_continuous_batching(ops):
    print("case: generate_batch", flush=True)
    params = _bf16_params(CFG, seed=20)
    model = ops.CachedTransformerLM(CFG, params, max_batch=8)
    g = torch.Generator().manual_seed(21)
    prompts = [torch.randint(0, CFG["vocab_size"], (n,), generator=g).tolist() for n in (3, 17, 58, 1, 33)]
    outs = model.generate_batch(prompts, 10, temperature=0)
    assert [len(o) for o in outs] == [10, 10, 64 - 58 + 1, 10, 10]     # the third one fills its context
    for p, o in zip(prompts, outs):
        _check_greedy(params, CFG, p, o)
    eos = outs[1][3]
    outs2 = model.generate_batch(prompts, 10, temperature=0, eos_token_id=eos)
    for o, o2 in zip(outs, outs2):
        want = o[:o.index(eos)] if eos in o else o
        assert o2 == want
    assert model.engine.allocator.num_free == model.engine.allocator.num_blocks
    with pytest.raises(ValueError):
        model.generate_batch([[1]] * 9, 1)


@pytest.mark.parametrize("d_ff", [352, 356])
@pytest.mark.parametrize("graphs", [False, True])
def test_decode_across_the_row_limit_of_the_fused_layers(ops, d_ff, graphs):
    """35 sequences that end one after the other: steps of more than 32 rows run rows_linear in tiles and separate rotation (with a
    d_ff that is no multiple of 8 all steps run library products), the others the fused layers; a sequence that sees both follows the oracle.  Eager and replayed."""
    print(f"case: decode across 32 rows, d_ff {d_ff} graphs {graphs}", flush=True)
    cfg = dict(CFG, d_ff=d_ff)
    params = _bf16_params(cfg, seed=31)
    model = ops.CachedTransformerLM(cfg, params, max_batch=36, decode_graphs=graphs)
    assert model._rows_fuse == (d_ff % 8 == 0)
    g = torch.Generator().manual_seed(32)
    seqs = [torch.randint(0, cfg["vocab_size"], (8 + (3 * i + 7) % 17 + (12 if i < 4 else 0),), generator=g) for i in range(35)]
    sids = [model.new_sequence() for _ in seqs]
    logits = model.prefill(sids, [s[:5] for s in seqs])
    rows, live, widths = [[logits[i]] for i in range(35)], list(range(35)), []
    for t in range(5, 40):
        live = [i for i in live if t < len(seqs[i])]
        if not live:
            break
        widths.append(len(live))
        logits = model.decode([sids[i] for i in live], [int(seqs[i][t]) for i in live])
        for j, i in enumerate(live):
            rows[i].append(logits[j])
    assert widths[0] == 35 and min(widths) <= 4 and widths.count(35) >= 2 and any(1 < w <= 32 for w in widths)
    for i, s in enumerate(seqs):
        _logit_close(torch.stack(rows[i])[None], mo.transformer_lm_reference(params, cfg, s[None])[:, 4:])
    for s in sids:
        model.free_sequence(s)


@pytest.mark.parametrize("n_tokens", [20, 50, 200, 1100])
def test_rows_of_a_prompt_are_indexed_like_torch_indexes(ops, n_tokens):
    """On either side of the sizes whose linear layers take row numbers: negative positions count from the end, none are few enough, rows that
    are not there are refused before anything is reserved; ids and rows may be on the GPU."""
    print(f"case: rows of {n_tokens} tokens", flush=True)
    cfg = dict(CFG, context_length=1200)
    model = ops.CachedTransformerLM(cfg, _bf16_params(cfg, seed=41), max_batch=4)
    ids = torch.randint(0, cfg["vocab_size"], (n_tokens,), generator=torch.Generator().manual_seed(42))
    parts = [ids[:n_tokens // 3], ids[n_tokens // 3:]]

    def logits(rows=None, parts=parts):
        sids = [model.new_sequence() for _ in parts]
        try:
            return model.prefill(sids, parts, **(dict(all_logits=True) if rows is None else dict(rows=rows)))
        finally:
            for s in sids:
                model.free_sequence(s)

    every = logits()
    assert every.shape[0] == n_tokens
    for rows in ([-1], [0, -n_tokens, n_tokens - 1, -2], list(range(-min(n_tokens, 90), 0)), torch.tensor([3, -3])):
        picked = torch.as_tensor(rows)
        _logit_close(logits(rows)[None], every[picked.cuda()][None].cpu())
        _logit_close(logits(picked.cuda())[None], every[picked.cuda()][None].cpu())
        _logit_close(logits(rows, [p.cuda() - cfg["vocab_size"] for p in parts])[None], every[picked.cuda()][None].cpu())      # (the same ids)
    assert logits([]).shape == (0, cfg["vocab_size"])
    free = model.engine.allocator.num_free
    for rows in ([n_tokens], [0, -n_tokens - 1]):
        with pytest.raises(IndexError):
            logits(rows)
    sids = [model.new_sequence() for _ in range(2)]
    model.prefill(sids, [[1, 2], [3]])
    one = model.step(sids, [[4], [5]], rows=[-1, 0])
    assert one.shape == (2, cfg["vocab_size"])
    with pytest.raises(IndexError):
        model.step(sids, [[4], [5]], rows=[2])
    assert model.engine.lengths[sids[0]] == 3                         # (nothing was appended)
    for s in sids:
        model.free_sequence(s)
    assert model.engine.allocator.num_free == free


def test_from_pretrained_reads_reference_files(ops, tmp_path):
    print("case: from_pretrained", flush=True)
    params = mo.random_lm_params(CFG, seed=22)
    (tmp_path / "model_config.json").write_text(json.dumps(CFG))
    torch.save({"model": {"_orig_mod." + k: v for k, v in params.items()}}, tmp_path / "ckpt.pt")
    model = ops.CachedTransformerLM.from_pretrained(str(tmp_path / "model_config.json"), str(tmp_path / "ckpt.pt"), max_batch=2)
    ids = torch.arange(20)[None] % CFG["vocab_size"]
    bf = {k: v.to(torch.bfloat16) for k, v in params.items()}
    _logit_close(model.forward(ids), mo.transformer_lm_reference(bf, CFG, ids))
    with pytest.raises(ValueError):
        ops.CachedTransformerLM(dict(CFG, num_heads=8), bf)            # d_head 16 is not supported by the kernels


# ---- linear layers of a decode step ----------------------------------------------------------------------
def _close_rows(got, ref, rounded, what):
    """Products of bf16 operands with fp32 sums: what is rounded to bf16 on the way (the normed operand, the result) is off by 2^-9 of itself at
    most, a sum of k roundings of random sign by no more of its norm."""
    got, ref = got.double().cpu(), ref.double().cpu()
    assert bool(torch.isfinite(got).all()), what
    assert float((got - ref).norm()) <= (rounded * 2 ** -8 + 1e-6) * float(ref.norm()), what


@pytest.mark.parametrize("T", [1, 16, 17, 32])
@pytest.mark.parametrize("k,n", [(8, 4), (64, 30), (72, 129), (512, 96), (1344, 512), (4096, 36)])
def test_rows_linear(ops, T, k, n):
    """Edges of the row tiles, of the 32 weight rows of a workgroup and of the 64-wide steps of k (fewer than four of them, remainders)."""
    g = torch.Generator().manual_seed(T * 1000 + k)

    def t(*shape, std=1.0):
        return (torch.randn(*shape, generator=g) * std).to(torch.bfloat16).cuda()

    table, w, norm = t(50, k + 8), t(2 * n, k, std=k ** -0.5), (torch.randn(k, generator=g) * 0.3 + 1).cuda()
    ids = torch.randint(0, 50, (T,), generator=g).cuda()
    rows, resid = table[:, :k], t(40, n + 4)[:, :n]
    x = rows[ids].double()
    normed = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5) * norm.double()
    wd = w.double()
    _close_rows(ops.rows_linear(rows[:T].contiguous(), w[:n].contiguous()), rows[:T].double() @ wd[:n].T, 1, "plain")
    _close_rows(ops.rows_linear(rows, w[:n].contiguous(), x_rows=ids, out_dtype=torch.float32), x @ wd[:n].T, 0, "fp32")
    _close_rows(ops.rows_linear(rows, w[:n].contiguous(), x_rows=ids, norm=norm, out_dtype=torch.float32), normed @ wd[:n].T, 1, "norm")
    pick = torch.randint(0, 40, (T,), generator=g).cuda()
    _close_rows(ops.rows_linear(rows, w[:n].contiguous(), x_rows=ids, resid=resid, resid_rows=pick), x @ wd[:n].T + resid[pick].double(), 1, "add")
    gate, up = (normed @ wd.T).split(n, 1)
    _close_rows(ops.rows_linear(rows, w, x_rows=ids, norm=norm, gate_up=True), torch.nn.functional.silu(gate) * up, 3, "gate_up")
    with pytest.raises(ValueError):
        ops.rows_linear(t(33, k), w)


@pytest.mark.parametrize("T,k,n", [(33, 64, 30), (64, 72, 129), (65, 512, 96), (200, 1344, 512), (1024, 4096, 36)])
def test_rows_linear_of_a_prompt(ops, T, k, n):
    """More rows than one launch's tile: edges of the tiles of 32 rows, against the same bound as a decode step's; 1025 rows are refused."""
    print(f"case: prompt linear {T} {k} {n}", flush=True)
    g = torch.Generator().manual_seed(T + k)

    def t(*shape, std=1.0):
        return (torch.randn(*shape, generator=g) * std).to(torch.bfloat16).cuda()

    table, w, norm = t(50, k + 8), t(2 * n, k, std=k ** -0.5), (torch.randn(k, generator=g) * 0.3 + 1).cuda()
    ids, pick = (torch.randint(0, m, (T,), generator=g).cuda() for m in (50, 40))
    rows, resid = table[:, :k], t(40, n + 4)[:, :n]
    x, wd = rows[ids].double(), w.double()
    normed = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5) * norm.double()
    one = w[:n].contiguous()
    _close_rows(ops.rows_linear(rows[ids].contiguous(), one, prompt=True), x @ wd[:n].T, 1, "plain")
    _close_rows(ops.rows_linear(rows, one, x_rows=ids, norm=norm, out_dtype=torch.float32, prompt=True), normed @ wd[:n].T, 1, "norm, fp32")
    _close_rows(ops.rows_linear(rows, one, x_rows=ids, resid=resid, resid_rows=pick, prompt=True), x @ wd[:n].T + resid[pick].double(), 1, "add")
    gate, up = (normed @ wd.T).split(n, 1)
    _close_rows(ops.rows_linear(rows, w, x_rows=ids, norm=norm, gate_up=True, prompt=True), torch.nn.functional.silu(gate) * up, 3, "gate_up")
    with pytest.raises(ValueError):
        ops.rows_linear(t(1025, k), w, prompt=True)


@pytest.mark.parametrize("T", [3, 20])
@pytest.mark.parametrize("k", [72, 200, 256])
def test_rows_linear_with_infinities(ops, T, k):
    """Infinite and NaN weights and rows give what the product gives, also in the last, partial step of k."""
    g = torch.Generator().manual_seed(k)
    x, w = torch.rand(T, k, generator=g).to(torch.bfloat16) + 0.5, torch.randn(40, k, generator=g).to(torch.bfloat16)
    last = k // 64 * 64 if k % 64 else k - 64                           # where the last step of k begins
    w[1, last], w[2, last + 7], w[3, k - 1], w[4, 0], w[5, last], w[6, last + 1] = float("inf"), -float("inf"), float("inf"), -float("inf"), float("nan"), 3e38
    x[1, k - 1] = float("inf")
    x[2, last] = float("nan")
    ref = x.float() @ w.float().T
    got = ops.rows_linear(x.cuda(), w.cuda(), out_dtype=torch.float32).cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(ref)) and torch.equal(torch.isinf(got), torch.isinf(ref))
    fine = torch.isfinite(ref)
    assert torch.equal(got[torch.isinf(ref)], ref[torch.isinf(ref)]) and torch.allclose(got[fine], ref[fine], rtol=1e-4, atol=1e-3)


@pytest.mark.parametrize("T,H,G,D", [(1, 2, 2, 32), (17, 4, 1, 64), (32, 8, 2, 128)])
def test_rows_qkv(ops, T, H, G, D):
    """Projection, rotation and cache write in one launch against the product and rope_and_cache: the product is rounded once less."""
    g = torch.Generator().manual_seed(D)
    k, nb = 200, 9

    def t(*shape, std=1.0):
        return (torch.randn(*shape, generator=g) * std).to(torch.bfloat16).cuda()

    x, w = t(T, k), t((H + 2 * G) * D, k, std=k ** -0.5)
    pos = torch.randint(0, 70, (T,), generator=g).int().cuda()                  # (some beyond the table: clamped into it)
    slots = torch.randperm(nb * 16, generator=g)[:T].cuda()
    slots[0] = -1 if T > 1 else slots[0]
    freq = ops.build_rope_cache(64, D)
    pools = [torch.full((nb, G, 16, D), 3.0, dtype=torch.bfloat16).cuda() for _ in range(4)]
    q = ops.rows_qkv(x, w, pos, freq, pools[0], pools[1], slots, H)
    qkv = (x.float() @ w.float().T).to(torch.bfloat16).view(T, H + 2 * G, D)
    ref = ops.rope_and_cache(qkv[:, :H], qkv[:, H:H + G], qkv[:, H + G:], pos, freq, pools[2], pools[3], slots)
    for got, want, what in ((q, ref, "q"), (pools[0], pools[2], "k"), (pools[1], pools[3], "v")):
        _close_rows(got, want, 2, what)
        assert torch.equal(got.float().cpu() == 3.0, want.float().cpu() == 3.0) or what == "q"       # the same rows are written
