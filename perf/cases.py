"""What is measured: one pass through the package's public operators and models, over the sizes they are used at.

listed() are twelve calls that stand for the library's uses, draw() gives more of the same ranges.  Lengths of a ragged
batch are the quantiles of their distribution, dealt to the sequences by the seed, so that the work of a case does not
depend on the seed.  exact() is plain torch in float64; where a storage format belongs to what is computed (a cache of
bf16 or e4m3 rows) the rounding to that format is part of it.
"""
from __future__ import annotations

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "llm-systems-from-scratch_amd"))

import mi355_attn as ma  # noqa: E402

DEV = "cuda:0"
BLOCK = 16
BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64


# ---- the cases ---------------------------------------------------------------------------------------------------------

def listed():
    return [
        # One step's attention of a small model with a handful of short sequences: launch latency and host time.
        dict(name="decode-small", kind="decode", batch=4, q_heads=8, kv_heads=8, head_dim=64, lengths="fixed", lo=256, hi=256,
             fp8=False, window=0, keep_first=0),
        # A loaded server's step, bf16 cache: 128 sequences of very different age.
        dict(name="decode-bf16-ragged", kind="decode", batch=128, q_heads=32, kv_heads=8, head_dim=128, lengths="uniform", lo=512,
             hi=16384, fp8=False, window=0, keep_first=0),
        # The same with an 8-bit cache, more sequences and more query heads per key head.
        dict(name="decode-fp8-ragged", kind="decode", batch=256, q_heads=64, kv_heads=8, head_dim=128, lengths="log", lo=128,
             hi=32768, fp8=True, window=0, keep_first=0),
        # Attention of the reference's sample model (configures/sample.yaml) in inference: many short heads of 32.
        dict(name="prefill-sample", kind="prefill", batch=64, q_heads=16, kv_heads=16, head_dim=32, lengths="fixed", lo=256, hi=256,
             packed=False, train=False, amp=False, window=0, keep_first=0),
        # Prompts of a large grouped-query model, packed.
        dict(name="prefill-gqa", kind="prefill", batch=8, q_heads=32, kv_heads=8, head_dim=128, lengths="fixed", lo=4096, hi=4096,
             packed=True, train=False, amp=False, window=0, keep_first=0),
        # The sample model's attention in training as `train.py --amp --flash-attn` calls it: fp32 Q and K (RoPE's table is
        # fp32), bf16 V, forward and gradients.
        dict(name="train-sample", kind="prefill", batch=64, q_heads=16, kv_heads=16, head_dim=32, lengths="fixed", lo=256, hi=256,
             packed=False, train=True, amp=True, window=0, keep_first=0),
        # Training on packed documents of unequal length.
        dict(name="train-gqa-ragged", kind="prefill", batch=16, q_heads=32, kv_heads=8, head_dim=128, lengths="log", lo=256, hi=4096,
             packed=True, train=True, amp=False, window=0, keep_first=0),
        # Portions of long prompts over an 8-bit cache: rotation and cache write, then attention through the block tables.
        dict(name="chunk-fp8", kind="chunk", batch=4, q_heads=32, kv_heads=8, head_dim=128, rows=2048, lengths="fixed", lo=6144,
             hi=6144, fp8=True),
        # The sample model served: eight prompts, then every sequence's given continuation token by token.
        dict(name="serve-sample", kind="serve", vocab=10000, context=256, width=512, layers=4, heads=16, ff=1344, batch=8, prompt=32,
             steps=32, graphs=True),
        # A mixture of experts in a decode step of 32 sequences (its weights are what is read), and over a batch of prompts.
        dict(name="moe-decode", kind="moe", tokens=32, width=2048, experts=16, top=4, ff=1024),
        dict(name="moe-prefill", kind="moe", tokens=8192, width=2048, experts=16, top=4, ff=1024),
        # A Mamba-2 mixer between its projections over four prompts.
        dict(name="mamba-prefill", kind="mamba", batch=4, lengths="fixed", lo=2048, hi=2048, heads=64, vdim=64, state=128, groups=1),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        pool = sum(_lengths(case)) * 4 * case["kv_heads"] * case["head_dim"] if case["kind"] in ("decode", "chunk") else 0
        # nothing dearer than the listed cases: 4.5 GB moved or kept, a prefill or training step of about a TFLOP
        if max(w["bytes"], pool) <= 4.6e9 and w["flops"] <= {"chunk": 0.8e12, "moe": 0.42e12}.get(case["kind"], 1.1e12):
            return case


def _draw(rng):
    kind = rng.choice(("decode", "decode", "prefill", "prefill", "train", "train", "chunk", "serve", "moe", "moe", "mamba"))
    if kind in ("decode", "prefill", "train", "chunk"):
        fp8 = kind in ("decode", "chunk") and rng.random() < 0.5
        head_dim = rng.choice((64, 128, 128) if fp8 else (32, 64, 128, 128))
        kv_heads = rng.choice((1, 2, 4, 8, 16))
        group = rng.choice((1, 2, 4, 8) if kv_heads < 16 else (1, 2))
        case = dict(kind=kind, q_heads=kv_heads * group, kv_heads=kv_heads, head_dim=head_dim, lengths=rng.choice(("fixed", "uniform", "log")))
        window, keep = ((rng.choice((512, 1024)), rng.choice((0, 4, 64))) if rng.random() < 0.2 else (0, 0))
        if kind == "decode":
            hi = _log_int(rng, 64, 32768)
            return dict(case, batch=_log_int(rng, 1, 256), lo=hi if case["lengths"] == "fixed" else max(1, hi // rng.choice((4, 32, 256))),
                        hi=hi, fp8=fp8, window=window, keep_first=keep)
        if kind == "chunk":
            hi = _log_int(rng, 16, 16384)
            return dict(case, batch=_log_int(rng, 1, 16), rows=_log_int(rng, 16, 4096), lo=hi if case["lengths"] == "fixed" else max(1, hi // 8),
                        hi=hi, fp8=fp8)
        train = kind == "train"
        packed = rng.random() < 0.5
        hi = _log_int(rng, 64, 8192)
        if not packed:
            case.update(lengths="fixed", kv_heads=case["q_heads"])       # the reference's own module has as many key heads
        return dict(case, kind="prefill", batch=_log_int(rng, 1, 64), lo=hi if case["lengths"] == "fixed" else max(1, hi // 16), hi=hi,
                    packed=packed, train=train, amp=not packed and rng.random() < 0.5, window=window if packed and not train else 0,
                    keep_first=keep if packed and not train else 0)
    if kind == "serve":
        width = rng.choice((256, 512, 1024))
        prompt = _log_int(rng, 8, 160)
        return dict(kind=kind, vocab=10000, context=256, width=width, layers=rng.randint(2, 4), heads=width // rng.choice((32, 64)),
                    ff=rng.choice((width * 2, width * 21 // 8, width * 4)), batch=_log_int(rng, 1, 32), prompt=prompt,
                    steps=rng.randint(8, 24), graphs=rng.random() < 0.7)
    if kind == "moe":
        width = rng.choice((512, 1024, 2048))
        return dict(kind=kind, tokens=_log_int(rng, 1, 8192), width=width, experts=rng.choice((8, 16, 32)), top=rng.choice((1, 2, 4)),
                    ff=rng.choice((width // 2, width)))
    hi = _log_int(rng, 64, 8192)
    lengths = rng.choice(("fixed", "uniform", "log"))
    return dict(kind="mamba", batch=_log_int(rng, 1, max(1, min(16, 16384 // hi))), lengths=lengths, lo=hi if lengths == "fixed" else max(1, hi // 16), hi=hi,
                heads=rng.choice((16, 32, 64)), vdim=64, state=rng.choice((64, 128)), groups=rng.choice((1, 2)))


def _lengths(case):
    """The batch's lengths, ascending: quantiles of the case's distribution."""
    n, lo, hi = case["batch"], case["lo"], case["hi"]
    if case["lengths"] == "fixed":
        return [hi] * n
    at = [(i + 0.5) / n for i in range(n)]
    if case["lengths"] == "uniform":
        return [min(hi, lo + int(u * (hi - lo + 1))) for u in at]
    return [max(lo, min(hi, round(lo * (hi / lo) ** u))) for u in at]


def _dealt(case, seed):
    g = torch.Generator().manual_seed(seed + 1)
    lens = _lengths(case)
    return [lens[i] for i in torch.randperm(len(lens), generator=g).tolist()]


# ---- inputs ------------------------------------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _normal(g, *shape, std=1.0, dtype=BF16):
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(dtype)


def _int32(values):
    return torch.tensor(values, dtype=torch.int32, device=DEV)


def _running(lens):
    out = [0]
    for n in lens:
        out.append(out[-1] + n)
    return out


def _tables(lens, seed):
    """Block tables of sequences of these lengths over a shuffled pool a tenth larger than needed: (tables, pool size)."""
    need = [-(-n // BLOCK) for n in lens]
    pool = math.ceil(sum(need) * 1.1)
    ids = torch.randperm(pool, generator=torch.Generator().manual_seed(seed + 2)).tolist()
    rows, at = torch.zeros(len(lens), max(need), dtype=torch.int32), 0
    for i, n in enumerate(need):
        rows[i, :n] = torch.tensor(ids[at:at + n], dtype=torch.int32)
        at += n
    return rows, pool


def _pool(g, shape, fp8):
    """A cache pool of N(0, 1) rows: (cache, scales or None)."""
    if not fp8:
        return _normal(g, *shape), None
    x = torch.randn(*shape, generator=g, device=DEV)
    scale = x.abs().amax(dim=(2, 3)) / 448.0
    return (x / scale[:, :, None, None]).clamp_(-448, 448).to(torch.float8_e4m3fn).view(torch.uint8), scale


def prepare(case, seed):
    return {"decode": _prepare_decode, "prefill": _prepare_prefill, "chunk": _prepare_chunk, "serve": _prepare_serve,
            "moe": _prepare_moe, "mamba": _prepare_mamba}[case["kind"]](case, seed)


def _prepare_decode(case, seed):
    g, lens = _gen(seed), _dealt(case, seed)
    rows, pool = _tables(lens, seed)
    B, H, G, D = case["batch"], case["q_heads"], case["kv_heads"], case["head_dim"]
    kc, ks = _pool(g, (pool, G, BLOCK, D), case["fp8"])
    vc, vs = _pool(g, (pool, G, BLOCK, D), case["fp8"])
    bound = rows.shape[1] * BLOCK
    return dict(case=case, lens=lens, q=_normal(g, B, H, D), kc=kc, vc=vc, ks=ks, vs=vs, tables=rows.to(DEV), ctx=_int32(lens), bound=bound,
                workspace=ma.paged_decode_workspace(B, H, D, bound, torch.device(DEV)))


def _prepare_prefill(case, seed):
    g, lens = _gen(seed), _dealt(case, seed)
    B, H, G, D, T = case["batch"], case["q_heads"], case["kv_heads"], case["head_dim"], sum(lens)
    qk = F32 if case["amp"] else BF16
    if case["packed"]:
        q, k, v = _normal(g, T, H, D, std=0.5), _normal(g, T, G, D, std=0.5), _normal(g, T, G, D, std=0.5)
        dout = _normal(g, T, H, D, std=0.5) if case["train"] else None
    else:
        S = case["hi"]
        # V is a view of the (batch, seq, heads * d_head) projection, Q and K come contiguous out of RoPE (model.py:367-378)
        q, k = (_normal(g, B, n, S, D, std=0.5, dtype=qk) for n in (H, G))
        v = _normal(g, B, S, G, D, std=0.5).permute(0, 2, 1, 3)
        dout = _normal(g, B, S, H, D, std=0.5).permute(0, 2, 1, 3) if case["train"] else None
    if case["train"]:
        for t in (q, k, v):
            t.requires_grad_()
    return dict(case=case, lens=lens, q=q, k=k, v=v, dout=dout, cu=_int32(_running(lens)), longest=max(lens))


def _prepare_chunk(case, seed):
    g = _gen(seed)
    B, H, G, D, n = case["batch"], case["q_heads"], case["kv_heads"], case["head_dim"], case["rows"]
    before = [-(-x // BLOCK) * BLOCK for x in _dealt(case, seed)]            # a portion begins with a block
    total = [b + n for b in before]
    rows, pool = _tables(total, seed)
    (kc, ks), (vc, vs) = _pool(g, (pool, G, BLOCK, D), case["fp8"]), _pool(g, (pool, G, BLOCK, D), case["fp8"])
    qkv = _normal(g, B * n, H + 2 * G, D, std=0.5)                           # the merged projection
    pos = torch.cat([torch.arange(b, b + n) for b in before])
    slots = torch.cat([rows[i, torch.arange(b, b + n) // BLOCK].long() * BLOCK + torch.arange(b, b + n) % BLOCK for i, b in enumerate(before)])
    return dict(case=case, before=before, q=qkv[:, :H], k=qkv[:, H:H + G], v=qkv[:, H + G:], kc=kc, vc=vc, ks=ks, vs=vs,
                tables=rows.to(DEV), ctx=_int32(total), cu=_int32(_running([n] * B)), cu_ctx=_int32(_running(total)), total=sum(total),
                bound=max(total), pos=pos.to(DEV, torch.int32), slots=slots.to(DEV), freq=ma.build_rope_cache(max(total), D, device=DEV))


def _prepare_serve(case, seed):
    g = _gen(seed)
    V, d, ff, B = case["vocab"], case["width"], case["ff"], case["batch"]
    sd = {"token_embeddings.weight": _normal(g, V, d), "lm_head.weight": _normal(g, V, d, std=d ** -0.5),
          "final_norm.weight": _normal(g, d, std=0.1, dtype=F32) + 1}
    for i in range(case["layers"]):
        pre = f"layers.{i}."
        for n in ("q_proj", "k_proj", "v_proj", "output_proj"):
            sd[f"{pre}attn.{n}.weight"] = _normal(g, d, d, std=d ** -0.5)
        for n, shape in (("gate_proj", (ff, d)), ("up_proj", (ff, d)), ("down_proj", (d, ff))):
            sd[f"{pre}ffn.{n}.weight"] = _normal(g, *shape, std=shape[1] ** -0.5)
        for n in ("attn_norm", "ffn_norm"):
            sd[f"{pre}{n}.weight"] = _normal(g, d, std=0.1, dtype=F32) + 1
    cfg = dict(vocab_size=V, context_length=case["context"], d_model=d, num_layers=case["layers"], num_heads=case["heads"], d_ff=ff, rope_theta=10000.0)
    model = ma.CachedTransformerLM(cfg, sd, max_batch=B, decode_graphs=case["graphs"])
    tokens = torch.randint(0, V, (B, _prompt(case, 0) + case["steps"]), generator=torch.Generator().manual_seed(seed))
    state = dict(case=case, model=model, sd=sd, prompts=[tokens[i, :_prompt(case, i)] for i in range(B)],
                 given=[[int(tokens[i, _prompt(case, i) + t]) for i in range(B)] for t in range(case["steps"])], tokens=tokens)
    if case["graphs"]:          # a server has taken a step of this batch size before
        sids = [model.new_sequence() for _ in range(B)]
        model.prefill(sids, state["prompts"])
        model.decode(sids, state["given"][0])
        for s in sids:
            model.free_sequence(s)
    return state


def _prompt(case, i):
    """Prompts get shorter by up to a half over the batch."""
    return max(1, case["prompt"] - i * (case["prompt"] // 2) // max(1, case["batch"]))


def _prepare_moe(case, seed):
    g = _gen(seed)
    T, d, E, ff = case["tokens"], case["width"], case["experts"], case["ff"]
    return dict(case=case, h=_normal(g, T, d), sub=_normal(g, T, d), router=_normal(g, E, d, std=d ** -0.5), bias=_normal(g, E, std=0.1, dtype=F32),
                gate_up=_normal(g, E, 2 * ff, d, std=d ** -0.5), down=_normal(g, E, d, ff, std=ff ** -0.5), norm=_normal(g, d, std=0.1, dtype=F32))


def _prepare_mamba(case, seed):
    g, lens = _gen(seed), _dealt(case, seed)
    H, P, N, G = case["heads"], case["vdim"], case["state"], case["groups"]
    inner, channels, T, B = H * P, H * P + 2 * G * N, sum(lens), case["batch"]
    params = dict(conv=_normal(g, 4, channels, std=0.5, dtype=F32), conv_b=_normal(g, channels, std=0.1, dtype=F32),
                  dt_bias=_normal(g, H, std=0.5, dtype=F32) - 3, neg_a=-torch.exp(_normal(g, H, dtype=F32)), d_skip=_normal(g, H, std=0.5, dtype=F32))
    return dict(case=case, lens=lens, proj=_normal(g, T, inner + channels + H), params=params,
                conv_state=torch.zeros(B, 4, channels, dtype=BF16, device=DEV), ssm_state=torch.zeros(B, H, N, P, dtype=F32, device=DEV),
                slots=_int32(list(range(B))), pos=torch.cat([torch.arange(n, dtype=torch.int32) for n in lens]).to(DEV),
                cu=_int32(_running(lens)), weight=_normal(g, inner, std=0.1, dtype=F32) + 1)


# ---- one pass ----------------------------------------------------------------------------------------------------------

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "decode":
        return ma.paged_attention_decode(s["q"], s["kc"], s["vc"], s["tables"], s["ctx"], k_scale=s["ks"], v_scale=s["vs"], max_context=s["bound"],
                                         workspace=s["workspace"], window=case["window"], keep_first=case["keep_first"])
    if kind == "prefill":
        q, k, v = s["q"], s["k"], s["v"]
        if case["packed"]:
            out = ma.flash_attn_varlen_prefill(q, k, v, s["cu"], s["cu"], s["longest"], s["longest"], window=case["window"],
                                               keep_first=case["keep_first"])
        else:
            out = ma.sdpa_slot(q, k, v, is_causal=True)
        if not case["train"]:
            return out
        dq, dk, dv = torch.autograd.grad(out, (q, k, v), s["dout"])
        return dict(out=out, dq=dq, dk=dk, dv=dv)
    if kind == "chunk":
        q, k, v, kc, vc = s["q"], s["k"], s["v"], s["kc"], s["vc"]
        if case["fp8"]:
            q = ma.rope_and_cache_fp8(q, k, v, s["pos"], s["freq"], kc, vc, s["ks"], s["vs"], s["slots"])
            out = ma.flash_attn_paged_prefill(q, kc, vc, s["cu"], s["tables"], s["ctx"], case["rows"], max_context=s["bound"], k_scale=s["ks"],
                                              v_scale=s["vs"], total_context=s["total"], cu_seqlens_k=s["cu_ctx"])
            return dict(out=out, kc=kc, vc=vc, ks=s["ks"], vs=s["vs"])
        q = ma.rope_and_cache(q, k, v, s["pos"], s["freq"], kc, vc, s["slots"])
        return dict(out=ma.flash_attn_paged_prefill(q, kc, vc, s["cu"], s["tables"], s["ctx"], case["rows"], max_context=s["bound"]), kc=kc, vc=vc)
    if kind == "serve":
        model = s["model"]
        sids = [model.new_sequence() for _ in s["prompts"]]
        logits = [model.prefill(sids, s["prompts"])]
        for tokens in s["given"]:
            logits.append(model.decode(sids, tokens))
        for i in sids:
            model.free_sequence(i)
        return torch.stack(logits)
    if kind == "moe":
        ids, weights, _ = ma.moe_route(s["h"], s["router"], s["bias"], case["top"])
        rows = ma.moe_experts(s["h"], ids, weights, s["gate_up"], s["down"])
        x, y = ma.residual_rms(None, s["norm"], sub=s["sub"], routed=rows, top=case["top"], weight_offset=1.0)
        return dict(ids=ids, weights=weights, rows=rows, x=x, y=y)
    inner = case["heads"] * case["vdim"]
    channels = inner + 2 * case["groups"] * case["state"]
    y = ma.ssm_mix(s["proj"], inner, inner + channels, s["params"], s["conv_state"], s["ssm_state"], s["slots"], s["pos"], s["cu"],
                   heads=case["heads"], vdim=case["vdim"], state=case["state"], groups=case["groups"])
    y = ma.gated_norm(y, s["proj"][:, :inner], s["weight"], 1, 1e-6, out=y)
    return dict(y=y, ssm_state=s["ssm_state"], conv_state=s["conv_state"])


# ---- what a pass cannot do without ---------------------------------------------------------------------------------------

def _visible(n, window, keep, before=0):
    """Pairs of a query and a key it sees: n causal queries behind `before` keys."""
    if not window:
        return n * before + n * (n + 1) // 2
    return sum(min(i + 1, window + max(0, min(keep, i + 1 - window))) for i in range(before, before + n))


def work(case):
    kind = case["kind"]
    if kind in ("decode", "prefill", "chunk"):
        H, G, D, lens = case["q_heads"], case["kv_heads"], case["head_dim"], _lengths(case)
    if kind == "decode":
        w, keep = case["window"], case["keep_first"]
        seen = [min(n, w + max(0, min(keep, n - w))) if w else n for n in lens]
        blocks = sum(-(-n // BLOCK) for n in seen)
        return dict(bytes=sum(seen) * 2 * G * D * (1 if case["fp8"] else 2) + 4 * blocks + (8 * G * blocks if case["fp8"] else 0) + 4 * len(lens) * H * D,
                    flops=4 * H * D * sum(seen))
    if kind == "prefill":
        T, pairs = sum(lens), sum(_visible(n, case["window"], case["keep_first"]) for n in lens)
        qk = 4 if case["amp"] else 2
        read_write = T * D * (qk * (H + G) + 2 * G + 2 * H)                  # q, k, v in, out
        if case["train"]:
            read_write += T * D * (2 * H + qk * (H + G) + 2 * G)             # dout in, dq, dk, dv out
        return dict(bytes=read_write, flops=4 * H * D * pairs * (7 if case["train"] else 2) // 2)    # two products forward, five backward
    if kind == "chunk":
        n, before = case["rows"], [-(-x // BLOCK) * BLOCK for x in lens]
        pairs, elem, new = sum(_visible(n, 0, 0, b) for b in before), 1 if case["fp8"] else 2, n * len(before)
        return dict(bytes=new * D * 2 * (2 * H + 2 * G) + 2 * G * D * elem * (sum(before) + new), flops=4 * H * D * pairs)
    if kind == "serve":
        d, ff, L, V, B = case["width"], case["ff"], case["layers"], case["vocab"], case["batch"]
        matrices = L * (4 * d * d + 3 * d * ff) + V * d
        lens = [_prompt(case, i) for i in range(B)]
        pairs = sum(_visible(n + case["steps"], 0, 0) for n in lens)
        cached = sum(n * case["steps"] + case["steps"] * (case["steps"] + 1) // 2 for n in lens)
        return dict(bytes=(1 + case["steps"]) * (2 * matrices + 4 * B * V) + cached * L * 4 * d,
                    flops=2 * (matrices - V * d) * (sum(lens) + B * case["steps"]) + 2 * V * d * B * (1 + case["steps"]) + 4 * d * L * pairs)
    if kind == "moe":
        T, d, E, ff, top = (case[n] for n in ("tokens", "width", "experts", "ff", "top"))
        used = E * (1 - (1 - top / E) ** T)                                  # experts that some token chooses, on average
        return dict(bytes=int(used * 6 * d * ff + 2 * E * d + T * d * (2 + 2 + 2 * top + 4 + 2)), flops=T * (6 * d * ff * top + 2 * E * d))
    H, P, N, G, T, B = case["heads"], case["vdim"], case["state"], case["groups"], sum(_lengths(case)), case["batch"]
    return dict(bytes=T * 2 * (2 * H * P + 2 * G * N + H + H * P) + B * (4 * H * N * P + 8 * (H * P + 2 * G * N)), flops=T * 4 * N * P * H)


def tolerance(case):
    # four times what the float64 results below are away, rounded up: bf16 operands and results, fp32 sums
    return {"decode": {"rel": 1e-2, "max": 0.1}, "prefill": {"rel": 1.5e-2, "max": 0.3}, "chunk": {"rel": 1.5e-2, "max": 0.3, "differ": 1e-4},
            "serve": {"rel": 3e-2, "max": 0.15}, "moe": {"rel": 1.5e-2, "max": 0.1, "differ": 1e-3}, "mamba": {"rel": 1.5e-2, "max": 0.3}}[case["kind"]]


# ---- the same in 64 bits -------------------------------------------------------------------------------------------------

def exact(case, seed):
    s = prepare(case, seed)
    with torch.no_grad():
        return {"decode": _exact_decode, "prefill": _exact_prefill, "chunk": _exact_chunk, "serve": _exact_serve, "moe": _exact_moe,
                "mamba": _exact_mamba}[case["kind"]](case, s)


def _seen(n_q, n_k, window, keep):
    """Keep-mask of the last n_q of n_k positions."""
    i, j = torch.arange(n_k - n_q, n_k, device=DEV)[:, None], torch.arange(n_k, device=DEV)[None]
    return (j <= i) if not window else (j <= i) & ((i - j < window) | (j < keep))


def _attend(q, k, v, window=0, keep=0):
    """One key head: q (group, n_q, D) the last n_q of the n_k positions of k, v (n_k, D), all float64."""
    n_q, n_k = q.shape[1], k.shape[0]
    sees = _seen(n_q, n_k, window, keep)
    return torch.stack([torch.softmax((h @ k.T / math.sqrt(k.shape[1])).masked_fill_(~sees, -math.inf), -1) @ v for h in q])


def _cached(cache, scale, table, n, head):
    """Rows 0..n-1 of one sequence and key head out of a pool, float64."""
    ids = table[:-(-n // BLOCK)].long()
    x = cache[ids, head]
    x = x.double() if scale is None else x.view(torch.float8_e4m3fn).double() * scale[ids, head].double()[:, None, None]
    return x.reshape(-1, x.shape[-1])[:n]


def _exact_decode(case, s):
    group = case["q_heads"] // case["kv_heads"]
    out = torch.empty(s["q"].shape, dtype=F64, device=DEV)
    for b, n in enumerate(s["lens"]):
        for h in range(case["kv_heads"]):
            k, v = (_cached(c, sc, s["tables"][b], n, h) for c, sc in ((s["kc"], s["ks"]), (s["vc"], s["vs"])))
            q = s["q"][b, h * group:(h + 1) * group].double()
            p = (q @ k.T / math.sqrt(case["head_dim"])).masked_fill_(~_seen(1, n, case["window"], case["keep_first"]), -math.inf)
            out[b, h * group:(h + 1) * group] = torch.softmax(p, -1) @ v
    return out


def _exact_prefill(case, s):
    """Attention and its gradients by the textbook formulas, a key head of a sequence at a time."""
    group, D, at = case["q_heads"] // case["kv_heads"], case["head_dim"], _running(s["lens"])
    names = ("out", "dq", "dk", "dv") if case["train"] else ("out",)
    like = dict(out=s["q"], dq=s["q"], dk=s["k"], dv=s["v"])
    res = {n: torch.empty(like[n].shape, dtype=F64, device=DEV) for n in names}
    for b, n in enumerate(s["lens"]):
        def part(t, h):
            return t[at[b]:at[b + 1], h] if case["packed"] else t[b, h]
        sees = _seen(n, n, case["window"], case["keep_first"])
        for g in range(case["kv_heads"]):
            k, v = part(s["k"], g).double(), part(s["v"], g).double()
            dk, dv = torch.zeros_like(k), torch.zeros_like(v)
            for h in range(g * group, (g + 1) * group):
                q = part(s["q"], h).double()
                p = torch.softmax((q @ k.T / math.sqrt(D)).masked_fill_(~sees, -math.inf), -1)
                o = p @ v
                part(res["out"], h).copy_(o)
                if case["train"]:
                    do = part(s["dout"], h).double()
                    dv += p.T @ do
                    ds = p * (do @ v.T - (do * o).sum(-1, keepdim=True)) / math.sqrt(D)
                    part(res["dq"], h).copy_(ds @ k)
                    dk += ds.T @ q
            if case["train"]:
                part(res["dk"], g).copy_(dk)
                part(res["dv"], g).copy_(dv)
    return res if case["train"] else res["out"]


def _rotate(x, cos, sin):
    """Adjacent pairs of x (T, heads, D) by the angles (T, D/2)."""
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack((a * cos[:, None] - b * sin[:, None], a * sin[:, None] + b * cos[:, None]), -1).reshape(x.shape)


def _exact_chunk(case, s):
    B, H, G, D, n = case["batch"], case["q_heads"], case["kv_heads"], case["head_dim"], case["rows"]
    cos, sin = (t[s["pos"].long()].double() for t in s["freq"])
    q = _rotate(s["q"].double(), cos, sin)
    new_k, new_v = _rotate(s["k"].double(), cos, sin).to(BF16), s["v"]              # rows as a bf16 cache holds them
    group, out = H // G, torch.empty(B * n, H, D, dtype=F64, device=DEV)

    def stored(rows, first):
        """(n, D) bf16 rows as the pool holds them."""
        if not case["fp8"]:
            return rows.double()
        pad = torch.cat((rows.float(), rows.new_zeros(-len(rows) % BLOCK, D).float())).view(-1, BLOCK, D)
        scale = pad.abs().amax((1, 2), keepdim=True) / 448.0
        return ((pad / scale).to(torch.float8_e4m3fn).double() * scale.double()).view(-1, D)[:len(rows)]

    for b, first in enumerate(s["before"]):
        rows = slice(b * n, (b + 1) * n)
        for g in range(G):
            k, v = (torch.cat((_cached(c, sc, s["tables"][b], first, g), stored(new[rows, g], first)))
                    for c, sc, new in ((s["kc"], s["ks"], new_k), (s["vc"], s["vs"], new_v)))
            heads = slice(g * group, (g + 1) * group)
            out[rows, heads] = _attend(q[rows, heads].transpose(0, 1), k, v).transpose(0, 1)
    return dict(out=out, kc=None, vc=None, **(dict(ks=None, vs=None) if case["fp8"] else {}))


def _exact_serve(case, s):
    """The decoder over every sequence's whole text; the logits that follow each prompt and each given token."""
    sd = {k: v.double() for k, v in s["sd"].items()}
    d, heads, steps = case["width"], case["heads"], case["steps"]
    hd = d // heads
    freq = ma.build_rope_cache(case["context"], hd, device=DEV).double()

    def norm(x, w):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-5) * w

    logits = []
    for i in range(case["batch"]):
        n = _prompt(case, i) + steps
        x = sd["token_embeddings.weight"][s["tokens"][i, :n].to(DEV)]
        for j in range(case["layers"]):
            pre = f"layers.{j}."
            h = norm(x, sd[pre + "attn_norm.weight"])
            q, k, v = ((h @ sd[f"{pre}attn.{m}.weight"].T).view(n, heads, hd) for m in ("q_proj", "k_proj", "v_proj"))
            q, k = _rotate(q, *freq[:, :n]), _rotate(k, *freq[:, :n])
            a = torch.stack([_attend(q[None, :, m], k[:, m].contiguous(), v[:, m].contiguous())[0] for m in range(heads)], 1)
            x = x + a.reshape(n, d) @ sd[pre + "attn.output_proj.weight"].T
            h = norm(x, sd[pre + "ffn_norm.weight"])
            f = torch.nn.functional.silu(h @ sd[pre + "ffn.gate_proj.weight"].T) * (h @ sd[pre + "ffn.up_proj.weight"].T)
            x = x + f @ sd[pre + "ffn.down_proj.weight"].T
        logits.append(norm(x[n - steps - 1:], sd["final_norm.weight"]) @ sd["lm_head.weight"].T)
    return torch.stack(logits, 1)


def _exact_moe(case, s):
    T, d, top, ff = case["tokens"], case["width"], case["top"], case["ff"]
    h = s["h"].double()
    chosen, ids = torch.topk(h @ s["router"].double().T + s["bias"].double(), top)
    weights = torch.softmax(chosen, -1)
    rows = torch.empty(T * top, d, dtype=F64, device=DEV)
    for e in range(case["experts"]):
        at = (ids.reshape(-1) == e).nonzero()[:, 0]
        if len(at):
            x = h[at // top]
            gate, up = (x @ w.T for w in s["gate_up"][e].double().split(ff))
            rows[at] = (torch.nn.functional.silu(gate) * up) @ s["down"][e].double().T * weights.reshape(-1)[at, None]
    x = s["sub"].double() + rows.view(T, top, d).sum(1)
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + 1e-6) * (1 + s["norm"].double())
    return dict(ids=ids.to(torch.int32), weights=weights, rows=rows, x=x, y=y)


def _exact_mamba(case, s):
    H, P, N, G = case["heads"], case["vdim"], case["state"], case["groups"]
    inner, channels = H * P, H * P + 2 * G * N
    p = {n: t.double() for n, t in s["params"].items()}
    proj, at = s["proj"].double(), _running(s["lens"])
    y = torch.empty(proj.shape[0], inner, dtype=F64, device=DEV)
    state = torch.empty(case["batch"], H, N, P, dtype=F64, device=DEV)
    for b, n in enumerate(s["lens"]):
        rows = proj[at[b]:at[b + 1]]
        x = torch.nn.functional.pad(rows[:, inner:inner + channels], (0, 0, 3, 0))
        x = torch.nn.functional.silu(sum(x[i:i + n] * p["conv"][i] for i in range(4)) + p["conv_b"])
        dt = torch.nn.functional.softplus(rows[:, inner + channels:] + p["dt_bias"])
        xh = x[:, :inner].view(n, H, P)
        B, C = (x[:, inner + i * G * N:inner + (i + 1) * G * N].view(n, G, N).repeat_interleave(H // G, 1) for i in range(2))
        S = torch.zeros(H, N, P, dtype=F64, device=DEV)
        decay = (p["neg_a"] * dt).cumsum(0)                                  # (n, H), in chunks of positions
        for first in range(0, n, 256):
            c = slice(first, min(n, first + 256))
            run, base = decay[c], decay[first - 1] if first else torch.zeros_like(decay[0])
            within = torch.exp((run.T[:, :, None] - run.T[:, None]).masked_fill_(~_seen(len(run), len(run), 0, 0), -math.inf))      # (H, i, j)
            Bc, Cc, xc = (t[c].transpose(0, 1).contiguous() for t in (B, C, xh * dt[:, :, None]))                                   # (H, i, .)
            out = (Cc @ Bc.transpose(1, 2).contiguous() * within) @ xc + torch.exp(run - base).T[:, :, None] * (Cc @ S)
            y[at[b] + first:at[b] + first + len(run)] = (out.transpose(0, 1) + p["d_skip"][:, None] * xh[c]).reshape(len(run), inner)
            last = run[-1]
            S = torch.exp(last - base)[:, None, None] * S + (Bc * torch.exp(last - run).T[:, :, None]).transpose(1, 2).contiguous() @ xc
        state[b] = S
    v = y * torch.nn.functional.silu(proj[:, :inner])
    y = v * torch.rsqrt(v.square().mean(-1, keepdim=True) + 1e-6) * s["weight"].double()
    return dict(y=y, ssm_state=state, conv_state=None)
