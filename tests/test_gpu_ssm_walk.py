"""The scan with outputs and state on different wavefronts (states of 64 or 128 rows, whole slices of vdim), at its edges: lengths around its blocks of 32
tokens and chunks of 128, resumed states, segments, sequences that stay whole among cut ones.  Bounds of test_gpu_zomipel.py: what rounding the
convolution's output and y to 8 bits leaves, and 1.5e-3 for the fp32 state from such inputs."""
import pytest
import torch

from test_gpu_zomipel import ops, rnd, rows_close, ssm_case, ssm_oracle, ssm_pools  # noqa: F401
from test_zomipel_host import conv_tile

pytestmark = pytest.mark.gpu
FORMS = [dict(heads=4, vdim=64, state=64, groups=2, taps=4), dict(heads=2, vdim=128, state=128, groups=1, taps=4), dict(heads=2, vdim=128, state=64, groups=2, taps=2)]


@pytest.mark.parametrize("m", FORMS, ids=lambda m: "-".join(str(v) for v in m.values()))
@pytest.mark.parametrize("segment", [0, 64, 128, 192])
def test_walk(ops, m, segment):  # noqa: F811
    """Every sequence in two calls, the second resumed where the first ended."""
    kw = {k: m[k] for k in ("heads", "vdim", "state", "groups")}
    lens, dtype = [1, 31, 32, 33, 127, 128, 129, 257, 390, 2], torch.bfloat16
    print(f"case: walk {m} {segment}", flush=True)
    case, params, xbc_at, dt_at = ssm_case(m, 1, 30, dtype)
    params["neg_a"] = params["neg_a"] * 0.1                               # long memories: what crosses an edge shows
    projs = [rnd(n, case.shape[1], seed=n, dtype=dtype) for n in lens]
    pc, sl = {k: v.cuda() for k, v in params.items()}, torch.randperm(len(lens) + 1, generator=torch.Generator().manual_seed(1))[:len(lens)].int()
    conv, state = ssm_pools(m, len(lens) + 1, dtype)
    cut, parts = [n // 3 for n in lens], []
    for a, b in (([0] * len(lens), cut), (cut, lens)):
        n = [y - x for x, y in zip(a, b)]
        got = ops.ssm_mix(torch.cat([p[x:y] for p, x, y in zip(projs, a, b)]).cuda(), xbc_at, dt_at, pc, conv, state, sl.cuda(),
                          torch.cat([torch.arange(x, y) for x, y in zip(a, b)]).int().cuda(), torch.tensor([0] + n).cumsum(0).int().cuda(), segment=segment, **kw)
        parts.append(torch.split(got.cpu(), n))
    for i, p in enumerate(projs):
        ref, S = ssm_oracle(m, p, params, xbc_at, dt_at, True)
        rows_close(torch.cat([parts[0][i], parts[1][i]]), ref, dtype, what=f"sequence {i}")
        s = state[int(sl[i])].cpu()[:, :, :m["vdim"]]
        assert float((s - S).pow(2).mean().sqrt() / S.pow(2).mean().sqrt()) <= 1.5e-3


def test_walk_of_whole_and_cut_sequences(ops):  # noqa: F811
    """A call of enough workgroups that long sequences are cut and the others walked whole, with states that are there already."""
    m = dict(heads=24, vdim=64, state=128, groups=1, taps=4)
    kw = {k: m[k] for k in ("heads", "vdim", "state", "groups")}
    lens, dtype = [5200, 300, 129, 640, 128, 40, 900, 100], torch.bfloat16
    print("case: walk, long ones cut", flush=True)
    assert ops.ops._ssm_plan(sum(lens), 8, 24, 64, 128, None) == (512, 2 * sum(lens) // 8)
    case, params, xbc_at, dt_at = ssm_case(m, 1, 31, dtype)
    projs = [rnd(n, case.shape[1], seed=n, dtype=dtype) for n in lens]
    pc, sl = {k: v.cuda() for k, v in params.items()}, torch.arange(8).int().cuda()
    args = (torch.cat(projs).cuda(), xbc_at, dt_at, pc)
    pos, cu = torch.cat([torch.arange(n) + 7 for n in lens]).int().cuda(), torch.tensor([0] + lens).cumsum(0).int().cuda()
    outs = []
    for segment in (None, 0):
        conv, state = (t * 1e-2 for t in ssm_pools(m, 8, dtype))
        state = state * 1e-4
        y = ops.ssm_mix(*args, conv, state, sl, pos, cu, segment=segment, **kw)
        outs.append((y.float().cpu(), state.cpu()))
    for a, b in zip(*outs):                               # fp32 sums in another order; y then rounded to 8 bits
        assert float((a - b).norm() / b.norm()) <= 1e-3


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_convolution_tiles(ops, tmp_path, dtype):  # noqa: F811
    """4, 8 and 16 tokens per thread, by the size of a call: two sequences of 2101 (fp32: 1501) tokens at once, in halves and in quarters with tokens left over; what
    is left in the ring is the same, the outputs but for the order of the scan's fp32 sums."""
    m = dict(heads=64, vdim=64, state=128, groups=1, taps=4)
    kw = {k: m[k] for k in ("heads", "vdim", "state", "groups")}
    print(f"case: convolution tiles {dtype}", flush=True)
    n = 2101 if dtype == torch.bfloat16 else 1501                         # (fp32 goes token by token behind the convolution)
    tile = conv_tile(tmp_path)
    assert [tile(2 * (n // parts), 64 * 64 + 2 * 128, 4) for parts in (1, 2, 4)] == [16, 8, 4]
    proj, params, xbc_at, dt_at = ssm_case(m, 2 * n, 32, dtype)
    proj, pc = proj.view(2, n, -1).cuda(), {k: v.cuda() for k, v in params.items()}
    outs = []
    for parts in (1, 2, 4):
        conv, state = ssm_pools(m, 2, dtype)
        cuts = [n * i // parts for i in range(parts + 1)]
        ys = [ops.ssm_mix(proj[:, a:b].reshape(2 * (b - a), -1), xbc_at, dt_at, pc, conv, state, torch.tensor([1, 0]).int().cuda(),
                          torch.arange(a, b).repeat(2).int().cuda(), torch.tensor([0, b - a, 2 * (b - a)]).int().cuda(), **kw).view(2, b - a, -1)
              for a, b in zip(cuts, cuts[1:])]
        outs.append((torch.cat(ys, 1).float().cpu(), conv.cpu()[:, [t % 4 for t in range(n - 3, n)]]))       # (the rows that a next token reads)
    for y, conv in outs[1:]:
        assert torch.equal(conv, outs[0][1])
        assert float((y - outs[0][0]).norm() / outs[0][0].norm()) <= 1e-3
