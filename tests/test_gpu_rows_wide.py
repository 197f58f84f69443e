"""rows_linear with eight wavefronts (k of 1024 and more, up to 256 workgroups): the line between the two forms on either side, wavefronts with one, two and more steps,
remainders of k, edges of the row tiles.  Bound of test_gpu_model.py: one rounding of what is rounded."""
import pytest
import torch

from test_gpu_model import _close_rows, ops  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,k,n", [(1, 1016, 96), (1, 1024, 30), (16, 1032, 33), (17, 1024, 512), (32, 1096, 36), (9, 2048, 8192), (31, 1352, 8196), (32, 4096, 64),
                                   (8, 14336, 40), (33, 1024, 96), (70, 2056, 129), (3, 4096, 4112), (8, 1280, 72), (9, 1280, 40), (16, 1536, 96), (16, 2048, 40),
                                   (4, 1536, 4128), (4, 2048, 8192)])
def test_rows_linear_on_eight_wavefronts(ops, T, k, n):  # noqa: F811
    print(f"case: rows on eight wavefronts {T} {k} {n}", flush=True)
    g, prompt = torch.Generator().manual_seed(T + k), T > 32

    def t(*shape, std=1.0):
        return (torch.randn(*shape, generator=g) * std).to(torch.bfloat16).cuda()

    x, w, resid = t(T, k), t(2 * n, k, std=k ** -0.5), t(T, n + 4)[:, :n]
    xd, wd, one = x.double(), w.double(), w[:n].contiguous()
    _close_rows(ops.rows_linear(x, one, out_dtype=torch.float32, prompt=prompt), xd @ wd[:n].T, 0, "fp32")
    _close_rows(ops.rows_linear(x, one, resid=resid, prompt=prompt), xd @ wd[:n].T + resid.double(), 1, "add")
    if k <= 4096:
        norm = (torch.randn(k, generator=g) * 0.3 + 1).cuda()
        normed = xd * torch.rsqrt(xd.square().mean(-1, keepdim=True) + 1e-5) * norm.double()
        gate, up = (normed @ wd.T).split(n, 1)
        _close_rows(ops.rows_linear(x, one, norm=norm, prompt=prompt), normed @ wd[:n].T, 1, "norm")
        _close_rows(ops.rows_linear(x, w, norm=norm, gate_up=True, prompt=prompt), torch.nn.functional.silu(gate) * up, 3, "gate_up")
