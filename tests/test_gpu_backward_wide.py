"""dK, dV and dS at head size 128 on wavefronts of 64 keys (key tiles with sixteen steps and more on average) against the form without dS in memory: rows and keys
around the tiles of 64 and 128 and their halves, a tile of rows that is the sequence's only one, wavefronts without keys or rows, more queries than keys
and the other way round, one to many steps, shares, fp32 gradients, several passes.  Tolerance of test_gpu_backward.py: one rounding of the result over a tensor."""
import pytest

from test_gpu_backward import _both_forms, _same_gradients, ops  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lens_q,lens_k,Hq,Hkv,causal", [
    ([1, 900, 33, 0, 830, 64, 65], None, 8, 1, True), ([31, 32, 33, 1800, 97, 95, 96], None, 16, 2, True), ([1700, 1, 129, 1023], [1800, 300, 64, 900], 6, 2, True),
    ([800, 1, 63, 900], [129, 64, 1, 127], 3, 1, False), ([2100, 2000], [40, 2100], 4, 4, True), ([700, 900, 64], [66, 193, 32], 4, 2, False),
    ([2113] * 5, None, 12, 12, True)])
def test_wide_packed(ops, monkeypatch, lens_q, lens_k, Hq, Hkv, causal):  # noqa: F811
    print(f"case: wide packed {lens_q} {lens_k} {Hq}/{Hkv} {causal}", flush=True)
    _same_gradients(*_both_forms(ops, monkeypatch, lens_q, lens_k or lens_q, Hq, Hkv, causal, True))


@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,causal,f32", [(3, 16, 2, 289, 289, True, True), (1, 12, 12, 2625, 2625, True, False), (2, 24, 3, 600, 130, False, False),
                                                       (5, 8, 8, 1700, 65, False, True), (9, 16, 1, 321, 500, True, False), (1, 32, 1, 1217, 1217, True, True)])
def test_wide_dense(ops, monkeypatch, B, Hq, Hkv, Sq, Sk, causal, f32):  # noqa: F811
    """(strided queries and gradients; one key head and several shares of its row tiles; fp32 gradients)"""
    print(f"case: wide dense {B} {Hq}/{Hkv} {Sq} {Sk} {causal}", flush=True)
    _same_gradients(*_both_forms(ops, monkeypatch, [Sq] * B, [Sk] * B, Hq, Hkv, causal, False, f32=f32))


@pytest.mark.parametrize("packed", [True, False])
def test_wide_in_passes(ops, monkeypatch, packed):  # noqa: F811
    print(f"case: wide in passes {packed}", flush=True)
    _same_gradients(*_both_forms(ops, monkeypatch, [1000] * 3, [1000] * 3, 28, 14, True, packed, workspace_part=0.45))
