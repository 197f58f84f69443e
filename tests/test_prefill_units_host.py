"""The order of a launch's query tiles over the eight XCDs, checked on the CPU."""
import ctypes
import os
import subprocess

import pytest

import mi355_attn


@pytest.fixture(scope="module")
def order(tmp_path_factory):
    d = tmp_path_factory.mktemp("units")
    src, lib = d / "units.cpp", d / "units.so"
    src.write_text('#include "xcd_order.hpp"\n'
                   'extern "C" int units(int u, int group, int groups, int chunk, int round, int* out) {\n'
                   '  const int n = mi355::xcd_units_grid(u, group, groups);\n'
                   '  for (int i = 0; out && i < n; ++i) { const auto x = mi355::xcd_unit(i, u, group, groups, chunk, round); out[2 * i] = x.unit; out[2 * i + 1] = x.head; }\n'
                   '  return n; }\n'
                   'extern "C" int fits(long long u, long long group, long long groups, int threads) { return mi355::xcd_units_fit(u, group, groups, threads); }\n'
                   'extern "C" int spread(int groups, int n_split) { return mi355::xcd_units_spread(groups, n_split); }\n')
    csrc = os.path.join(os.path.dirname(os.path.dirname(mi355_attn.__file__)), "csrc")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-I", csrc, str(src), "-o", str(lib)], check=True)
    fn = ctypes.CDLL(str(lib)).units
    fits = ctypes.CDLL(str(lib)).fits
    fits.argtypes = [ctypes.c_longlong] * 3 + [ctypes.c_int]

    def units(u, group, groups, chunk, rnd):
        n = fn(u, group, groups, chunk, rnd, None)
        out = (ctypes.c_int * (2 * n))()
        fn(u, group, groups, chunk, rnd, out)
        return [(out[2 * i], out[2 * i + 1]) for i in range(n)]
    units.grid = lambda u, group, groups: fn(u, group, groups, 1, 0, None)
    units.fits, units.spread = fits, ctypes.CDLL(str(lib)).spread
    return units


@pytest.mark.parametrize("rnd", [0, 32])
@pytest.mark.parametrize("group", [1, 4, 5])
@pytest.mark.parametrize("u,groups", [(1, 1), (1, 8), (3, 7), (2, 9), (11, 16), (6, 37), (64, 8), (5, 129)])
def test_every_unit_once(order, u, groups, group, rnd):
    """Every unit of every head has one workgroup, and at most seven more have none; an XCD (workgroup modulo 8) keeps to its own kv heads beyond the first
    groups % 8 of them, takes whole chunks, and begins a chunk's units in order."""
    for chunk in {group, group * max(1, groups // 16), group * max(1, groups // 8)}:
        got = order(u, group, groups, chunk, rnd)
        work = [x for x in got if x[0] >= 0]
        assert len(got) - len(work) <= 7
        assert sorted(work) == sorted((i, h) for i in range(u) for h in range(group * groups))
        front = -(-(groups % 8 * group * u) // 8) * 8
        assert all(h >= groups // 8 * 8 * group for i, h in got[:front] if i >= 0)
        for xcd in range(8):
            mine = got[front + xcd::8]
            assert {h // group % 8 for _, h in mine} <= {xcd}
            if rnd == 0:
                for c in range(0, len(mine), chunk * u):
                    units = [i for i, _ in mine[c:c + chunk * u]]
                    assert units == sorted(units) and len({h for _, h in mine[c:c + chunk * u]}) <= chunk


@pytest.mark.parametrize("group", [1, 4, 5])
@pytest.mark.parametrize("u,groups,n_split", [(1, 1, 30), (1, 2, 16), (6, 12, 5), (2, 3, 64), (3, 16, 4), (1, 8, 20), (5, 9, 1), (4, 37, 3)])
def test_shares_of_split_keys_reach_every_xcd(order, u, groups, group, n_split):
    """Workgroups of a launch whose shares follow each other, single tiles by number where the rule says so, else in order without a gap: no XCD (id modulo 8) gets
    more than one of those with work more than another."""
    ids = [i >= 0 for i, _ in order(u, group, groups, group, 0)] if order.spread(groups, n_split) else [True] * (u * group * groups)
    with_work = [sum((ids * n_split)[xcd::8]) for xcd in range(8)]
    assert sum(with_work) == u * group * groups * n_split and max(with_work) - min(with_work) <= 1


@pytest.mark.parametrize("D,prompt,chunk", [(32, 1, 2), (64, 1, 2), (128, 2, 2)])
def test_two_shares_of_a_whole_prompt(D, prompt, chunk):
    """Heads of 32 and 64: whole prompts are not cut in two, chunks and calls with per-head terms still are, and four shares stay."""
    from mi355_attn import _lib
    lib = _lib.load()
    assert lib.mi355_prefill_suggest_prompt_kv_splits(1, 8, D, 8192, 8192, 8192, 1, 256) == prompt
    assert lib.mi355_prefill_suggest_kv_splits(1, 8, D, 8192, 8192, 8192, 1, 256) == chunk
    assert lib.mi355_prefill_suggest_prompt_kv_splits(1, 4, D, 8192, 8192, 8192, 1, 256) == 4


@pytest.mark.parametrize("threads", [256, 512])
def test_grids_of_single_units_stay_below_the_threads_of_a_launch(order, threads):
    """A grid's threads are counted in 32 bits.  Where single units are said to fit, the grid with its empty workgroups has fewer; where they are not, it is within
    seven workgroups of that, or beyond."""
    most = (1 << 32) // threads
    for u, group, groups in ((1, 1, most - 1), (1, 1, most - 9), (1, 1, most // 2), (2, 1, most // 2 - 1), (3, 4, most // 12 - 1), (3, 4, most // 12 + 1), (7, 1, 9)):
        if order.fits(u, group, groups, threads):
            assert order.grid(u, group, groups) * threads < 1 << 32
        else:
            assert (u * group * groups + 7) * threads >= 1 << 32
    assert not order.fits(1 << 20, 64, 1 << 20, threads)


def named(B, Hq, Hkv, D, Sq, Sk, mask=1, packed=0, blocks=0, lse=0, split=1, window=0):
    from mi355_attn import _lib
    waves = ctypes.c_int(0)
    kernel = _lib.load().mi355_prefill_kernel(B, Hq, Hkv, D, Sq, Sk, mask, packed, blocks, lse, split, window, 256, ctypes.byref(waves))
    return kernel, waves.value


TILES, W64, SHORT, KEYS = 1, 2, 3, 4


def test_launches_beyond_a_grid_stay_with_the_persistent_kernel():
    """Dense calls of head size 128 with 2^24 workgroups of 32 rows and more: more threads than a launch counts, but for the kernel that takes any number of tiles."""
    assert named(1 << 19, 31, 31, 128, 32, 32) == (KEYS, 4)
    assert named(1 << 19, 32, 32, 128, 32, 32) == named(1 << 20, 16, 16, 128, 32, 32) == named(1 << 19, 64, 32, 128, 20, 20, mask=0) == named(1 << 17, 128, 128, 128, 1, 32, lse=1) == (W64, 4)
    assert named(0, 1, 1, 128, 1, 1)[0] == named(1, 3, 2, 128, 1, 1)[0] == named(1, 1, 1, 96, 1, 1)[0] == 0


def test_calls_of_heads_of_32_and_64_go_where_they_are_faster():
    """Both sides of the lines between the kernels, as measured (us): short heads against keys dealt, keys dealt against query tiles, four wavefronts against eight."""
    for B, Hq, Hkv, D, S in ((16, 64, 16, 64, 68), (64, 8, 8, 64, 73), (32, 8, 2, 64, 158), (8, 64, 16, 64, 74), (16, 16, 8, 32, 67)):
        assert named(B, Hq, Hkv, D, S, S)[0] == SHORT          # 11.1 / 17.1, 6.9 / 10.5, 8.0 / 12.1, 6.6 / 10.0, 4.8 / 5.6
    for B, Hq, Hkv, D, S, mask in ((1, 16, 16, 64, 165, 0), (2, 4, 1, 64, 238, 1), (8, 1, 1, 64, 195, 0), (2, 16, 16, 32, 208, 1), (1, 4, 1, 32, 199, 0)):
        assert named(B, Hq, Hkv, D, S, S, mask) == (KEYS, 4)  # 6.0 / 9.8, 5.4 / 9.2, 6.0 / 10.4, 5.2 / 7.0, 4.9 / 7.7
    for B, Hq, Hkv, S, lse in ((32, 8, 4, 312, 1), (64, 4, 2, 303, 1), (16, 16, 16, 305, 1)):
        assert named(B, Hq, Hkv, 64, S, S, lse=lse) == (TILES, 4)                         # 17.6 / 22.4, 17.4 / 22.6, 18.1 / 22.0
    assert named(64, 8, 1, 64, 191, 191, packed=1, lse=1) == (TILES, 4)                   # 18.0 / 23.7
    for B, Hq, Hkv, D, S in ((1, 16, 16, 32, 7093), (3, 16, 4, 64, 933), (4, 32, 4, 64, 970), (8, 8, 4, 32, 2769)):
        assert named(B, Hq, Hkv, D, S, S, 0, lse=1) == (TILES, 8)                         # 151 / 164, 24 / 26, 44 / 46, 94 / 99
    for B, Hq, Hkv, D, S in ((24, 4, 4, 32, 1309), (1, 32, 4, 64, 2658), (3, 8, 8, 64, 5902)):
        assert named(B, Hq, Hkv, D, S, S, 0, lse=1) == (TILES, 4)                         # 45.7 / 50.3, 79 / 89, 256 / 278


def test_packed_heads_of_128_with_lengths_far_apart_stay_with_the_wide_kernel():
    """Lengths on the device may be far shorter than the longest, which then waits for its heads on their dies: four wavefronts only where they win either way (us wide / tiles)."""
    for B, Hq, Hkv, S, mask in ((2, 8, 4, 4480, 0), (8, 4, 1, 2779, 0), (2, 16, 16, 2448, 0), (12, 8, 2, 1119, 0), (3, 4, 1, 6731, 0)):
        assert named(B, Hq, Hkv, 128, S, S, mask, packed=1) == (W64, 4)               # 108 / 207, 75 / 124, 75 / 108, 45 / 63, 156 / 172
    assert named(6, 16, 16, 128, 708, 1442, blocks=91) == named(12, 8, 1, 128, 754, 1556, blocks=98) == (W64, 4)   # 63 / 91, 55 / 71
    for B, Hq, Hkv, S, mask in ((60, 16, 16, 300, 1), (24, 4, 4, 248, 0), (32, 32, 16, 119, 0), (6, 8, 8, 981, 1), (2, 16, 16, 1286, 1)):
        assert named(B, Hq, Hkv, 128, S, S, mask, packed=1) == (TILES, 4)             # 97 / 44, 27 / 13, 57 / 20, 41 / 31, 48 / 37
