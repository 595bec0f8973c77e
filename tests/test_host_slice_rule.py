"""The slice count of a ragged-M launch of few tiles (csrc/fm_slices.h) is worked out
by two kernels and has to be the same in both: compiled with and without fused
multiply-adds it is, and it is the cheapest count of its cost model in exact arithmetic,
the largest of equals."""

import ctypes
import subprocess
import types
from fractions import Fraction
from itertools import product
from pathlib import Path

import pytest

import nanopysche_amd.flow_moe as fmm
from nanopysche_amd import _lib

CSRC = Path(__file__).resolve().parents[1] / "nanopysche_amd" / "csrc"
SOURCE = f"""
#include "{CSRC / 'fm_slices.h'}"
extern "C" void counts(int nk, int bf16, int tiles, int* out) {{   // of 1 .. tiles tiles, 32 workgroups an XCD
  for (int n = 1; n <= tiles; ++n) out[n - 1] = fm::slice_count(n, 32 / ((n + 7) / 8), nk, bf16 != 0);
}}
extern "C" int count(int nk, int bf16, int tiles, int workgroups) {{
  return fm::slice_count(tiles, workgroups / 8 / ((tiles + 7) / 8), nk, bf16 != 0);
}}
"""


@pytest.fixture(scope="module")
def built(tmp_path_factory):
    d = tmp_path_factory.mktemp("slices")
    (d / "slices.cpp").write_text(SOURCE)
    libs = []
    for name, flags in (("fused", ["-mfma", "-ffp-contract=fast"]), ("unfused", ["-ffp-contract=off"])):
        so = d / f"{name}.so"
        subprocess.run(["g++", "-O3", "-shared", "-fPIC", *flags, "-D__device__=", "-D__forceinline__=inline",
                        str(d / "slices.cpp"), "-o", str(so)], check=True)
        libs.append(ctypes.CDLL(str(so)))
    return libs


def _counts(lib, nk, bf16, tiles=256):
    out = (ctypes.c_int * tiles)()
    lib.counts(nk, int(bf16), tiles, out)
    return list(out)


def _best(tiles, nk, bf16):
    by_cu, by_k = 32 // ((tiles + 7) // 8), nk // 8
    launch, part = (Fraction(5), Fraction(tiles, 14)) if bf16 else (Fraction(13, 2), Fraction(tiles, 11))
    cost = {1: Fraction(nk)}
    cost.update({s: Fraction(nk, s) + launch + part * s for s in range(2, 9) if s <= by_cu and s <= by_k})
    least = min(cost.values())
    return 1 if cost[1] == least else max(s for s, c in cost.items() if c == least)


@pytest.mark.parametrize("bf16", [True, False])
def test_both_builds_and_exact_arithmetic_agree(built, bf16):
    for nk in (2, 15, 16, 20, 32, 34, 53, 64, 88, 112, 128, 224, 448, 4096):
        a, b = (_counts(lib, nk, bf16) for lib in built)
        assert a == b == [_best(n, nk, bf16) for n in range(1, 257)]


def test_counts_of_equal_cost(built):
    """BF16, 16 tiles of 64 steps and 32 of 128: 7 and 8 slices cost the same."""
    for nk, tiles in ((64, 16), (128, 32)):
        assert [_counts(lib, nk, True)[tiles - 1] for lib in built] == [8, 8]


@pytest.mark.parametrize("kind", [_lib.QUANT_BF16, _lib.QUANT_POW2])
def test_the_workspace_does_not_change_the_count(built, kind):
    """With the slots that the host allocates (a workgroup each), every number of tiles that the
    plan can hold gets the slices that 256 workgroups would give it, in as many slots."""
    bf16 = kind == _lib.QUANT_BF16
    sizes = set()
    for E, tokens, N, steps in product((1, 4, 8), (64, 200, 700), (256, 384, 1024, 4096), (20, 34, 64, 88, 224)):
        m_tiles = -(-tokens // 128) + E
        plan = types.SimpleNamespace(m_tiles=m_tiles, num_experts=E)
        w = types.SimpleNamespace(N=N, K=steps * (64 if bf16 else 128))
        slots = fmm._slice_slots(kind, plan, w, 256)
        sizes.add(slots)
        assert slots % 8 == 0 and slots <= 256
        for tiles in range(1, min(256, (m_tiles + E + 1) // 2 * -(-N // 256)) + 1):
            n = built[0].count(steps, int(bf16), tiles, slots)
            assert n == built[0].count(steps, int(bf16), tiles, 256)
            assert n == 1 or -(-tiles // 8) * 8 * n <= slots
    assert min(sizes) == 16 and max(sizes) == 256
