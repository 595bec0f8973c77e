"""The slice count of a ragged-M launch of few tiles (csrc/fm_slices.h) is worked out
by two kernels and has to be the same in both: compiled with and without fused
multiply-adds it is, and it is the cheapest count of its cost model in exact arithmetic,
the largest of equals."""

import ctypes
import subprocess
from fractions import Fraction
from pathlib import Path

import pytest

CSRC = Path(__file__).resolve().parents[1] / "nanopysche_amd" / "csrc"
SOURCE = f"""
#include "{CSRC / 'fm_slices.h'}"
extern "C" void counts(int nk, int bf16, int tiles, int* out) {{   // of 1 .. tiles tiles, 32 workgroups an XCD
  for (int n = 1; n <= tiles; ++n) out[n - 1] = fm::slice_count(n, 32 / ((n + 7) / 8), nk, bf16 != 0);
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
