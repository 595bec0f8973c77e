"""The expert block refuses indices and weights that do not fit its tokens before it
launches anything (no GPU: the library is not reached)."""

import types

import pytest
import torch

import nanopysche_amd.flow_moe as fmm
from nanopysche_amd import _lib
from nanopysche_amd.recipes import FP8RecipeConfig, FP8RecipeType


@pytest.fixture
def launched(monkeypatch):
    names = []
    monkeypatch.setattr(_lib, "call", lambda name, *a: names.append(name))
    monkeypatch.setattr(_lib, "require_device", lambda *a: None)
    monkeypatch.setattr(_lib, "stream_of", lambda t: 0)
    return names


@pytest.mark.parametrize("recipe", ["flow_moe", "blockwise", "mxfp8", "none"])
@pytest.mark.parametrize("rows_of,n", [("indices", 65), ("indices", 63), ("both", 96), ("weights", 63)])
def test_rows_that_do_not_fit_are_refused(launched, recipe, rows_of, n):
    E, H, D, T, K = 4, 256, 256, 64, 2
    blk = fmm.FP8FlowMoECompute(fmm.FP8FlowMoEConfig(True, FP8RecipeConfig(recipe != "none", FP8RecipeType(recipe))),
                                D, H, E, fp8_gemm_threshold=0)
    blk.set_weights(*(torch.randn(E * H, D).bfloat16() for _ in range(3)))
    idx = torch.randint(0, E, (n if rows_of in ("indices", "both") else T, K))
    w = torch.rand(n if rows_of in ("weights", "both") else T, K)
    with pytest.raises(ValueError, match=f"are for {n} tokens, x has {T}"):
        blk(torch.randn(T, D).bfloat16(), w, idx)
    assert launched == []


def test_rows_that_fit_are_launched(launched):
    """The same call with matching rows goes on to its launches, weights first."""
    E, H, D, T, K = 4, 256, 256, 64, 2
    blk = fmm.FP8FlowMoECompute(fmm.FP8FlowMoEConfig(True, FP8RecipeConfig(True, FP8RecipeType("flow_moe"))),
                                D, H, E, fp8_gemm_threshold=0)
    blk.set_weights(*(torch.randn(E * H, D).bfloat16() for _ in range(3)))
    blk._record = False
    ctx = types.SimpleNamespace(needs_input_grad=(False,) * 7, save_for_backward=lambda *a: None)
    blk._forward(ctx, torch.randn(T, D).bfloat16(), torch.rand(T, K), *blk._w, torch.randint(0, E, (T, K)))
    assert launched[0] == "fm_route_sort_weights" and launched[-1] == "fm_unpermute"
