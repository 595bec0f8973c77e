"""The expert block's backward reads its saved tensors in the layout and type that a
saved-tensor hook returns them in (no GPU: the launches' arguments are looked at)."""

import contextlib
import ctypes
import types

import pytest
import torch

import nanopysche_amd.flow_moe as fmm
from nanopysche_amd import _lib
from nanopysche_amd.recipes import FP8RecipeConfig, FP8RecipeType

E, H, D, T, K = 4, 256, 256, 64, 2


@pytest.mark.parametrize("recipe", ["flow_moe", "blockwise", "mxfp8", "none"])
@pytest.mark.parametrize("turned", [False, True])
def test_backward_takes_what_the_hook_returns(monkeypatch, recipe, turned):
    calls = []

    def call(name, *a):
        if name == "fm_permute" and a[7] is not None:   # the router weights that scale dY's rows
            calls.append((name, list((ctypes.c_float * (T * K)).from_address(a[7]))))
        elif name == "fm_swiglu_backward":
            calls.append((name, a[:4]))

    monkeypatch.setattr(_lib, "call", call)
    monkeypatch.setattr(_lib, "require_device", lambda *a: None)
    monkeypatch.setattr(_lib, "stream_of", lambda t: 0)
    monkeypatch.setattr(fmm, "_cus", lambda dev: 256)
    stream = types.SimpleNamespace(wait_stream=lambda other: None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda dev: stream)
    monkeypatch.setattr(torch.cuda, "stream", lambda s: contextlib.nullcontext())
    blk = fmm.FP8FlowMoECompute(fmm.FP8FlowMoEConfig(True, FP8RecipeConfig(recipe != "none", FP8RecipeType(recipe))),
                                D, H, E, fp8_gemm_threshold=0)
    blk.overlap_streams = False
    blk.set_weights(*(torch.randn(E * H, D).bfloat16() for _ in range(3)))
    blk._record = True
    saved = []
    ctx = types.SimpleNamespace(needs_input_grad=(True,) * 7, save_for_backward=lambda *a: saved.extend(a))
    weights = torch.rand(T, K)
    blk._forward(ctx, torch.randn(T, D).bfloat16(), weights, *blk._w, torch.randint(0, E, (T, K)))
    wts, GU, Y = saved
    if turned:
        wts = wts.double().t().contiguous().t()
        GU = torch.cat((GU, GU[:, :64]), dim=1)[:, :2 * H]
        Y = torch.cat((Y, Y[:, :64]), dim=1)[:, :D]
    ctx.saved_tensors, ctx.shape = (wts, GU, Y), (T, D)
    calls.clear()
    blk._backward(ctx, torch.randn(T, D))
    assert [n for n, _ in calls] == ["fm_permute", "fm_swiglu_backward"]
    assert calls[0][1] == weights.flatten().tolist()
    at, ld = GU.data_ptr(), 2 * H + (64 if turned else 0)
    assert calls[1][1] == (at, ld, at + 2 * H, ld)
