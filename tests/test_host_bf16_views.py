"""Which BF16 parameters the expert block's GEMMs read in place (no GPU needed)."""

import contextlib
import types

import pytest
import torch

import nanopysche_amd.flow_moe as fmm
from nanopysche_amd import _lib
from nanopysche_amd.flow_moe import ExpertWeights


def _at(elements, *shape):
    """A contiguous bf16 tensor that starts so many elements past a 16-byte boundary."""
    n = 1
    for s in shape:
        n *= s
    flat = torch.zeros(n + 16, dtype=torch.bfloat16)
    start = (-flat.data_ptr() % 16) // 2 + elements
    return flat[start:start + n].view(*shape)


@pytest.mark.parametrize("H", [128, 256, 384, 512])
@pytest.mark.parametrize("which", [None, 0, 1, 2])
@pytest.mark.parametrize("elements", [1, 4])
def test_parameters_off_16_bytes_are_copied(H, which, elements):
    E, D = 2, 256
    ws = [_at(elements if i == which else 0, E * H, D) for i in range(3)]
    assert [w.data_ptr() % 16 != 0 for w in ws] == [i == which for i in range(3)]
    jobs = []
    ew = ExpertWeights(_lib.QUANT_BF16, paired=True).refresh(*ws, E, True, defer=jobs)
    in_place = ew.w13.data2 is not None
    assert in_place == (which is None) and (jobs == []) == (which is None)
    for op in (ew.w13, ew.w2t, ew.w2, ew.w13t):
        assert op.data.data_ptr() % 16 == 0 and (op.data2 is None or op.data2.data_ptr() % 16 == 0)


@pytest.mark.parametrize("H", [128, 256, 384])
@pytest.mark.parametrize("which", [0, 1, 2])
def test_weights_changed_after_the_forward_are_refused(monkeypatch, H, which):
    """A backward whose operands are the parameters raises, as autograd does for a saved
    tensor, when one was changed in place since its forward; copied operands hold the
    forward's weights and go on."""
    E, D, T, K = 2, 256, 64, 1
    launched = []
    monkeypatch.setattr(_lib, "call", lambda name, *a: launched.append(name))
    monkeypatch.setattr(_lib, "require_device", lambda *a: None)
    monkeypatch.setattr(_lib, "stream_of", lambda t: 0)
    monkeypatch.setattr(fmm, "_cus", lambda dev: 256)
    for in_place in (True, False):
        ws = [_at(0 if in_place else 1, E * H, D) for _ in range(3)]
        blk = fmm.FP8FlowMoECompute(fmm.FP8FlowMoEConfig(), D, H, E)
        blk.set_weights(*ws)
        ctx = types.SimpleNamespace(needs_input_grad=(True, False) + (True,) * 5)
        ctx.save_for_backward = lambda *a: setattr(ctx, "saved_tensors", a)
        x, w = torch.zeros(T, D, dtype=torch.bfloat16), torch.rand(T, K)
        blk._forward(ctx, x, w, *ws, torch.randint(0, E, (T, K)))
        ws[which].add_(1)
        launched.clear()
        if in_place:
            with pytest.raises(RuntimeError, match="after the forward"):
                blk._backward(ctx, torch.zeros(T, D, dtype=torch.bfloat16))
            assert launched == []
        else:
            blk.overlap_streams = False
            stream = types.SimpleNamespace(wait_stream=lambda s: None)
            monkeypatch.setattr(torch.cuda, "current_stream", lambda dev=None: stream)
            monkeypatch.setattr(torch.cuda, "stream", lambda s: contextlib.nullcontext())
            blk._backward(ctx, torch.zeros(T, D, dtype=torch.bfloat16))
            assert launched
