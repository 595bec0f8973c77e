"""Entries without a device check of their own refuse CPU tensors where they ask for
the launch's stream, before the library is called (no GPU needed)."""

import pytest
import torch

import nanopysche_amd as fm
from nanopysche_amd import _lib
from nanopysche_amd.flow_moe import ExpertWeightOperand, ExpertWeights
from nanopysche_amd.norm import rmsnorm_backward
from nanopysche_amd.routing import RoutingPlan, expert_counts, load_balancing_loss


@pytest.fixture
def launched(monkeypatch):
    """A machine with a GPU, as far as the stream lookup sees it: -1 is the current device."""
    names = []
    monkeypatch.setattr(_lib, "call", lambda name, *a: names.append(name))
    monkeypatch.setattr(torch._C, "_cuda_getCurrentRawStream", lambda index: 4096 + index, raising=False)
    return names


def _i32(n):
    return torch.zeros(n, dtype=torch.int32)


def _grouped_gemm():
    plan = RoutingPlan(512, 1, 2, 768, _i32(2), _i32(3), _i32(512), _i32(768), _i32(6), _i32(2))
    w = ExpertWeightOperand(torch.zeros(2, 256, 256, dtype=torch.bfloat16), None, 256, 256 * 256, N=256, K=256)
    return fm.fp8_grouped_gemm(torch.zeros(768, 256, dtype=torch.bfloat16), w, plan)


def _mx_weights():
    w = [torch.zeros(2 * 128, 128, dtype=torch.bfloat16) for _ in range(3)]
    return ExpertWeights(_lib.QUANT_MX).refresh(*w, 2)


ENTRIES = {
    "fp8_grouped_gemm": _grouped_gemm,
    "mx_weights": _mx_weights,
    "expert_counts": lambda: expert_counts(torch.zeros(4, 2, dtype=torch.int64), 8),
    "load_balancing_loss": lambda: load_balancing_loss(torch.zeros(4, 8), _i32(8), 4),
    "rmsnorm_backward": lambda: rmsnorm_backward(torch.zeros(4, 512), torch.zeros(4, 512), torch.ones(512), torch.ones(4)),
}


@pytest.mark.parametrize("entry", ENTRIES)
def test_cpu_tensors_are_refused(launched, entry):
    with pytest.raises(ValueError, match="ROCm device"):
        ENTRIES[entry]()
    assert launched == []


@pytest.mark.parametrize("device", ["cpu", "meta"])
def test_no_stream_of_a_tensor_off_the_gpu(launched, device):
    with pytest.raises(ValueError, match="ROCm device"):
        _lib.stream_of(torch.empty(1, device=device))
