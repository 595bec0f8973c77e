"""BF16 expert weights read in place at hidden sizes that are odd multiples of
128: a 256-row weight tile then holds the end of w1 and the start of w3."""

import pytest
import torch

import nanopysche_amd as fm
from nanopysche_amd import _lib
from nanopysche_amd.flow_moe import ExpertWeightOperand
from tests.helpers import randn_bf16, zipf_routing

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("E,H,D,T,zeros", [(3, 128, 128, 300, ()), (8, 384, 256, 1500, (2,)), (5, 640, 384, 700, ())])
def test_split_inside_a_tile_matches_stacked(dev, E, H, D, T, zeros):
    """x [w1; w3]^T from the two tensors equals, bit for bit, that from their stack."""
    _, idx = zipf_routing(T, E, 2, 0.8, seed=H, zero_experts=zeros)
    w1, w3 = (randn_bf16((E * H, D), seed=s, std=0.02).to(dev) for s in (1, 2))
    x = randn_bf16((T, D), seed=3).to(dev)
    pt = fm.fused_permute_pad(x, idx.to(dev), E, granularity=None)
    stacked = torch.cat([w1.view(E, H, D), w3.view(E, H, D)], 1).contiguous()
    ref = ExpertWeightOperand(stacked, None, D, 2 * H * D, N=2 * H, K=D)
    two = ExpertWeightOperand(w1, None, D, H * D, N=2 * H, K=D, data2=w3, split=H)
    used = int(pt.plan.offsets[-1])
    for dt in (torch.bfloat16, torch.float32):
        a = fm.fp8_grouped_gemm(pt.rows, ref, pt.plan, out_dtype=dt)[:used]
        b = fm.fp8_grouped_gemm(pt.rows, two, pt.plan, out_dtype=dt)[:used]
        assert torch.equal(a, b)


@pytest.mark.parametrize("H", [128, 384, 1408])
def test_block_copies_no_weights(dev, H, monkeypatch):
    """A BF16 block of any hidden size (D a multiple of 256) gives the copying block's
    output and gradients without a weight launch."""
    E, D, T = 4, 256, 500
    w, idx = zipf_routing(T, E, 2, 0.8, seed=4)
    w1, w2, w3 = (randn_bf16((E * H, D), seed=s, std=0.02).to(dev) for s in (5, 6, 7))
    x, go = randn_bf16((T, D), seed=8).to(dev), randn_bf16((T, D), seed=9).to(dev)
    called, real = [], _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: (called.append(name), real(name, *a))[1])
    got = []
    for views in (True, False):
        monkeypatch.setattr(fm.ExpertWeights, "KMAJOR", views)
        called.clear()
        blk = fm.FP8FlowMoECompute(fm.FP8FlowMoEConfig(), D, H, E)
        leaves = [t.clone().requires_grad_() for t in (x, w.to(dev), w1, w2, w3)]
        blk.set_weights(*leaves[2:])
        out = blk(leaves[0], leaves[1], idx.to(dev), 0, E)
        got.append((out.detach(), *torch.autograd.grad(out, leaves, go)))
        assert ("fm_route_sort_weights" in called) == (not views)
    for a, b in zip(*got):
        assert torch.equal(a, b)
