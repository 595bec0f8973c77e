"""fm_grouped_gemm_few (BF16, few tokens per expert) at the edges of its token passes
and K chunks, against float64: bf16 products are exact in fp32, so a sum over K is
off by at most K 2^-24 sum |terms|."""

import pytest
import torch

import nanopysche_amd as fm
from nanopysche_amd import _lib
from nanopysche_amd.flow_moe import ExpertWeightOperand, _Act, _dt, _gemm_m, _token_operand
from tests.helpers import randn_bf16

pytestmark = pytest.mark.gpu

COUNTS = [(1,), (0, 16, 1), (17, 0, 15, 32), (33, 5, 0, 0, 64), (140, 3)]


def _run(w, plan, tokens, out):
    out.fill_(7.0)
    _lib.call("fm_grouped_gemm_few", _token_operand(tokens, _lib.QUANT_BF16), w.operand(), int(w.kmajor),
              _lib.ptr(plan.counts), _lib.ptr(plan.offsets), plan.num_experts, w.N, w.K, _lib.ptr(out), _dt(out),
              out.stride(0), _lib.stream_of(out))
    return out


@pytest.mark.parametrize("form", ["nk", "nk_split", "kn", "kn_split"])
@pytest.mark.parametrize("counts", COUNTS)
@pytest.mark.parametrize("N,K", [(64, 64), (256, 128), (192, 448), (640, 1408)])
def test_matches_float64(dev, counts, N, K, form):
    E = len(counts)
    idx = torch.cat([torch.full((c,), e, dtype=torch.int64) for e, c in enumerate(counts)])[:, None].to(dev)
    plan = fm.route_tokens(idx, E)
    tokens = randn_bf16((plan.rows_max, K), seed=1).to(dev)
    W = randn_bf16((E, N, K), seed=2, std=0.1).to(dev)
    kn = form.startswith("kn")
    rows = W.transpose(1, 2).contiguous() if kn else W
    ld, n_rows = rows.shape[2], rows.shape[1]
    if form.endswith("split"):
        cut = n_rows // 128 * 64
        if not 0 < cut < n_rows:
            pytest.skip("too few rows to split")
        # equal group strides: pad the shorter part
        a, b = (torch.zeros(E, n_rows, ld, dtype=torch.bfloat16, device=dev) for _ in range(2))
        a[:, :cut], b[:, :n_rows - cut] = rows[:, :cut], rows[:, cut:]
        w = ExpertWeightOperand(a, None, ld, n_rows * ld, N=N, K=K, kmajor=kn, data2=b, split=cut)
    else:
        w = ExpertWeightOperand(rows, None, ld, n_rows * ld, N=N, K=K, kmajor=kn)
    f32 = _run(w, plan, tokens, torch.empty(plan.rows_max, N, device=dev))
    bf = _run(w, plan, tokens, torch.empty(plan.rows_max, N, dtype=torch.bfloat16, device=dev))
    offs = plan.offsets.tolist()
    for e, c in enumerate(counts):
        r = offs[e]
        x, we = tokens[r:r + c].double(), W[e].double()
        bound = K * 2.0 ** -24 * (x.abs() @ we.abs().t()) + 1e-30
        assert torch.all((f32[r:r + c].double() - x @ we.t()).abs() <= bound)
        assert torch.equal(bf[r:r + c], f32[r:r + c].bfloat16())
        for out in (f32, bf):
            assert torch.all(out[r + c:offs[e + 1]] == 0)
    assert torch.all(f32[offs[E]:] == 7.0)


@pytest.mark.parametrize("H", [128, 384])
def test_small_block_against_larger_tile(dev, H, monkeypatch):
    """A BF16 block of a few tokens, forward and backward, within bf16 rounding of the 256-row tile's."""
    from nanopysche_amd import flow_moe as fmm

    E, D, T = 6, 256, 21
    g = torch.Generator().manual_seed(H)
    idx = torch.stack([torch.randperm(E, generator=g)[:2] for _ in range(T)]).to(dev)
    leaves = [randn_bf16((T, D), seed=1), torch.rand(T, 2, generator=g),
              *(randn_bf16((E * H, D), seed=s, std=0.05) for s in (2, 3, 4))]
    got = []
    for limit in (128, 0):
        monkeypatch.setattr(fmm, "_FEW_TOKENS", limit)
        t = [v.to(dev).requires_grad_() for v in leaves]
        blk = fm.FP8FlowMoECompute(fm.FP8FlowMoEConfig(), D, H, E)
        blk.set_weights(*t[2:])
        out = blk(t[0], t[1], idx, 0, E)
        got.append((out.detach(), *torch.autograd.grad(out, t, torch.ones_like(out))))
    for a, b in zip(*got):
        assert (a.double() - b.double()).norm() <= 4e-3 * b.double().norm() + 1e-30


def test_forms_outside_the_rule_keep_their_kernel(dev, monkeypatch):
    """Pitches and alignments that only the tile entry takes go there, and what it refuses stays refused."""
    E, N, K = 2, 128, 128
    idx = torch.tensor([[0], [1], [1]], device=dev)
    plan = fm.route_tokens(idx, E)
    tokens = fm.fused_permute_pad(randn_bf16((3, K), seed=1).to(dev), plan, E, granularity=None).rows
    act = _Act(tokens, K, None, 0, False)   # as the block passes them
    W = randn_bf16((E, N, K), seed=2).to(dev)
    w = ExpertWeightOperand(W, None, K, N * K, N=N, K=K)
    ref = torch.empty(plan.rows_max, N, dtype=torch.bfloat16, device=dev)
    called, real = [], _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: (called.append(name), real(name, *a))[1])
    _gemm_m(_lib.QUANT_BF16, act, w, plan, ref)
    assert called == ["fm_grouped_gemm_few"]
    wide = torch.zeros(plan.rows_max, N + 4, dtype=torch.bfloat16, device=dev)[:, :N]     # pitch 4 mod 8
    _gemm_m(_lib.QUANT_BF16, act, w, plan, wide)
    assert called[1:] == ["fm_grouped_gemm_ragged_m"]
    for e, c in enumerate((1, 2)):
        r = int(plan.offsets[e])
        assert (wide[r:r + c].double() - ref[r:r + c].double()).norm() <= 4e-3 * ref[r:r + c].double().norm()
    narrow = ExpertWeightOperand(W[:, :64].contiguous(), None, K, 64 * K, N=64, K=K)
    with pytest.raises(RuntimeError, match="multiple of 128"):
        _gemm_m(_lib.QUANT_BF16, act, narrow, plan, ref)


@pytest.mark.parametrize("counts", [(3, 0, 1), (32, 17, 128)])
def test_public_gemm_multiplies_padding_rows(dev, counts):
    """fp8_grouped_gemm of a caller's buffer: every row of a group is multiplied, whatever
    its padding rows hold and however few the tokens."""
    E, N, K = len(counts), 256, 256
    idx = torch.cat([torch.full((c,), e, dtype=torch.int64) for e, c in enumerate(counts)])[:, None].to(dev)
    plan = fm.route_tokens(idx, E)
    tokens = randn_bf16((plan.rows_max, K), seed=1).to(dev)
    W = randn_bf16((E, N, K), seed=2, std=0.1).to(dev)
    out = fm.fp8_grouped_gemm(tokens, ExpertWeightOperand(W, None, K, N * K, N=N, K=K), plan, out_dtype=torch.float32)
    offs = plan.offsets.tolist()
    for e in range(E):
        x, we = tokens[offs[e]:offs[e + 1]].double(), W[e].double()
        bound = K * 2.0 ** -24 * (x.abs() @ we.abs().t()) + 1e-30
        assert torch.all((out[offs[e]:offs[e + 1]].double() - x @ we.t()).abs() <= bound)
