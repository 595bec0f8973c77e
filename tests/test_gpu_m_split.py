"""Ragged-M GEMM whose few tiles are cut in slices of K, against float64 (BF16): bf16
products are exact in fp32, so a sum over K, in slices or not, is off by at most
K 2^-24 sum |terms|, and the bf16 output by half a unit of its last place more."""

import pytest
import torch

import nanopysche_amd as fm
from nanopysche_amd import _lib
from nanopysche_amd.flow_moe import ExpertWeightOperand, ExpertWeights, _gemm_kind, _gemm_m, _m_split, _token_operand
from tests.helpers import randn_bf16

pytestmark = pytest.mark.gpu


def _slots_written(ws):
    """256 KiB partials that hold anything, in a workspace that was all NaN."""
    return int((~torch.isnan(ws).view(-1, 65536)).any(dim=1).sum())


@pytest.mark.parametrize("form", ["nk", "nk_split", "kn", "kn_split"])
@pytest.mark.parametrize("counts,masked,K,groups,slots", [
    ((300, 0, 1, 257), False, 4224, 32, 10 * 8),   # 2 x 5 tiles of 66 steps in 8 slices; an expert without tokens
    ((130, 600, 20, 90), True, 4096, 32, 8 * 8),   # every second expert: 2 x 4 tiles of 64 steps
    ((700, 300), False, 4096, 1, 0),               # 8 workgroups for 5 tiles of one column: not sliced
    ((520,), False, 2176, 2, 3 * 2),               # 3 tiles of 34 steps in two slices of 17
])
def test_matches_float64(dev, counts, masked, K, groups, slots, form):
    E, N = len(counts), 256 if groups < 32 else 512
    idx = torch.cat([torch.full((c,), e, dtype=torch.int64) for e, c in enumerate(counts)])[:, None].to(dev)
    plan = fm.route_tokens(idx, E)
    offs = plan.offsets.tolist()
    tokens = randn_bf16((plan.rows_max, K), seed=1).to(dev)
    W = randn_bf16((E, N, K), seed=2, std=0.1).to(dev)
    kn = form.startswith("kn")
    rows = W.transpose(1, 2).contiguous() if kn else W
    kw = {}
    if form.endswith("split"):
        cut = K // 256 * 128 if kn else 128   # [N][K]: inside a 256-row tile
        b = torch.zeros_like(rows)
        b[:, :rows.shape[1] - cut] = rows[:, cut:]
        kw = dict(data2=b, split=cut)
        rows = rows.clone()
        rows[:, cut:] = float("nan")   # the second part comes from data2
    w = ExpertWeightOperand(rows, None, rows.shape[2], N * K, N=N, K=K, kmajor=kn, **kw)
    mask = torch.tensor([e % 2 for e in range(E)], dtype=torch.int32, device=dev) if masked else None
    out = torch.full((plan.rows_max, N), 7.0, dtype=torch.bfloat16, device=dev)
    ws = torch.full((groups * 8 * 65536,), float("nan"), device=dev)
    _lib.call("fm_grouped_gemm_ragged_m_split", _gemm_kind(_lib.QUANT_BF16) | (_lib.GEMM_W_KMAJOR if kn else 0),
              _token_operand(tokens, _lib.QUANT_BF16), w.operand(), plan.m_tiles, _lib.addr(plan.tile_expert),
              _lib.addr(plan.offsets), E, N, K, _lib.addr(mask), 1, _lib.addr(out), N, _lib.addr(ws), ws.numel() * 4,
              _lib.stream_of(out))
    assert _slots_written(ws) == slots
    for e in range(E):
        got = out[offs[e]:offs[e + 1]].double()
        if masked and e % 2 == 0:
            assert torch.all(got == 7.0)
            continue
        x, we = tokens[offs[e]:offs[e + 1]].double(), W[e].double()
        ref = x @ we.t()
        bound = K * 2.0 ** -24 * (x.abs() @ we.abs().t()) + 2.0 ** -8 * ref.abs() + 1e-30
        assert torch.all((got - ref).abs() <= bound)
    assert torch.all(out[offs[E]:] == 7.0)


@pytest.mark.parametrize("kind", ["pow2", "mx"])
@pytest.mark.parametrize("operand", ["w13", "w2t"])
@pytest.mark.parametrize("kmajor", [True, False])   # the block's tokens: block-major scales
@pytest.mark.parametrize("counts,row_tiles", [((300, 0, 1, 257), 5), ((130, 200), 2)])
def test_paired_matches_unsliced(dev, counts, row_tiles, kmajor, operand, kind):
    """FP8: the sliced sums against the same products in one sweep of K, both in
    fp32: K 2^-23 sum |terms| apart at most, and a bf16 rounding each."""
    E, K, N = len(counts), 6400, 768   # 50 steps
    idx = torch.cat([torch.full((c,), e, dtype=torch.int64) for e, c in enumerate(counts)])[:, None].to(dev)
    plan = fm.route_tokens(idx, E)
    pow2 = kind == "pow2"
    k = _lib.QUANT_POW2 if pow2 else _lib.QUANT_MX
    x = randn_bf16((sum(counts), K), seed=1).to(dev)
    if operand == "w13":   # gate | up: N = 2 H rows of K = D
        w1, w3 = (randn_bf16((E * N // 2, K), seed=s, std=0.1).to(dev) for s in (2, 3))
        ew = ExpertWeights(k, paired=True).refresh(w1, w1, w3, E, False)
        w, W = ew.w13, torch.cat([w1.view(E, N // 2, K), w3.view(E, N // 2, K)], 1).transpose(1, 2)
    else:                  # down: K = H rows of N = D, transposed
        w2 = randn_bf16((E * K, N), seed=2, std=0.1).to(dev)
        ew = ExpertWeights(k, paired=True).refresh(w2, w2, w2, E, False)
        w, W = ew.w2t, w2.view(E, K, N)
    pt = fm.fused_permute_pad(x, plan, E, granularity="1x128" if pow2 else "1x32", pow2_scale=pow2,
                              kmajor_scales=kmajor, paired_rows=True)
    assert w.K == K and w.N == N and w.paired and w.kmajor == (pow2 and operand == "w2t")
    ws = torch.full((256 * 65536,), float("nan"), device=dev)
    gk = _gemm_kind(k) | _lib.GEMM_PAIRED | (_lib.GEMM_W_KMAJOR if w.kmajor else 0) | (
        _lib.GEMM_W_PAIRED if w.kmajor and w.paired else 0)
    args = (gk, _token_operand(pt.rows, k), w.operand(), plan.m_tiles, _lib.addr(plan.tile_expert),
            _lib.addr(plan.offsets), E, N, K, None, 1)
    a, b = (torch.full((plan.rows_max, N), 7.0, dtype=torch.bfloat16, device=dev) for _ in range(2))
    _lib.call("fm_grouped_gemm_ragged_m", *args, _lib.addr(a), _lib.DTYPE_BF16, N, _lib.stream_of(a))
    _lib.call("fm_grouped_gemm_ragged_m_split", *args, _lib.addr(b), N, _lib.addr(ws), ws.numel() * 4,
              _lib.stream_of(b))
    assert _slots_written(ws) == 6 * 3 * row_tiles   # in 6 slices of 8 or 9
    offs = plan.offsets.tolist()
    for e, c in enumerate(counts):
        # quantisation moves a term by 1/8 of its size at most (e4m3, three mantissa bits, each factor 1/16)
        xe = x[idx[:, 0] == e].abs().double()
        terms = 1.25 * (xe @ W[e].abs().double())
        g, h = a[offs[e]:offs[e] + c].double(), b[offs[e]:offs[e] + c].double()
        assert torch.all((g - h).abs() <= K * 2.0 ** -23 * terms + 2.0 ** -8 * (g.abs() + h.abs()))
    assert torch.all(b[offs[E]:] == 7.0)


@pytest.mark.parametrize("kind,T,N", [("bf16", 1024, 2048), ("pow2", 512, 1024)])
def test_sliced_launch_in_a_graph(dev, kind, T, N, monkeypatch):
    """Captured sliced launches replay to the eager result, with eager work between the replays."""
    E, K = 4, 4096
    plan = fm.route_tokens(torch.arange(T, device=dev)[:, None] % E, E)
    k = _lib.QUANT_BF16 if kind == "bf16" else _lib.QUANT_POW2
    x = randn_bf16((T, K), seed=1).to(dev)
    w2 = randn_bf16((E * K, N), seed=2, std=0.1).to(dev)
    w = ExpertWeights(k, paired=True).refresh(w2, w2, w2, E, False).w2t
    tokens = fm.fused_permute_pad(x, plan, E, granularity=None if kind == "bf16" else "1x128",
                                  pow2_scale=kind == "pow2", kmajor_scales=True, paired_rows=kind == "pow2").rows
    called, real = [], _lib.call
    monkeypatch.setattr(_lib, "call", lambda name, *a: (called.append(name), real(name, *a))[1])
    eager, out = (torch.empty(plan.rows_max, N, dtype=torch.bfloat16, device=dev) for _ in range(2))
    _gemm_m(k, tokens, w, plan, eager)
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        _gemm_m(k, tokens, w, plan, out)
    assert called == ["fm_grouped_gemm_ragged_m_split"] * 2
    used = int(plan.offsets[E])
    for _ in range(4):
        out.fill_(7.0)
        graph.replay()
        other = torch.full((64 << 18,), 3.0, device=dev)   # a slice workspace's memory, in use
        _gemm_m(k, tokens, w, plan, torch.empty_like(eager))
        assert torch.equal(out[:used], eager[:used])
        del other
        torch.cuda.synchronize()


def test_rule(dev):
    """Few tiles of a long K, by the host's bound; BF16 of 64 or 88 steps under a mask."""
    def w(N, K):
        return ExpertWeightOperand(None, None, K, N * K, N=N, K=K)

    def plan(n):
        return fm.route_tokens(torch.arange(n, device=dev)[:, None] % 4, 4)

    def out(N):
        return torch.empty(256, N, dtype=torch.bfloat16, device=dev)

    bf, p2 = _lib.QUANT_BF16, _lib.QUANT_POW2
    some = torch.ones(4, dtype=torch.int32, device=dev)
    assert _m_split(bf, plan(1024), w(2048, 4096), out(2048), None)
    assert not _m_split(bf, plan(1024), w(2048, 1024), out(2048), None)
    assert not _m_split(bf, plan(3072), w(2048, 4096), out(2048), None)
    assert not _m_split(bf, plan(8192), w(2048, 14336), out(2048), None)
    assert not _m_split(bf, plan(1024), w(2048, 4096), out(2048).float(), None)
    assert _m_split(p2, plan(512), w(1024, 4096), out(1024), None)
    assert not _m_split(p2, plan(2048), w(2048, 4096), out(2048), None)
    assert _m_split(bf, plan(8192), w(2048, 5632), out(2048), some)
    assert not _m_split(bf, plan(8192), w(2048, 4096), out(2048), some)
    assert _m_split(bf, plan(2048), w(2048, 4096), out(2048), some)
    assert not _m_split(p2, plan(8192), w(2048, 14336), out(2048), some)
