"""BF16 ragged-M GEMM whose few tiles are cut in slices of K, against float64: bf16
products are exact in fp32, so a sum over K, in slices or not, is off by at most
K 2^-24 sum |terms|, and the bf16 output by half a unit of its last place more."""

import pytest
import torch

import nanopysche_amd as fm
from nanopysche_amd import _lib
from nanopysche_amd.flow_moe import ExpertWeightOperand, _gemm_kind, _m_split, _token_operand
from tests.helpers import randn_bf16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", ["nk", "kn", "kn_split"])
@pytest.mark.parametrize("counts,masked,K,groups", [
    ((300, 0, 1, 257), False, 4224, 32),    # 5 tiles of 66 steps in up to 4 slices; an expert without tokens
    ((130, 600, 20, 90), True, 4096, 32),   # every second expert
    ((700, 300), False, 4096, 1),           # 8 workgroups for 5 tiles of one column: not sliced
    ((520,), False, 2176, 2),               # 34 steps in two slices of 17
])
def test_matches_float64(dev, counts, masked, K, groups, form):
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
        cut = K // 256 * 128
        b = torch.zeros_like(rows)
        b[:, :K - cut] = rows[:, cut:]
        kw = dict(data2=b, split=cut)
    w = ExpertWeightOperand(rows, None, rows.shape[2], N * K, N=N, K=K, kmajor=kn, **kw)
    mask = torch.tensor([e % 2 for e in range(E)], dtype=torch.int32, device=dev) if masked else None
    out = torch.full((plan.rows_max, N), 7.0, dtype=torch.bfloat16, device=dev)
    ws = torch.full((groups * 8 * 65536,), float("nan"), device=dev)
    _lib.call("fm_grouped_gemm_ragged_m_split", _gemm_kind(_lib.QUANT_BF16) | (_lib.GEMM_W_KMAJOR if kn else 0),
              _token_operand(tokens, _lib.QUANT_BF16), w.operand(), plan.m_tiles, _lib.addr(plan.tile_expert),
              _lib.addr(plan.offsets), E, N, K, _lib.addr(mask), 1, _lib.addr(out), N, _lib.addr(ws), ws.numel() * 4,
              _lib.stream_of(out))
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


def test_rule(dev):
    """Few tiles of a long K, by the host's bound; any launch under a mask."""
    def w(N, K):
        return ExpertWeightOperand(None, None, K, N * K, N=N, K=K)

    def plan(n):
        return fm.route_tokens(torch.arange(n, device=dev)[:, None] % 4, 4)

    def out(N):
        return torch.empty(256, N, dtype=torch.bfloat16, device=dev)

    some = torch.ones(4, dtype=torch.int32, device=dev)
    assert _m_split(plan(1024), w(2048, 4096), out(2048), None)
    assert not _m_split(plan(1024), w(2048, 3968), out(2048), None)
    assert not _m_split(plan(8192), w(2048, 4096), out(2048), None)
    assert _m_split(plan(8192), w(2048, 4096), out(2048), some)
    assert not _m_split(plan(1024), w(2048, 4096), out(2048).float(), None)
