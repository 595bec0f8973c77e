"""Weight gradients of experts with few tokens (the 128 x 128 kernel) against the
256 x 256 kernels: the MFMA order is the same, so the bits are."""

import pytest
import torch

import nanopysche_amd as fm
from nanopysche_amd import _lib
from nanopysche_amd.flow_moe import _gemm_kind, _operand
from tests.helpers import randn_bf16

pytestmark = pytest.mark.gpu
KINDS = {"bf16": _lib.QUANT_BF16, "pow2": _lib.QUANT_POW2}


def _wide(t, ld, paired):
    """The operand's bytes with a row pitch of ``ld`` elements (pairs of rows for the paired layout)."""
    t = t.view(torch.int16) if t.dtype == torch.bfloat16 else t.view(torch.uint8)
    n = 2 if paired else 1
    out = torch.zeros(t.shape[0] // n, n * ld, dtype=t.dtype, device=t.device)
    out[:, :n * t.shape[1]] = t.reshape(t.shape[0] // n, n * t.shape[1])
    return out


@pytest.mark.parametrize("kind,paired", [("bf16", False), ("pow2", False), ("pow2", True)])
@pytest.mark.parametrize("counts,M,N,masked", [
    ([0, 100, 128, 129, 384, 700], 384, 1152, False),     # 0 .. 6 K steps of 128; a 9th tile column, 3 tile rows
    ([300], 256, 128, False),                             # one expert, fewer tiles than a chunk
    ([1, 0, 513, 0, 40, 256, 200, 90], 256, 1024, True),
    ([0, 1, 128, 200] * 16, 256, 128, False),             # as many experts as lanes, the first without tokens
    ([130, 0, 40, 257] * 16, 256, 256, True),
])
@pytest.mark.parametrize("out", [torch.bfloat16, torch.float32])
def test_few_token_weight_gradient_bits(dev, kind, paired, counts, M, N, masked, out):
    if masked and paired:
        pytest.skip("paired operands take no expert mask")
    k, E, T = KINDS[kind], len(counts), sum(counts)
    idx = torch.cat([torch.full((n,), e, dtype=torch.int64) for e, n in enumerate(counts)])
    idx = idx[torch.randperm(T, generator=torch.Generator().manual_seed(3))].view(T, 1)
    gran = None if kind == "bf16" else "1x128"
    kw = dict(granularity=gran, pow2_scale=kind == "pow2", return_transpose=True, paired_cols=paired)
    pa = fm.fused_permute_pad(randn_bf16((T, M), seed=31).to(dev), idx.to(dev), E, **kw)
    pb = fm.fused_permute_pad(randn_bf16((T, N), seed=32).to(dev), pa.plan, E, **kw)
    plan, split = pa.plan, M // 2 // 128 * 128
    mask = torch.tensor([e % 2 for e in range(E)], dtype=torch.int32, device=dev) if masked else None

    def run(ld):
        ops = []
        for t in (pa.rows_t, pb.rows_t):
            data = t if kind == "bf16" else t.data
            sc = {} if kind == "bf16" else dict(s_row=1, s_kb=t.scale.stride(0))
            if ld != plan.rows_max:
                data = _wide(data, ld, paired)
            ops.append(_operand(data, None if kind == "bf16" else t.scale, ld=ld, **sc))
            keep.append(data)
        o1 = torch.full((E * split, N), 7.0, dtype=out, device=dev)
        o2 = torch.full((E * (M - split), N), 7.0, dtype=out, device=dev)
        dt = _lib.DTYPE_F32 if out == torch.float32 else _lib.DTYPE_BF16
        _lib.call("fm_grouped_gemm_ragged_k", _gemm_kind(k) | (_lib.GEMM_PAIRED if paired else 0), *ops,
                  _lib.addr(plan.offsets), E, M, N, _lib.addr(mask), 1, _lib.addr(o1), split * N, _lib.addr(o2),
                  (M - split) * N, split, dt, N, _lib.stream_of(o1))
        torch.cuda.synchronize()
        return o1, o2

    keep = []
    a, b = run(plan.rows_max), run(2048 * E)   # few tokens per expert; a pitch that says many
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    for e, n in enumerate(counts):
        blk = a[0][e * split:(e + 1) * split]
        if masked and e % 2 == 0:
            assert torch.all(blk == 7.0)
        else:
            assert torch.all(blk == 0) if n == 0 else bool(blk.any())
