"""The router's products on the matrix cores (bf16 x; fp32 factors as three bf16
pieces) at the edges of their tiles, against float64: token tiles of 16 / 32 /
64, expert fragments and groups, chunks of D with a part-filled last step,
slices of tokens.

Bounds: every product of pieces is exact in fp32, so a sum over n is off by at
most (n + 2) 2^-24 sum |terms|, the 2 for the low pieces joining the high ones
(n 2^-23 for the nine pairs of pieces of two fp32 factors), whatever its order."""

import pytest
import torch

import nanopysche_amd as fm
from nanopysche_amd import _lib
from nanopysche_amd.routing import router_backward, router_forward

pytestmark = pytest.mark.gpu

SHAPES = [(1, 8, 9), (16, 72, 16), (17, 136, 17), (33, 264, 33), (65, 1000, 48), (130, 512, 64), (200, 776, 65),
          (64, 2048, 128), (129, 1160, 160), (1000, 384, 256), (37, 200, 5), (100, 4104, 3),
          (3001, 128, 250)]


def _inputs(dev, T, D, E, gate, seed=3):
    g = torch.Generator().manual_seed(seed)
    x = torch.randn(T, D, generator=g).bfloat16().to(dev)
    w = (torch.randn(E, D, generator=g) * 0.05).to(gate).to(dev)
    b = (torch.randn(E, generator=g) * 0.1).to(gate).to(dev)
    sb = (torch.randn(E, generator=g) * 0.2).to(dev)
    return g, x, w, b, sb


@pytest.mark.parametrize("gate", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,D,E", SHAPES)
def test_products_at_tile_edges(dev, T, D, E, gate):
    g, x, w, b, sb = _inputs(dev, T, D, E, gate)
    K = min(E, 6)
    wts, idx, aux, st = router_forward(x, w, b, sb, K, "softmax", None, None, 1e-3)
    x64, w64 = x.double(), w.double()
    ref = x64 @ w64.t() + b.double() + sb.double()
    bound = (D + 2) * 2.0 ** -24 * (x64.abs() @ w64.abs().t() + b.double().abs() + sb.double().abs()) + 1e-30
    assert torch.all((st.logits.double() - ref).abs() <= bound)
    # the selection, counts and loss of these logits
    lg = st.logits.double()
    assert torch.equal(torch.gather(lg, 1, idx), lg.topk(K, dim=1).values)
    assert torch.equal(st.counts.long(), torch.bincount(idx.flatten(), minlength=E))
    probs = torch.softmax(lg, dim=1)
    loss = E * (st.counts.double() / T * probs.mean(dim=0)).sum() + 1e-3 * torch.logsumexp(lg, 1).square().mean()
    assert abs(float(aux) - float(loss)) <= 1e-5 * abs(float(loss))
    # backward: dx, dw, db of the dlogits it forms
    dws = torch.randn(T, K, generator=g).to(dev)
    daux = torch.tensor(0.5, device=dev)
    dx, dW, db, dl = router_backward(st, x, w, dws, daux, bias_dtype=torch.float32)
    dl64 = dl.double()
    size = dl64.abs() @ w64.abs()
    assert torch.all((dx.double() - dl64 @ w64).abs() <= 2.0 ** -8 * (dl64 @ w64).abs() + (E + 2) * 2.0 ** -23 * size + 1e-30)
    size = dl64.abs().t() @ x64.abs()
    out = 2.0 ** -8 if gate == torch.bfloat16 else 0.0
    assert torch.all((dW.double() - dl64.t() @ x64).abs() <= out * (dl64.t() @ x64).abs() + (T + 2) * 2.0 ** -24 * size + 1e-30)
    assert torch.all((db.double() - dl64.sum(0)).abs() <= (T + 2) * 2.0 ** -24 * dl64.abs().sum(0) + 1e-30)
    only = router_backward(st, x, w, dws, daux, need_w=False, need_b=False)[0]
    assert torch.equal(only, dx)


@pytest.mark.parametrize("pitch,start", [(4, 0), (0, 4), (12, 4)])
@pytest.mark.parametrize("T,D,E", [(33, 264, 33), (37, 200, 5), (100, 4104, 3), (64, 512, 64)])
def test_gate_rows_off_16_bytes(dev, T, D, E, pitch, start):
    """A bf16 gate whose rows lie on 8 bytes keeps the FMA kernel: the bits of the fp32-x
    path (the same values, read wider), in the logits and in the whole forward."""
    g, x, w, b, sb = _inputs(dev, T, D, E, torch.bfloat16)
    flat = torch.zeros(E * (D + pitch) + 8, dtype=torch.bfloat16, device=dev)
    view = flat[start:start + E * (D + pitch)].view(E, D + pitch)[:, :D]
    view.copy_(w)
    assert flat.data_ptr() % 16 == 0 and (view.data_ptr() % 16 or 2 * view.stride(0) % 16)
    ref = fm.router_logits(x.float(), view, b, sb)
    assert torch.equal(fm.router_logits(x, view, b, sb), ref)
    K = min(E, 4)
    got = router_forward(x, view, b, sb, K, "sigmoid", None, None, 1e-3)
    want = router_forward(x.float(), view, b, sb, K, "sigmoid", None, None, 1e-3)
    for u, v in zip((*got[:3], got[3].logits, got[3].counts), (*want[:3], want[3].logits, want[3].counts)):
        assert torch.equal(u, v)
    dws, daux = torch.randn(T, K, generator=g).to(dev), torch.tensor(0.5, device=dev)
    for u, v in zip(router_backward(got[3], x, view, dws, daux, bias_dtype=torch.float32),
                    router_backward(got[3], x, w, dws, daux, bias_dtype=torch.float32)):
        assert torch.equal(u, v)


@pytest.mark.parametrize("T,D,E", [(40, 136, 9), (64, 264, 40), (64, 4104, 3)])
def test_dx_of_fp32_factors_has_every_product(dev, T, D, E):
    """dlogits a and gate b, all low mantissa bits set, in expert 0; the product's two
    fp32 halves (a b = p + r exactly) against -1 in two other experts: dx[t, t] is 0.  The terms
    stay below 2, so the sums (at most four of that size: the two high pieces and what is
    carried) are off by 2^-22 at most, where the three smallest pairs of pieces alone are 2^-21."""
    n = min(T, D)
    k = torch.arange(n) % 32
    a = 1 + k / 128 + 2.0 ** -7 - 2.0 ** -23
    b = 1 + k.flip(0) / 128 + 2.0 ** -7 - 2.0 ** -23
    a, b = a.float(), b.float()
    prod = a.double() * b.double()
    p = prod.float()
    r = (prod - p.double()).float()
    assert torch.equal(p.double() + r.double(), prod) and float(p.max()) < 2
    dl, w = torch.zeros(T, E), torch.zeros(E, D)
    dl[:n, 0], w[0, :n] = a, b
    dl[:, 1] = dl[:, E - 1] = -1
    w[1, :n], w[E - 1, :n] = p, r
    dl, w, x = dl.to(dev), w.to(dev), torch.zeros(T, D, dtype=torch.bfloat16, device=dev)
    dx = torch.empty_like(x)
    ws = torch.empty(_lib.size_of("fm_router_workspace_bytes", T, D, E), dtype=torch.uint8, device=dev)
    _lib.call("fm_router_backward", _lib.addr(dl), E, _lib.addr(x), _lib.DTYPE_BF16, D, T, D, _lib.addr(w),
              _lib.DTYPE_F32, D, E, _lib.addr(dx), D, None, _lib.DTYPE_F32, 0, None, _lib.DTYPE_F32, _lib.addr(ws),
              ws.numel(), _lib.stream_of(x))
    assert float(dx.diagonal()[:n].abs().max()) <= 2.0 ** -22


@pytest.mark.parametrize("gate", [torch.bfloat16, torch.float32])
def test_logits_keep_small_terms_beside_a_large_one(dev, gate):
    """2^25 first, -2^25 last and 30 ones between, one in each step of 64 columns, in one
    chunk of D: 30.  A chain of MFMAs is at most 256 columns; the large term's ulp of 4 swallows the
    ones of its own chain (at most 3 of the first, and 4 of the last with two roundings of at
    most 2), never those carried between chains.  One chain over all columns gives 0."""
    T, D, E = 16384, 2048, 256
    x, w = torch.zeros(T, D, dtype=torch.bfloat16, device=dev), torch.zeros(E, D, dtype=gate, device=dev)
    x[:, 65:D - 64:64] = 1
    w[:, 65:D - 64:64] = 1
    x[:, 0], x[:, D - 1] = 2.0 ** 12, -(2.0 ** 12)
    w[:, 0] = w[:, D - 1] = 2.0 ** 13
    ref = float(x[0].double() @ w[0].double())
    assert ref == 30
    got = router_forward(x, w, None, None, 4, "softmax", None, None, 0.0)[3].logits
    assert float((got - ref).abs().max()) <= 11
    assert torch.equal(fm.router_logits(x, w), got)


def test_weight_and_bias_gradients_keep_small_terms(dev):
    """2^25 in the first token, -2^25 in the last: the ones of the token slices between (each slice's own
    sum is exact) all reach dW, and db has the ones of the large term's own tile of 64 within the 2 that
    rounding the tile's sum to its ulp of 4 costs."""
    T, D, E = 16384, 512, 12
    dl = torch.zeros(T, E, device=dev)
    x = torch.zeros(T, D, dtype=torch.bfloat16, device=dev)
    dl[0], dl[1:64], dl[T - 1] = 2.0 ** 25, 1, -(2.0 ** 25)
    dl[256 + 5:T - 256:256] = 1
    x[0], x[T - 1] = 1, 1
    x[256 + 5:T - 256:256] = 1
    w = torch.zeros(E, D, device=dev)
    dw, db = torch.empty(E, D, device=dev), torch.empty(E, device=dev)
    ws = torch.empty(_lib.size_of("fm_router_workspace_bytes", T, D, E), dtype=torch.uint8, device=dev)
    _lib.call("fm_router_backward", _lib.addr(dl), E, _lib.addr(x), _lib.DTYPE_BF16, D, T, D, _lib.addr(w),
              _lib.DTYPE_F32, D, E, None, 0, _lib.addr(dw), _lib.DTYPE_F32, D, _lib.addr(db), _lib.DTYPE_F32,
              _lib.addr(ws), ws.numel(), _lib.stream_of(x))
    assert torch.all(dw == 62)
    assert float((db - 125).abs().max()) <= 2


@pytest.mark.parametrize("gate", [torch.bfloat16, torch.float32])
def test_infinite_and_nan_inputs(dev, gate):
    """A non-finite x or gate value reaches the outputs it reaches in fp32 arithmetic, as the same class."""
    T, D, E = 70, 264, 40
    _, x, w, b, sb = _inputs(dev, T, D, E, gate)
    w[3, 5], w[4, 6] = float("inf"), float("nan")
    x[9, 7], x[10, 8], x[11, 9] = float("inf"), float("-inf"), float("nan")
    w[:, 9] = 0.25      # a value whose low pieces are zero, against the infinities
    x[12, 9] = float("inf")
    got = fm.router_logits(x, w, b, sb)
    ref = x.float() @ w.float().t() + b.float() + sb
    for same in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(same(got), same(ref))


def test_selection_order_of_special_scores(dev):
    """NaN above every number, ties (-0 and +0 among them) to the lower expert, -inf still selectable."""
    E, K = 200, 5
    lg = torch.full((4, E), float("-inf"))
    lg[0, 150], lg[0, 20] = 1.0, 1.0
    lg[1, 199], lg[1, 64], lg[1, 65] = float("nan"), float("inf"), float("inf")
    lg[2, 3], lg[2, 70] = -0.0, 0.0
    lg[3] = 2.0
    _, idx = fm.topk_gating(lg.to(dev), K)
    assert idx.cpu().tolist() == [[20, 150, 0, 1, 2], [199, 64, 65, 0, 1], [3, 70, 0, 1, 2], [0, 1, 2, 3, 4]]
