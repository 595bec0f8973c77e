"""The router forward's workspace is that of the path its sizes take (size functions
of the library alone, no GPU needed)."""

import pytest

from nanopysche_amd import _lib

BF16, F32 = _lib.DTYPE_BF16, _lib.DTYPE_F32


def _of(T, D, E, x=BF16, w=BF16):
    return _lib.size_of("fm_router_forward_workspace_bytes_of", T, D, E, x, w)


@pytest.mark.parametrize("x", [BF16, F32])
@pytest.mark.parametrize("T,D,E,w", [(16384, 2048, 8, BF16), (16384, 2048, 8, F32), (17, 4096, 8, BF16), (1, 512, 1, F32)])
def test_one_pass_gates_hold_no_chunk_sums(T, D, E, x, w):
    """Per 16 tokens: E softmax sums, one logsumexp sum, E counts."""
    assert _lib.load().fm_router_forward_fused(E, D, w) == 1
    assert _of(T, D, E, x, w) == (T + 15) // 16 * (2 * E + 1) * 4


@pytest.mark.parametrize("T", [1, 33, 4096, 16384])
@pytest.mark.parametrize("D,E", [(200, 5), (2048, 9), (7168, 8), (7168, 256), (384, 64)])
@pytest.mark.parametrize("w", [BF16, F32])
def test_the_size_without_d_is_enough_for_every_d(T, D, E, w):
    most = _lib.size_of("fm_router_forward_workspace_bytes", T, E)
    plain = 1024 * (E + 1) * 4
    assert plain == _of(T, D, E, F32, w) <= _of(T, D, E, BF16, w) <= most
