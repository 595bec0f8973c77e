"""Which BF16 parameters the expert block's GEMMs read in place (no GPU needed)."""

import pytest
import torch

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
