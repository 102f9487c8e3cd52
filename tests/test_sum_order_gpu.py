"""The order in which the norms add a row's squares is fixed, whatever lanes hold the row, so that a seed renders the same
bits from one layout of the kernels to the next.

The rows hold ones and elements so small that a square added to a sum of at least 1 is lost (t^2 < 2^-24), while a sum
of their own would not be. In the fixed order every one of them follows a one, so the results have the bits of the rows
with zeros in their place.
"""
from __future__ import annotations

import pytest
import torch

from hummingbird_amd import elementwise

pytestmark = pytest.mark.gpu
DEV = "cuda"
TINY = 0.98 * 2.0 ** -12  # rounded to bf16 too, its square is below 2^-24


@pytest.mark.parametrize("channels", [520, 1536, 2048, 5000])
def test_row_norms_add_a_lane_s_chunks_in_order(channels):
    """Lane l of a wave of 64 adds the 4-element chunks l, l + 64, ... of an fp32 row: the first 64 chunks begin with a
    one. Both norms, rows of less than and more than one turn of the workgroup."""
    print(f"\n[case] row norm order C{channels}", flush=True)
    ones = torch.zeros(channels, device=DEV)
    ones[0:256:4] = 1.0
    x = torch.where(ones == 1, 1.0, TINY).expand(1, 3, channels).contiguous()
    ones = ones.expand(1, 3, channels).contiguous()
    weight = torch.rand(channels, device=DEV) + 0.5
    big = ones == 1

    def norms(row):
        plain = elementwise.rms_modulate(row, weight, 0.0)[big]
        if channels > 2048:
            return plain
        h, y = elementwise.residual_rms(torch.zeros_like(row), row, weight, 0.0)
        assert torch.equal(h, row)
        return torch.cat([plain, y[big]])
    assert torch.equal(norms(x), norms(ones))
