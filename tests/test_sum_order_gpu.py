"""The order in which the norms add a row's squares is fixed, whatever lanes hold the row, so that a seed renders the same
bits from one layout of the kernels to the next.

The rows hold ones and elements so small that a square added to a sum of at least 1 is lost (t^2 < 2^-24), while a sum
of their own would not be. In the fixed order every one of them follows a one, so the results have the bits of the rows
with zeros in their place.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from hummingbird_amd import cross_attention as xattn
from hummingbird_amd import dense_attention as da
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


@pytest.mark.parametrize("length,heads,dim", [(100, 2, 64), (1000, 24, 64), (100, 2, 128)])
def test_queries_add_their_squares_in_order(length, heads, dim):
    """A query row is added dim by dim, by 64-query workgroups (one row per lane), 128-query ones (two) and at head_dim
    128. Dim 0 is the one; its norm weight puts the normalised value just above a rounding midpoint (and a mean of
    squares larger by 2^-19 / D would put it below), and the keys have no other dim."""
    print(f"\n[case] query order L{length} H{heads} D{dim}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(1)
    bf16, width = torch.bfloat16, heads * dim
    q = torch.full((1, length, 2 * width), TINY, device=DEV, dtype=bf16)
    zeros = torch.zeros_like(q)
    q[..., ::dim] = zeros[..., ::dim] = 1.0
    assert float(q[0, 0, 1].float() ** 2) < 2.0 ** -24
    kv = torch.zeros((1, 33, 3 * width), device=DEV, dtype=bf16)
    kv[..., :width:dim] = torch.randn((1, 33, heads), generator=gen, device=DEV).to(bf16)  # k; k_diff weighs all alike
    kv[..., 2 * width:] = torch.randn((1, 33, width), generator=gen, device=DEV).to(bf16)
    weight = np.ones(dim)
    weight[0] = (1 + 2.0 ** -8) * (1 + 2.0 ** -21) / np.sqrt(dim)
    weight = torch.from_numpy(weight.astype(np.float32)).to(DEV)
    context = xattn.prepare_cross_kv(kv, torch.ones(dim, device=DEV), heads, dim, 1e-6)
    got = xattn.cross_attention(q, context, weight, 0.0)
    assert torch.equal(got, xattn.cross_attention(zeros, context, weight, 0.0))


@pytest.mark.parametrize("length", [1350, 3390, 3456])
def test_workgroup_sizes_give_the_same_bits(length):
    """24 heads at lengths on both sides of the lines between 64- and 128-query workgroups (256 CUs: 24 x 22 64-query ones,
    24 x 53, and 24 x 27 128-query ones) against the same heads one by one, which run 64-query ones at every length."""
    print(f"\n[case] workgroup sizes L{length}", flush=True)
    heads, dim, half = 24, 64, 16
    gen = torch.Generator(device=DEV).manual_seed(2)
    qkv = torch.randn((1, length, 5, heads, dim), generator=gen, device=DEV).to(torch.bfloat16)
    weight = 1 + 0.02 * torch.randn(dim, generator=gen, device=DEV)
    cos, sin = da.rope_tables(length, 10000.0 ** (-torch.arange(half, device=DEV) / half))

    def run(x):
        return da.dense_attention(x.reshape(1, length, -1).contiguous(), weight, weight, cos, sin, None, x.shape[3], dim,
                                  half, 1e-6)
    whole = run(qkv).reshape(length, heads, dim)
    for head in (0, heads - 1):
        assert torch.equal(run(qkv[:, :, :, head:head + 1]).reshape(length, dim), whole[:, head])
