"""GPU parity of the fp32 kernels at the edges of their own code: the DyT's tanh over its whole range, the key and query
tiles' edges, and gains and values of many magnitudes through the split matrix operands."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from hummingbird_amd import workloads
from tests import test_dense_gpu as dense
from tests.test_band_gpu import oracle, run_hip
from tests.util import assert_fp32_parity

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("alpha", [0.02, 0.5, 4.0, 60.0])
def test_band_fp32_dyt_over_the_range_of_tanh(alpha):
    """Keys and queries whose alpha x lies in the small-argument polynomial (alpha 0.02), on both sides of the switch at
    0.625 (planted exactly, one ulp below and above), in the exponential form and past saturation (1e30, infinity),
    against the oracle (np.tanh) at the fp32 contract."""
    print(f"\n[case] fp32 DyT alpha {alpha}", flush=True)
    h, d = 2, 64
    inp = workloads.band_inputs(1, 200, h, d, 40, seed=3, dtype="fp32")
    for n in ("q_norm", "k_norm"):
        inp[n] = dict(inp[n], alpha=np.float32(alpha))
    edge = np.float32(0.625) / np.float32(alpha)
    planted = np.array([0.0, -0.0, 1e-30, -1e-20, edge, np.nextafter(edge, np.float32(0)), -edge,
                        -np.nextafter(edge, np.float32(9)), 1e30, -1e30, np.inf, -np.inf], np.float32)
    qkv = inp["qkv"]
    for sec in (0, 1, 3, 4):  # q, k, q_diff, k_diff of one row per section
        qkv[0, 20 + sec, sec * h * d:sec * h * d + planted.size] = planted
    got = run_hip(inp, dtype=torch.float32)
    assert_fp32_parity(got, oracle(inp, "xla", compute="fp32"), f"alpha {alpha}")


def dense_both(inp: dict, lam: bool = True) -> tuple[np.ndarray, np.ndarray]:
    got = dense.run_hip(inp, dtype=torch.float32, lam=lam)
    return got, dense.oracle(inp, "xla", compute="fp32", lam=lam)


@pytest.mark.parametrize("length,dim", [(1, 64), (31, 64), (32, 128), (33, 64), (64, 64), (65, 128), (96, 64), (129, 64)])
def test_dense_fp32_at_tile_edges(length, dim):
    """Key counts around the 32-key tile and query counts around the 64-query block (an odd and an even number of tiles
    through the two stages at head_dim 64, one stage at 128)."""
    print(f"\n[case] fp32 dense L{length} D{dim}", flush=True)
    got, ref = dense_both(workloads.dense_inputs(2, length, 2, dim, seed=length, dtype="fp32", half=dim // 4,
                                                  mask_tail=min(16, length // 4)))
    assert_fp32_parity(got, ref, f"L{length} D{dim}")


@pytest.mark.parametrize("half", [0, 16, 32])
def test_dense_fp32_gains_over_many_magnitudes(half):
    """Norm gains of 1e-4 .. 1e4 per dim with the other side's inverse (logits of the usual size, each operand far
    outside the half range): the split operands' powers of two follow the gains. RoPE pairs share a gain, as their dims
    mix: with unequal ones the logits themselves would reach 1e8."""
    print(f"\n[case] fp32 dense gains half {half}", flush=True)
    inp = workloads.dense_inputs(1, 150, 2, 64, seed=7, dtype="fp32", half=half)
    gain = (10.0 ** np.random.default_rng(1).uniform(-4, 4, 64)).astype(np.float32)
    gain[half:2 * half] = gain[:half]
    inp["q_weight"], inp["k_weight"] = inp["q_weight"] * gain, inp["k_weight"] / gain
    got, ref = dense_both(inp)
    assert_fp32_parity(got, ref, f"gains half {half}")


@pytest.mark.parametrize("scale", [1e-30, 1e-6, 1.0, 1e6, 1e30])
def test_dense_fp32_values_over_many_magnitudes(scale):
    """V of any magnitude, and growing by 1e12 from the first key tile to the last, with a tile of zeros among them: the
    result as a whole, and each dim by itself."""
    print(f"\n[case] fp32 dense V {scale}", flush=True)
    h, d, length = 2, 64, 200
    inp = workloads.dense_inputs(1, length, h, d, seed=8, dtype="fp32")
    grow = (scale * 10.0 ** np.linspace(-6, 6, length)).astype(np.float32)
    grow[64:96] = 0
    inp["qkv"][0, :, 2 * h * d:3 * h * d] *= grow[:, None]
    got, ref = dense_both(inp)
    assert_fp32_parity(got, ref, f"V {scale}")
    for dim in range(h * d):
        assert_fp32_parity(got[0, :, dim], ref[0, :, dim], f"V {scale} dim {dim}")


@pytest.mark.parametrize("window,dim", [(0, 64), (31, 64), (32, 64), (33, 128), (95, 64), (200, 128)])
def test_band_fp32_values_over_many_magnitudes(window, dim):
    """The band with windows around the 32-key tile and V growing by 1e12 along the sequence: every query still has
    fp32 accuracy relative to its own neighbourhood, so the rows are compared one by one."""
    print(f"\n[case] fp32 band V w{window} D{dim}", flush=True)
    h, length = 2, 300
    inp = workloads.band_inputs(1, length, h, dim, window, seed=9, dtype="fp32", half=dim // 4)
    grow = (10.0 ** np.linspace(-6, 6, length)).astype(np.float32)
    inp["qkv"][0, :, 2 * h * dim:3 * h * dim] *= grow[:, None]
    got, ref = run_hip(inp, dtype=torch.float32), oracle(inp, "xla", compute="fp32")
    for row in range(length):
        assert_fp32_parity(got[0, row], ref[0, row], f"w{window} D{dim} row {row}")
