"""GPU parity of the fp32 kernels at the edges of their own code: the DyT's tanh over its whole range."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from hummingbird_amd import workloads
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
