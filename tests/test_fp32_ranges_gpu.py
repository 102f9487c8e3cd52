"""fp32 attention keeps fp32 accuracy in every dim and row, whatever other values of V a dim, a key tile or another tile
holds, against the oracle at the fp32 contract taken dim by dim and row by row (not relative to the largest output)."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest
import torch

from hummingbird_amd import _lib
from hummingbird_amd import band_attention as ba
from hummingbird_amd import cross_attention as xattn
from hummingbird_amd import dense_attention as da
from hummingbird_amd import workloads
from tests import test_band_gpu as band
from tests import test_cross_gpu as cross
from tests import test_dense_gpu as dense
from tests.util import FP32_REL, assert_fp32_parity

pytestmark = pytest.mark.gpu
SPIKES = [1e4, 1e7, 1e10, 1e12, 1e38, np.inf]


def check_dims(got: np.ndarray, ref: np.ndarray, skip: set, what: str) -> None:
    """Every column of (N, W) results within the contract of its own largest value."""
    cols = [c for c in range(ref.shape[1]) if c not in skip]
    g, r = got[:, cols].astype(np.float64), ref[:, cols].astype(np.float64)
    worst = (np.abs(g - r).max(0) / np.abs(r).max(0)).max()
    assert worst <= FP32_REL, f"{what}: relative max error of a dim {worst:.3g}"


def check_rows(got: np.ndarray, ref: np.ndarray, skip: set, what: str, rel: float = FP32_REL) -> None:
    """Every row of (N, W) results within the contract of its own largest value."""
    cols = [c for c in range(ref.shape[1]) if c not in skip]
    g, r = got[:, cols].astype(np.float64), ref[:, cols].astype(np.float64)
    worst = (np.abs(g - r).max(1) / np.abs(r).max(1)).max()
    assert worst <= rel, f"{what}: relative max error of a row {worst:.3g}"


@pytest.mark.parametrize("spike", SPIKES)
@pytest.mark.parametrize("dim", [64, 128])
def test_dense_v_spike_costs_its_own_dim_only(dim, spike):
    """One large value in dim 0 of one key of head 0, early in the sequence: all tiles after it, and the other dims of its
    own. An infinite one makes its dim NaN or infinite and leaves the others."""
    print(f"\n[case] fp32 dense V spike {spike} D{dim}", flush=True)
    h, length = 2, 200
    inp = workloads.dense_inputs(1, length, h, dim, seed=11, dtype="fp32", half=dim // 4)
    inp["qkv"][0, 40, 2 * h * dim] = spike
    with np.errstate(invalid="ignore", over="ignore"):
        ref = dense.oracle(inp, "xla", compute="fp32")
    check_dims(dense.run_hip(inp, dtype=torch.float32)[0], ref[0], {0}, f"spike {spike}")


@pytest.mark.parametrize("factor", [1e-12, 1e-7, 1e-4, 1e5, 1e8])
def test_dense_v_dims_of_many_magnitudes(factor):
    """One dim of V larger or smaller than the others throughout: each keeps its own accuracy."""
    print(f"\n[case] fp32 dense V dim x {factor}", flush=True)
    h, dim = 2, 64
    inp = workloads.dense_inputs(1, 150, h, dim, seed=12, dtype="fp32")
    inp["qkv"][0, :, 2 * h * dim + 5] *= np.float32(factor)
    check_dims(dense.run_hip(inp, dtype=torch.float32)[0], dense.oracle(inp, "xla", compute="fp32")[0], set(),
               f"dim x {factor}")


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("at", [0, 33, 127])
def test_dense_weight_on_a_masked_key(at, dim):
    """Every query gives nearly all of its weight to one key whose value is masked away, so the results are sums over
    probabilities of 1e-10, in the masked key's tile and in the others. A row's probabilities share the error of the
    masked key's logit, 24: 32 roundings of it (the norms of q and k, the product, its scale, the exponential's argument)
    are at most 32 x 24 x 2^-24 = 4.6e-5 of them."""
    print(f"\n[case] fp32 dense sink at {at} D{dim}", flush=True)
    h, length = 1, 128
    inp = workloads.dense_inputs(1, length, h, dim, seed=13, dtype="fp32", half=0, mask_tail=0, gain_mean=np.sqrt(24 / np.sqrt(dim)))
    qkv = inp["qkv"].reshape(length, 5, dim)
    axis = np.random.default_rng(1).standard_normal(dim).astype(np.float32)
    for q, k in ((0, 1), (3, 4)):
        qkv[:, q] = axis + 0.1 * qkv[:, q]
        qkv[:, k] -= np.outer(qkv[:, k] @ axis, axis) / (axis @ axis)
        qkv[at, k] = axis
    inp["valid"][0, at] = 0
    got, ref = dense.run_hip(inp, dtype=torch.float32), dense.oracle(inp, "xla", compute="fp32")
    assert np.abs(ref).max() < 1e-7
    check_rows(got[0], ref[0], set(), f"sink at {at}", rel=4.6e-5)


@pytest.mark.parametrize("workspace", [True, False], ids=["ws", "no-ws"])
@pytest.mark.parametrize("channels", [1, 64])
@pytest.mark.parametrize("spike", SPIKES)
def test_band_v_spike_outside_the_window(spike, channels, workspace):
    """Spikes that a query does not weigh, in its own key tile or in an earlier one of its block: key 70 lies in the tiles
    of queries to 95, which end at their own windows of 9. One channel of the head, or all (rows that weigh those are
    compared only in the other head)."""
    print(f"\n[case] fp32 band V spike {spike} x{channels} ws {workspace}", flush=True)
    h, d, length, w, key = 2, 64, 200, 9, 70
    inp = workloads.band_inputs(1, length, h, d, w, seed=14, dtype="fp32", half=16)
    inp["qkv"][0, key, 2 * h * d:2 * h * d + channels] *= np.float32(spike if np.isfinite(spike) else 1)
    if not np.isfinite(spike):
        inp["qkv"][0, key, 2 * h * d:2 * h * d + channels] = spike
    with np.errstate(invalid="ignore", over="ignore"):
        ref = band.oracle(inp, "xla", compute="fp32")[0]
    if workspace:
        got = band.run_hip(inp, dtype=torch.float32)[0]
    else:
        cap, ba.FP32_WORKSPACE_CAP = ba.FP32_WORKSPACE_CAP, 0
        try:
            got = band.run_hip(inp, dtype=torch.float32)[0]
        finally:
            ba.FP32_WORKSPACE_CAP = cap
    spiked = set(range(channels))
    inside = np.abs(np.arange(length) - key) <= w
    check_rows(got[inside], ref[inside], spiked, f"rows that weigh the spike {spike}")
    # 0 x inf is NaN in the matrix products, so an infinite value reaches the rows of its key tiles in its own dims
    check_rows(got[~inside], ref[~inside], spiked if np.isinf(spike) else set(), f"rows that do not weigh the spike {spike}")
    check_dims(got, ref, spiked, f"spike {spike}")


@pytest.mark.parametrize("spike", [1e8, np.inf])
def test_cross_v_spike_costs_its_own_dim_only(spike):
    print(f"\n[case] fp32 cross V spike {spike}", flush=True)
    h, d = 2, 64
    inp = workloads.cross_inputs(1, 100, 77, h, d, seed=15, dtype="fp32")
    inp["kv"][0, 5, 2 * h * d + 3] = spike
    with np.errstate(invalid="ignore", over="ignore"):
        ref = cross.oracle(inp, "fp32")
    check_dims(cross.run_hip(inp, torch.float32)[0], ref[0], {3}, f"spike {spike}")


@pytest.mark.parametrize("size", [2.0 ** -20, 4.0, 64.0])
@pytest.mark.parametrize("dim", [64, 128])
def test_dense_tables_of_any_size(dim, size):
    """Tables times a power of two (a scaled rotary embedding) over all dims, with gains divided by it: exactly the results
    of plain tables and gains, however far the operands are from what the gains bound."""
    print(f"\n[case] fp32 dense tables x {size} D{dim}", flush=True)
    inp = workloads.dense_inputs(1, 100, 2, dim, seed=18, dtype="fp32", half=dim // 2)
    ref = dense.oracle(inp, "xla", compute="fp32")
    small = dict(inp, q_weight=inp["q_weight"] / np.float32(size), k_weight=inp["k_weight"] / np.float32(size))
    qkv, freq = torch.from_numpy(inp["qkv"]).to("cuda"), torch.from_numpy(inp["inv_freq"]).to("cuda")
    cos, sin, mask = da.tables(100, freq, torch.from_numpy(inp["valid"]).to("cuda"), dim, torch.float32)
    got = da.dense_attention(qkv, *(torch.from_numpy(small[n]).to("cuda") for n in ("q_weight", "k_weight")), cos * size,
                             sin * size, mask, 2, dim, dim // 2, inp["eps"], lam=torch.from_numpy(inp["lam"]).to("cuda"))
    assert_fp32_parity(got.cpu().numpy(), ref, f"tables x {size}")


@pytest.mark.parametrize("workspace", [True, False], ids=["ws", "no-ws"])
@pytest.mark.parametrize("power", [10, 20, 30])
def test_band_dyt_far_below_its_bound(power, workspace):
    """alpha 2^-power with gamma 2^power: keys and queries of ordinary size, 2^-power of what gamma bounds."""
    print(f"\n[case] fp32 band DyT power {power} ws {workspace}", flush=True)
    inp = workloads.band_inputs(1, 150, 2, 64, 40, seed=19, dtype="fp32", half=16, alpha=2.0 ** -power,
                                gamma_mean=2.0 ** power)
    ref = band.oracle(inp, "xla", compute="fp32")
    cap = ba.FP32_WORKSPACE_CAP
    try:
        ba.FP32_WORKSPACE_CAP = cap if workspace else 0
        got = band.run_hip(inp, dtype=torch.float32)
    finally:
        ba.FP32_WORKSPACE_CAP = cap
    check_rows(got[0], ref[0], set(), f"power {power}")


@pytest.mark.parametrize("shape", [(1, 1, 1, 2, 64), (2, 100, 77, 2, 64), (1, 70, 128, 2, 128)],
                         ids=lambda s: "B%dL%dNk%dH%dD%d" % s)
@pytest.mark.parametrize("other", ["larger", "uneven"])
def test_cross_attend_reads_the_scales_that_the_preparation_used(shape, other):
    """The k_weight that hb_cross_attend gets only bounds the logits: another one, or the same storage edited after the
    preparation, does not change the fp32 results."""
    print(f"\n[case] fp32 cross other k_weight {shape} {other}", flush=True)
    b, length, nk, h, d = shape
    inp = workloads.cross_inputs(b, length, nk, h, d, seed=20, dtype="fp32")
    q, kv = (torch.from_numpy(inp[n]).to("cuda") for n in ("q", "kv"))
    qw, kw = (torch.from_numpy(inp[n]).to("cuda") for n in ("q_weight", "k_weight"))
    lam = torch.from_numpy(inp["lam"]).to("cuda")
    context = xattn.prepare_cross_kv(kv, kw, h, d, inp["eps"])
    ref = xattn.cross_attention(q, context, qw, inp["eps"], lam=lam)
    assert_fp32_parity(ref.cpu().numpy(), cross.oracle(inp, "fp32"), f"cross {shape}")
    factor = 8.0 if other == "larger" else 2.0 ** torch.arange(d, device="cuda").remainder(7)
    bound = dataclasses.replace(context, k_weight=kw * factor)
    assert torch.equal(xattn.cross_attention(q, bound, qw, inp["eps"], lam=lam), ref)
    kw *= factor
    assert torch.equal(xattn.cross_attention(q, context, qw, inp["eps"], lam=lam), ref)


@pytest.mark.parametrize("dim", [64, 128])
def test_dense_stages_share_no_k_weight(dim):
    """hb_dense_attend with another k_weight than hb_dense_prep: the keys are those that were prepared."""
    print(f"\n[case] fp32 dense stages D{dim}", flush=True)
    h, length, half = 2, 150, dim // 4
    inp = workloads.dense_inputs(1, length, h, dim, seed=21, dtype="fp32", half=half)
    dev = {n: torch.from_numpy(inp[n]).to("cuda") for n in ("qkv", "q_weight", "k_weight", "inv_freq", "valid", "lam")}
    cos, sin, mask = da.tables(length, dev["inv_freq"], dev["valid"], dim, torch.float32)
    workspace = torch.empty(da.workspace_bytes(torch.float32, 1, length, h, dim), dtype=torch.uint8, device="cuda")
    out = torch.empty((1, length, h * dim), device="cuda")
    lib, stream = _lib.load(), torch.cuda.current_stream().cuda_stream

    def args(k_weight):
        return (stream, dev["qkv"].data_ptr(), _lib.HB_F32, 5 * h * dim, dev["q_weight"].data_ptr(), k_weight.data_ptr(),
                cos.data_ptr(), sin.data_ptr(), half)
    shape = (1, length, h, dim, inp["eps"], workspace.data_ptr(), workspace.numel())
    _lib.check(lib.hb_dense_prep(*args(dev["k_weight"]), mask.data_ptr(), *shape), "prep")
    for weight in (dev["k_weight"], dev["k_weight"] * 2.0 ** torch.arange(dim, device="cuda").remainder(5)):
        _lib.check(lib.hb_dense_attend(*args(weight), dev["lam"].data_ptr(), out.data_ptr(), *shape), "attend")
        assert_fp32_parity(out.cpu().numpy(), dense.oracle(inp, "xla", compute="fp32"), f"stages D{dim}")


def test_identical_branches_cancel_in_split_and_wide_tiles():
    """k = k_diff and q = q_diff without lambda: exact zeros, whichever form the key tiles take."""
    print("\n[case] fp32 dense identical branches", flush=True)
    h, d, length = 2, 64, 160
    inp = workloads.dense_inputs(1, length, h, d, seed=16, dtype="fp32")
    q = inp["qkv"].reshape(1, length, 5, h * d)
    q[:, :, 3], q[:, :, 4] = q[:, :, 0], q[:, :, 1]
    inp["qkv"][0, 70, 2 * h * d] = 1e9  # the tile of keys 64-95 of head 0 is wide
    assert np.count_nonzero(dense.run_hip(inp, dtype=torch.float32, lam=False)) == 0


def test_v_code_values_survive():
    """The values that carry a tile's code (dim 0, the keys of positions 0-7: 0-3 and 8-11) come back, zeros among
    them: window 0 returns each query its own key's value, times 1 - lambda."""
    print("\n[case] fp32 band values under the code", flush=True)
    h, d, length = 1, 64, 96
    for scale in (1.0, 1e9):
        inp = workloads.band_inputs(1, length, h, d, 0, seed=17, dtype="fp32", half=16)
        v = inp["qkv"][0, :, 2 * h * d:3 * h * d]
        v[::2, 0] = 0
        v[20] *= np.float32(scale)  # split tiles, and a wide one
        got, ref = band.run_hip(inp, dtype=torch.float32), band.oracle(inp, "xla", compute="fp32")
        assert np.all(got[0, ::2, 0] == 0)
        for row in range(length):
            assert_fp32_parity(got[0, row, :1], ref[0, row, :1], f"row {row} scale {scale}")
