"""Query rows prepared in the MFMA operand layout (csrc/query.h): every rotary width (the partner chunk in the same
lane, in the other lane half, none), every workgroup form of the dense kernel and both of the tiled band kernel, with
norm parameters that are aligned only as floats."""
import numpy as np
import pytest
import torch

from hummingbird_amd import band_attention as ba
from hummingbird_amd import dense_attention as da
from hummingbird_amd import workloads
from oracle import band as oband
from oracle import dense as odense
from tests.util import assert_bf16_parity

pytestmark = pytest.mark.gpu
DEV = "cuda"


def off_by_one_float(x) -> torch.Tensor:
    """The same values at an address that is 4 mod 16."""
    buf = torch.empty(len(x) + 1, dtype=torch.float32, device=DEV)
    buf[1:] = torch.from_numpy(x)
    assert buf[1:].data_ptr() % 16 == 4
    return buf[1:]


def check(got: torch.Tensor, ref: np.ndarray) -> None:
    """The bf16 contract, 2e-2, of each output, per unit of it where it is larger than 1 (with 33 keys a few of the million
    pass 2, where one bf16 step alone is 2^-6). `ref` has the fused kernels' cast points: the plain chain also rounds its
    logits to bf16, which alone moves a probability by 2 %."""
    scale = np.maximum(1.0, np.abs(ref))
    assert_bf16_parity(got.float().cpu().numpy() / scale, ref / scale)


# one 128-query block per head: at D = 64, 2 heads run as 64-query workgroups and 130 as 128-query ones; at D = 128
# workgroups of 8 waves, one and a chip full
@pytest.mark.parametrize("heads, dim, half", [(n, 64, h) for n in (2, 130) for h in (0, 8, 16, 24, 32)] +
                         [(n, 128, h) for n in (2, 256) for h in range(0, 65, 8)])
def test_dense_rotary_widths(heads, dim, half):
    length = 33
    print(f"[case] dense {heads} x {dim}, half {half}", flush=True)
    d = workloads.dense_inputs(1, length, heads, dim, seed=half + dim, half=half, mask_tail=3)
    cos, sin, mask = da.tables(length, torch.from_numpy(d["inv_freq"]).to(DEV), torch.from_numpy(d["valid"]).to(DEV),
                               dim, torch.bfloat16)
    got = da.dense_attention(torch.from_numpy(d["qkv"]).to(DEV, torch.bfloat16), off_by_one_float(d["q_weight"]),
                             off_by_one_float(d["k_weight"]), cos, sin, mask, heads, dim, half, d["eps"],
                             lam=torch.from_numpy(d["lam"]).to(DEV))
    ref = odense.dense_fused(d["qkv"], d["q_weight"], d["k_weight"], d["inv_freq"], d["valid"], heads, dim, d["eps"],
                             d["lam"], "bf16")
    check(got, ref)


@pytest.mark.parametrize("dim, half", [(64, h) for h in (0, 8, 16, 24, 32)] + [(128, h) for h in range(0, 65, 8)])
def test_tiled_band_rotary_widths(dim, half):
    length, window = 161, 130
    print(f"[case] band {dim}, half {half}", flush=True)
    b = workloads.band_inputs(1, length, 2, dim, window, seed=half + dim, half=half)
    norm = lambda n: {k: torch.as_tensor(np.asarray(v)).to(DEV) for k, v in n.items()}  # noqa: E731
    got = ba.band_attention(torch.from_numpy(b["qkv"]).to(DEV, torch.bfloat16), norm(b["q_norm"]), norm(b["k_norm"]),
                            torch.from_numpy(b["inv_freq"]).to(DEV), 2, dim, window,
                            lam=torch.from_numpy(b["lam"]).to(DEV))
    ref = oband.band_fused(b["qkv"], b["q_norm"], b["k_norm"], b["inv_freq"], 2, dim, window, b["lam"], "bf16")
    check(got, ref)


@pytest.mark.parametrize("heads, length", [(100, 700), (101, 700), (102, 700), (110, 700), (116, 700), (117, 700)])
def test_dense_forms_past_two_workgroups_a_cu(heads, length):
    """11 blocks of 64 queries a head: 1100 to 1287 on 256 CUs, both sides of where 64-query workgroups end (five a CU),
    with a ragged last block; every head against the exact softmax of a sample of its queries."""
    print(f"[case] dense {heads} heads, L = {length}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(heads)
    qkv = torch.randn(1, length, 5 * heads * 64, device=DEV, generator=gen).bfloat16()
    one = torch.ones(64, device=DEV)
    got = da.dense_attention(qkv, one, one, None, None, None, heads, 64, 0, 1e-6).double().reshape(length, heads, 64)
    q, k, v, qd, kd = (t.double().reshape(length, heads, 64).transpose(0, 1) for t in qkv[0].split(heads * 64, dim=-1))
    rms = lambda t: t * torch.rsqrt((t * t).mean(-1, keepdim=True) + 1e-6)  # noqa: E731
    rows = torch.tensor([0, 63, 64, 127, 128, 639, 640, 699], device=DEV)

    def attend(a, b):
        logits = (rms(a[:, rows])[:, :, None] * rms(b)[:, None]).sum(-1) / 8.0
        return (torch.softmax(logits, -1)[..., None] * v[:, None]).sum(2)
    ref = (attend(q, k) - attend(qd, kd)).transpose(0, 1)
    assert (got[rows] - ref).abs().max() <= 2e-2  # the bf16 contract
