"""The row-per-workgroup norms (hb_rms_modulate, hb_residual_rms) where the row leaves lanes, waves or turns uneven:
one chunk, a partial wave, the widest row that has a lane per chunk, wider rows that take turns, more rows than a
launch has workgroups, and a weight that is aligned only as floats. fp32 contract of the block's other tests: 2e-6 of
the row's largest value; bf16: one rounding step of it, 2^-8."""
import pytest
import torch

from hummingbird_amd import elementwise as ew

pytestmark = pytest.mark.gpu
DEV = "cuda"


def reference(x, w, eps, scale, shift):
    x = x.double()
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()
    return y * (1 + scale.double()[:, None]) + shift.double()[:, None]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows, channels", [(3, 8), (2, 520), (5, 2040), (3, 2048), (2, 2056), (2, 6152),
                                            ((1 << 19) + 9, 8)])
def test_norm_shapes(dtype, rows, channels):
    print(f"[case] {dtype} {rows} x {channels}", flush=True)
    gen = torch.Generator(device=DEV).manual_seed(channels)
    h = torch.randn(2, rows, channels, device=DEV, generator=gen).to(dtype)
    x = torch.randn(2, rows, channels, device=DEV, generator=gen).to(dtype)
    scale, shift = (0.3 * torch.randn(2, 2, channels, device=DEV, generator=gen)).to(dtype)
    buf = torch.empty(channels + 1, device=DEV)
    w = buf[1:].copy_(1 + 0.1 * torch.randn(channels, device=DEV, generator=gen))
    assert w.data_ptr() % 16 == 4
    got = ew.rms_modulate(h, w, 1e-5, scale, shift)
    ref = reference(h, w, 1e-5, scale, shift)
    # bf16 rounds after the norm, 1 + scale, the product and the shift: at most four steps of 2^-8 (2^-9 each, and
    # an operand can be twice the result)
    bound = (2e-6 if dtype == torch.float32 else 4 * 2.0 ** -8) * ref.abs().amax(-1, keepdim=True).clamp_min(1.0)
    assert ((got.double() - ref).abs() <= bound).all()
    if channels <= 2048:
        out_h, out_y = ew.residual_rms(h, x, w, 1e-5, scale=scale, shift=shift)
        assert torch.equal(out_h, ew.gated_residual(h, x))
        assert torch.equal(out_y, ew.rms_modulate(out_h, w, 1e-5, scale, shift))
