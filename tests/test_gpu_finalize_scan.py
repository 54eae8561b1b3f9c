"""mtd_finalize on both sides of the volume side from which it looks for the
spectrum's band: sides up to 128 transform every plane, larger ones scan the
rows first and read the counts only where a wave found something. Spectra with
a few voxels in a row (most waves of the block find nothing), a band, and every
voxel; counts that are not zero beside empty voxels; the OTF at any address."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("kind", ["few", "band", "dense"])
@pytest.mark.parametrize("V", [32, 78, 124, 128, 130, 140, 256, 320])
def test_scan_line(gpu_ctx, V, kind, shift):
    """Bound: 1e-5 of the norm, the parity bar of FP32 transforms (at most 3 x 3
    lines of 9 passes, each below 2^-22 of its rms)."""
    import torch
    import mtd_transmission_amd as m
    nx = V // 4
    g = m.geom_derive(8 * nx, nx, V, 4 * nx, 4 * nx, 1.2, 1.333, 6.33e-7, nx * 6.33e-7 / 9.6 / nx)
    print(f"finalize V={V} {kind} otf+{shift}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(V)
    vol = torch.randn((V, V, V), dtype=torch.complex64, device="cuda", generator=gen)
    cnt = torch.randint(0, 4, (V, V, V), dtype=torch.int32, device="cuda", generator=gen)
    if kind == "band":
        vol[: V // 3] = 0
        vol[V - V // 4:] = 0
    elif kind == "few":
        keep = torch.zeros((V, V, V), dtype=torch.bool, device="cuda")
        for z, y, x in ((0, 0, 0), (V // 2, V // 2, V - 1), (V - 1, 3, V // 2), (V // 3, V - 1, 1)):
            keep[z, y, x] = True
        vol *= keep
    re, im = (torch.full((V, V, V), 7.0, device="cuda") for _ in range(2))
    buf = torch.full((V ** 3 + 1,), 9, dtype=torch.uint8, device="cuda")
    otf = buf[shift: V ** 3 + shift]
    gpu_ctx.finalize(g, vol, cnt, re, im, otf)
    t = vol.to(torch.complex128) / cnt.clamp(min=1)
    assert torch.equal(otf.view(V, V, V), (t.real != 0).to(torch.uint8))
    assert int(buf[0 if shift else V ** 3]) == 9
    t = torch.fft.fftshift(torch.fft.ifftn(torch.fft.ifftshift(t), norm="forward"))
    kv = 2 * np.pi / g.lambda_
    t *= -g.delta_f ** 3 / (2 * g.n0 * kv * kv)
    got = torch.complex(re, im).to(torch.complex128)
    assert float((got - t).norm() / t.norm()) < 1e-5
