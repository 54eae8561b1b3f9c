"""The forward model's factor of a bin, kv R Tp^3 / h(|fd|^2), is rounded to
FP32 once. The spectrum of a single voxel at index 0 is +-1 at every bin, exactly
(every pass multiplies its one value by W^0 and adds zeros; not so for a chirp, so no
length here has a prime factor above 13), so each sample is
the factor itself: half a unit in the last place from its 64-bit value (the
factor's own double rounding adds less than 2^-50). A scaled transform, a rounded
weight and their product are each another half unit off."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V,nx", [(64, 16), (78, 16), (256, 64), (512, 125)])
def test_factor_rounded_once(gpu_ctx, V, nx):
    import torch
    import mtd_transmission_amd as m
    lam = 6.33e-7
    g = m.geom_derive(8 * nx, nx, V, 4 * nx, 4 * nx, 1.2, 1.333, lam, nx * lam / 9.6 / nx)
    print(f"V={V} nx={nx}", flush=True)
    C, R = 2 * nx, g.rayon
    dn = torch.zeros((V, V, V), device="cuda")
    dn[0, 0, 0] = 1.0
    pos = torch.tensor([nx, nx + nx // 2, nx, nx - nx // 3], dtype=torch.int32).cuda()
    S = torch.full((2, C, C), 7.0, dtype=torch.complex64, device="cuda")
    gpu_ctx.forward_spectra(g, dn, None, pos, S)
    S = S.cpu().numpy()
    f = np.arange(-nx, nx)
    r2 = f[None, :] ** 2 + f[:, None] ** 2
    pupil = r2 < g.coef_na * nx * nx
    kv = 2 * 3.14159 / g.lambda_
    want = kv * R / np.sqrt(np.where(pupil, R * R - r2, 1.0)) / (V * g.delta_f) ** 3
    for a in range(2):
        assert not S[a][~pupil].any() and not S[a].real.any()
        got = np.abs(S[a].imag[pupil]).astype(np.float64)
        assert (np.abs(got - want[pupil]) <= want[pupil] * (2.0 ** -24 + 2.0 ** -48)).all()
