"""The height pass of a volume whose band does not fit the folded form: speculars
past the pupil's rim, near the Ewald sphere, beside one at the centre. The
adjoint (and with it the plain method, the same passes) then takes the whole
transform, chosen on the device."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# planes that a folded block holds in registers
HELD = {448: 168, 512: 192, 576: 216, 640: 232}


def _speculars(nx, R, wide):
    """Speculars and the height band of their hits, relative to V/2."""
    t = np.array([0.8, 2.4, 4.0])
    far = 0.995 * R if wide else 0.9 * nx
    f = np.stack([np.trunc(far * np.cos(t)), np.trunc(far * np.sin(t))], 1).astype(int)
    f = np.concatenate([[(0, 0)], np.clip(f, -nx, nx - 1)])
    fz = np.sqrt(np.maximum(R * R - (f * f).sum(1), 0.0))
    rim = np.sqrt(R * R - nx * nx + 1.0)
    return f, int(np.round(rim - fz.max())), int(np.round(R - fz.min()))


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("V", [448, 512, 576, 640])
def test_adjoint_band(gpu_ctx, V, wide):
    """Bound: 2e-6 of the norm, as the folded pass has it (30 roundings of 2^-24
    over the passes' levels, the sums' of at most 4 terms among them)."""
    import torch
    import mtd_transmission_amd as m
    nx = V // 4
    lam = 6.33e-7
    g = m.geom_derive(8 * nx, nx, V, 4 * nx, 4 * nx, 1.2, 1.333, lam, nx * lam / 9.6 / nx)
    R, C = int(g.rayon), 2 * nx
    f, lo, hi = _speculars(nx, R, wide)
    print(f"V={V} band {lo}..{hi} of {HELD[V]}", flush=True)
    assert hi - lo + 1 > HELD[V] if wide else hi - lo + 1 <= HELD[V] - 16
    A = len(f)
    pos = torch.from_numpy(np.concatenate([f[:, 0], f[:, 1]]) + nx).to(torch.int32).cuda()
    gen = torch.Generator(device="cuda").manual_seed(V)
    S = torch.randn((A, C, C), dtype=torch.complex64, device="cuda", generator=gen)
    re, im = (torch.full((V, V, V), 7.0, device="cuda") for _ in range(2))
    gpu_ctx.adjoint_spectra(g, S, pos, re, im)
    one = torch.full((V, V, V), 7.0, device="cuda")
    gpu_ctx.adjoint_spectra(g, S, pos, one, None)
    assert torch.equal(one, re)
    del one
    ax = torch.arange(-nx, nx, device="cuda")
    fx, fy = ax[None, :].expand(C, C), ax[:, None].expand(C, C)
    r2 = fx * fx + fy * fy
    h = torch.sqrt((R * R - r2).clamp(min=0).double())
    t = torch.zeros(V ** 3, dtype=torch.complex128, device="cuda")
    for a, (sx, sy) in enumerate(f.tolist()):
        if R * R - sx * sx - sy * sy < 0:
            continue
        d = h - float(np.sqrt(R * R - sx * sx - sy * sy))
        z = (torch.sign(d) * torch.floor(d.abs() + 0.5)).long() + V // 2
        X, Y = fx - sx + V // 2, fy - sy + V // 2
        ok = (r2 < nx * nx) & (z >= 0) & (z < V) & (X >= 0) & (X < V) & (Y >= 0) & (Y < V)
        q = (2 * 3.14159 / lam) * R / h[ok]
        i = (z[ok] * V + Y[ok]) * V + X[ok]
        t.index_add_(0, i, 1j * q * S[a].to(torch.complex128)[ok])
    t = t.view(V, V, V)
    for d in range(3):
        t = torch.fft.fftshift(torch.fft.ifft(torch.fft.ifftshift(t, d), dim=d, norm="forward"), d)
    t *= (1.0 / (V * g.delta_f)) ** 3
    num = (re.double() - t.real).square().sum() + (im.double() - t.imag).square().sum()
    assert float((num / t.abs().square().sum()).sqrt()) < 2e-6
