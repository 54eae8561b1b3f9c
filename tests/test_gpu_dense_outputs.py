"""Dense Ewald outputs that stay in the last cache come from the gather alone, larger
ones from the gather and a fill."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _geometry(m, nx, V):
    lam = 6.33e-7
    return m.geom_derive(8 * nx, nx, V, 4 * nx, 4 * nx, 1.2, 1.333, lam, nx * lam / 9.6 / nx)


@pytest.mark.parametrize("A", [1, 3])
@pytest.mark.parametrize("V", [64, 78, 286, 288, 302, 304])
def test_dense_outputs(gpu_ctx, V, A):
    """Both sides of the fill's line: counts exact, sums of at most A terms of one
    product each within A 2^-22 of the largest, zeros everywhere else."""
    import torch
    import mtd_transmission_amd as m
    nx = 15
    g = _geometry(m, nx, V)
    assert g.rayon < V // 2
    print(f"V={V} A={A}", flush=True)
    C, R = 2 * nx, int(g.rayon)
    p = [(0, 0), (9, -4), (-13, 2)][:A]
    pos = torch.tensor([x + nx for x, _ in p] + [y + nx for _, y in p], dtype=torch.int32).cuda()
    gen = torch.Generator(device="cuda").manual_seed(V)
    S = torch.randn((A, C, C), dtype=torch.complex64, device="cuda", generator=gen)
    vol = torch.full((V, V, V), 7.0, dtype=torch.complex64, device="cuda")
    cnt = torch.full((V, V, V), 7, dtype=torch.int32, device="cuda")
    gpu_ctx.ewald_scatter(g, S, pos, vol, cnt)
    f = np.arange(-nx, nx)
    fx, fy = np.broadcast_arrays(f[None, :], f[:, None])
    r2 = fx * fx + fy * fy
    ok = r2 < g.coef_na * nx * nx
    h = np.sqrt((R * R - r2[ok]).astype(np.float64))
    k0 = float(np.float32(np.float32(2 * 3.14159 / g.lambda_) * np.float32(g.n0)))
    beta = (k0 / 3.14159) * (-2 * 3.14159) * (h / R)
    want, hits = np.zeros(V ** 3, np.complex128), np.zeros(V ** 3, np.int32)
    for a, (sx, sy) in enumerate(p):
        d = h - np.sqrt(float(R * R - sx * sx - sy * sy))
        z = (np.sign(d) * np.floor(np.abs(d) + 0.5)).astype(int) + V // 2
        i = (z * V + fy[ok] - sy + V // 2) * V + fx[ok] - sx + V // 2
        np.add.at(want, i, 1j * beta * S[a].cpu().numpy()[ok])
        np.add.at(hits, i, 1)
    assert np.array_equal(cnt.cpu().numpy().reshape(-1), hits)
    got = vol.cpu().numpy().reshape(-1)
    assert not got[hits == 0].any()
    assert np.abs(got - want).max() <= A * 2.0 ** -22 * np.abs(want).max()
