"""The runtime-length transforms take fewer lines a block where a launch would leave
CUs without one."""
import pytest

pytestmark = pytest.mark.gpu


def _geometry(m, nx, V):
    lam = 6.33e-7
    return m.geom_derive(8 * nx, nx, V, 4 * nx, 4 * nx, 1.2, 1.333, lam, nx * lam / 9.6 / nx)


@pytest.mark.parametrize("C", [18, 20, 34, 92, 182, 300, 1000])
def test_alone_or_among_many(gpu_ctx, C):
    """An angle's spectrum and its fields have the same bits alone (fewest lines a
    block) and among 70 (most)."""
    import torch
    import mtd_transmission_amd as m
    nx, A = C // 2, 70
    g = _geometry(m, nx, 4 * nx)
    print(f"C={C}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(C)
    f = torch.randn((A, C, C), dtype=torch.complex64, device="cuda", generator=gen)
    pos = torch.randint(0, C, (2 * A,), dtype=torch.int32, device="cuda", generator=gen)
    many, back = torch.empty_like(f), torch.empty_like(f)
    gpu_ctx.field_to_spectrum(g, f, pos, many)
    gpu_ctx.spectra_to_fields(g, many, pos, back)
    for a in (0, 1, A - 1):
        p = pos[[a, A + a]].contiguous()
        one, two = torch.empty_like(f[:1]), torch.empty_like(f[:1])
        gpu_ctx.field_to_spectrum(g, f[a:a + 1].contiguous(), p, one)
        gpu_ctx.spectra_to_fields(g, one, p, two)
        assert torch.equal(torch.view_as_real(one[0]), torch.view_as_real(many[a]))
        assert torch.equal(torch.view_as_real(two[0]), torch.view_as_real(back[a]))
