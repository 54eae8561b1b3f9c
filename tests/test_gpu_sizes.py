"""The plain method at the transform lengths the other parity cases do not
reach, against the FP32 oracle: 768^2 holograms (24 x 32 two-step FFT) with
crop 192 and a 384^3 volume, 2048^2 holograms with crop 128 and 256^3, and
1024^2 holograms with crop 320 and a 640^3 volume. A few angles each (seeded
ellipsoid phantom, Fermat spiral, Poisson noise); speculars bit-exact, index
volume within rel-L2 1e-5 of the FP32 oracle and within the FP64 bound
(twice the FP32 oracle's own distance, at least 1e-5) of the FP64 oracle."""
import numpy as np
import pytest

import lengths as L
from cases import rel_l2
from lengths import fp64_bound
from oracle import ref

pytestmark = pytest.mark.gpu

LAM, N0, NA = 6.33e-7, 1.333, 1.2
TOL = 1e-5


def _say(msg):
    print(msg, flush=True)


@pytest.mark.parametrize("n,nx,V,A", [(768, 96, 384, 5), (2048, 64, 256, 3),
                                      (1024, 160, 640, 4)])
def test_plain_at_size(gpu_ctx, n, nx, V, A):
    import torch
    import mtd_transmission_amd as m
    from mtd_transmission_amd import synth
    _say(f"plain method N={n} crop={2 * nx} V={V} A={A}")
    pix = nx * LAM / (NA * n)
    cx, cy = n // 2 - round(0.3 * n), n // 2 + round(0.3 * n)
    ph = synth.scale_phantom(synth.make_phantom(40 + n, 3), 0.45 * n * pix / 33.8e-6)
    kx, ky = synth.scan_fermat(A, nx, 0.95)
    holos, mask = synth.simulate_torch(n, nx, cx, cy, pix, LAM, N0, kx, ky, ph, seed=n + 1)
    gl = m.geom_derive(n, nx, V, cx, cy, NA, N0, LAM, pix)
    go = ref.derive_geom(n, nx, V, cx, cy, NA, N0, LAM, pix, 1, 1, 1)
    re = torch.empty((V, V, V), device="cuda")
    im = torch.empty_like(re)
    pos = torch.empty((2 * A,), dtype=torch.int32, device="cuda")
    gpu_ctx.reconstruct_plain(gl, holos, mask, re, im, pos)
    torch.cuda.synchronize()
    h = holos.cpu().numpy()
    f32, p32 = ref.preprocess(h, go, mask, "f32")
    assert np.array_equal(pos.cpu().numpy(), p32)
    idx32 = ref.reconstruct(f32, p32, go, "f32")[0]
    got = re.cpu().numpy() + 1j * im.cpu().numpy()
    e32 = rel_l2(got, idx32)
    del idx32
    f64, p64 = ref.preprocess(h, go, mask, "f64")
    if V <= 384:
        idx32 = ref.reconstruct(f32, p32, go, "f32")[0]
        idx64 = ref.reconstruct(f64, p64, go, "f64")[0]
        e64, bound = rel_l2(got, idx64), fp64_bound(idx32, idx64)
    else:  # the oracle's exact sum at sampled voxels
        sel = np.random.default_rng(V).integers(0, V ** 3, size=400)
        o32 = L.index_at(f32, p32, go, "f32", sel)
        o64 = L.index_at(f64, p64, go, "f64", sel)
        e64, bound = rel_l2(got.ravel()[sel], o64), fp64_bound(o32, o64)
    _say(f"  index rel-L2 vs f32 {e32:.3e}  vs f64 {e64:.3e} (bound {bound:.2e})")
    assert e32 < TOL and e64 <= bound


@pytest.mark.parametrize("V", [64, 128, 256, 364, 512])
@pytest.mark.parametrize("kind", ["band", "rows", "empty", "nan"])
def test_finalize_sparse(gpu_ctx, V, kind):
    """finalize of spectra with empty rows and planes (found by its first pass)
    against the dense transform in 64 bits: a band, scattered rows at the
    block edges of a few planes (first and last among them), nothing at all,
    and a NaN (real part), which spreads over the volume. The bound is the 1e-5 parity bar."""
    import torch
    import mtd_transmission_amd as m
    nx = V // 4
    g = m.geom_derive(8 * nx, nx, V, 4 * nx, 4 * nx, 1.2, 1.333, 6.33e-7, nx * 6.33e-7 / 9.6 / nx)
    print(f"finalize sparse V={V} {kind}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(V)
    keep = torch.zeros((V, V, V), dtype=torch.bool, device="cuda")
    if kind == "band":
        keep[V // 3:V // 2, V // 4:-V // 4, 3:] = True
    elif kind == "rows":
        for z in (0, V // 2 + 1, V - 1):
            for y in (0, 7, 8, V // 2, V - 1):
                keep[z, y, z % 5::7] = True
    elif kind == "nan":
        keep[V // 2, 3, 5] = True
    vol = torch.randn((V, V, V), dtype=torch.complex64, device="cuda", generator=gen) * keep
    if kind == "nan":
        vol[V // 2, 3, 5] = float("nan")
    cnt = torch.randint(0, 4, (V, V, V), dtype=torch.int32, device="cuda", generator=gen)
    re = torch.full((V, V, V), 7.0, device="cuda")
    im = torch.full((V, V, V), 7.0, device="cuda")
    otf = torch.full((V, V, V), 9, dtype=torch.uint8, device="cuda")
    for _ in range(2):  # the second call finds the first one's work volume
        gpu_ctx.finalize(g, vol, cnt, re, im, otf)
    torch.cuda.synchronize()
    assert torch.equal(otf.bool(), (vol.real != 0) & (otf < 2))
    if kind == "nan":
        # one part of the voxel: quarter turns move it to the other part whole
        assert bool((re.isnan() | im.isnan()).all())
        return
    t = vol.to(torch.complex128) / cnt.clamp(min=1)
    t = torch.fft.fftshift(torch.fft.ifftn(torch.fft.ifftshift(t), norm="forward"))
    kv = 2 * np.pi / g.lambda_
    t *= -g.delta_f ** 3 / (2 * g.n0 * kv * kv)
    got = torch.complex(re, im).to(torch.complex128)
    if kind == "empty":
        assert not bool(got.any())
    else:
        assert float((got - t).norm() / t.norm()) < 1e-5


def _fold_bands(V):
    # planes a block holds in registers
    nb = {448: 168, 512: 192, 576: 216, 640: 232, 704: 256, 768: 288, 1024: 368}[V]
    return [(0, 1), (V - 1, V - 1), (0, nb - 1), (V - nb, V - 1), (7, nb - 1), (7, nb), (16, 16 + nb),
            (V // 2 - nb // 2, V // 2 + nb // 2), (0, V - 1)]


@pytest.mark.parametrize("V,lo,hi", [(V, *b) for V in (448, 512, 576, 640, 704, 768, 1024)
                                     for b in _fold_bands(V)])
def test_finalize_folded_height_pass(gpu_ctx, V, lo, hi):
    """The height pass folds a band of planes onto a short transform: bands at the edges of the
    volume and of what a block holds in registers, against the closed form of a
    few normalised deltas at 100000 voxels. Bound: 30 roundings of 2^-24 over
    the three passes' 29 radix-2 levels at 1024, rounded to 2e-6."""
    import torch
    import mtd_transmission_amd as m
    nx = V // 4
    g = m.geom_derive(8 * nx, nx, V, 4 * nx, 4 * nx, 1.2, 1.333, 6.33e-7, nx * 6.33e-7 / 9.6 / nx)
    print(f"finalize folded V={V} planes {lo}..{hi}", flush=True)
    rng = np.random.default_rng(V + lo + hi)
    vol = torch.zeros((V, V, V), dtype=torch.complex64, device="cuda")
    cnt = torch.zeros((V, V, V), dtype=torch.int32, device="cuda")
    deltas = []
    for z in [lo, hi] + list(rng.integers(lo, hi + 1, 3)):
        y, x = rng.integers(0, V, 2)
        v = complex(np.complex64(rng.standard_normal() + 1j * rng.standard_normal()))
        vol[z, y, x], cnt[z, y, x] = v, 1
        deltas = [d for d in deltas if d[0] != (z, y, x)] + [((z, y, x), v)]
    re = torch.full((V, V, V), 7.0, device="cuda")
    im = torch.full((V, V, V), 7.0, device="cuda")
    gpu_ctx.finalize(g, vol, cnt, re, im, None)
    idx = torch.from_numpy(rng.integers(0, V ** 3, 100_000)).cuda()
    got = (re.view(-1)[idx].double() + 1j * im.view(-1)[idx].double()).cpu().numpy()
    z, rem = np.divmod(idx.cpu().numpy(), V * V)
    y, x = np.divmod(rem, V)
    want = np.zeros(idx.numel(), complex)
    for u, v in deltas:
        ph = sum((a - V // 2) * (b - V // 2) for a, b in zip(u, (z, y, x))) % V
        want += v * np.exp(2j * np.pi * ph / V)
    kv = 2 * np.pi / g.lambda_
    want *= -g.delta_f ** 3 / (2 * g.n0 * kv * kv)
    assert np.linalg.norm(got - want) / np.linalg.norm(want) < 2e-6


@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("V,nx", [(256, 64), (256, 20), (416, 61), (416, 104), (512, 125)])
@pytest.mark.parametrize("spec", ["centre", "rim", "corner"])
def test_forward_band_height_pass(gpu_ctx, V, nx, cplx, spec):
    """The forward model's height pass keeps a band of planes: one angle at the
    centre (half the band), the pupil's rim, and a specular past the rim, whose
    band takes several rounds, against a 64-bit transform. Bound: as the
    folded height pass, 2e-6."""
    import math
    import torch
    import mtd_transmission_amd as m
    lam = 6.33e-7
    g = m.geom_derive(8 * nx, nx, V, 4 * nx, 4 * nx, 1.2, 1.333, lam, nx * lam / 9.6 / nx)
    print(f"forward band V={V} nx={nx} {spec} cplx={cplx}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(V + nx)
    dn = torch.randn((2, V, V, V), device="cuda", generator=gen)
    if not cplx:
        dn[1] = 0
    R, C = g.rayon, 2 * nx
    far = int(0.75 * nx)
    p = {"centre": [(0, 0)], "rim": [(0, 0), (nx - 1, 0), (0, -(nx - 1)), (nx // 2, nx // 3)],
         "corner": [(far, far), (-far, far), (0, 0)]}[spec]
    A = len(p)
    pos = torch.tensor([a + nx for a, _ in p] + [b + nx for _, b in p], dtype=torch.int32).cuda()
    S = torch.full((A, C, C), 7.0, dtype=torch.complex64, device="cuda")
    gpu_ctx.forward_spectra(g, dn[0].contiguous(), dn[1].contiguous() if cplx else None, pos, S)
    t = torch.complex(dn[0].double(), dn[1].double())
    t = torch.fft.fftshift(torch.fft.fftn(torch.fft.ifftshift(t)))
    tp3 = (1.0 / (V * g.delta_f)) ** 3
    f = torch.arange(-nx, nx, device="cuda")
    fx, fy = f[None, :], f[:, None]
    r2 = fx * fx + fy * fy
    pupil = r2 < nx * nx
    h = torch.sqrt((R * R - r2).clamp(min=0).double())
    num = den = 0.0
    for a, (sx, sy) in enumerate(p):
        d = h - math.sqrt(R * R - sx * sx - sy * sy)
        z = (torch.sign(d) * torch.floor(d.abs() + 0.5)).long() + V // 2
        X, Y = fx - sx + V // 2, fy - sy + V // 2
        ok = pupil & (z >= 0) & (z < V) & (X >= 0) & (X < V) & (Y >= 0) & (Y < V)
        X, Y = X.expand(C, C), Y.expand(C, C)
        want = torch.zeros((C, C), dtype=torch.complex128, device="cuda")
        want[ok] = (-1j * (2 * 3.14159 / lam) * R * tp3 / h[ok]) * t[z[ok], Y[ok], X[ok]]
        assert not bool(S[a][~ok].any())
        num += float((S[a].to(torch.complex128) - want).abs().square().sum())
        den += float(want.abs().square().sum())
    assert (num / den) ** 0.5 < 2e-6
