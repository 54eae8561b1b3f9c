"""The Volkov unwrapping's transform lengths: compiled crop sides (balanced
and unbalanced register splits, column blocks that do and do not divide the
side) and runtime-length ones, against the FP64 oracle; and phases of fields
whose |u|^2 leaves the float range."""
import numpy as np
import pytest

from cases import LAM, N0, NA, rel_l2
from lengths import fp64_bound
from oracle import ref

pytestmark = pytest.mark.gpu


def _crops(C, A, seed):
    """Centred crops whose demodulated fields wrap several times."""
    rng = np.random.default_rng(seed)
    y, x = np.mgrid[0:C, 0:C] / C - 0.5
    out = []
    for _ in range(A):
        cx, cy = rng.uniform(-0.1, 0.1, 2)
        r2 = (x - cx) ** 2 + (y - cy) ** 2
        phi = 9.0 * np.exp(-r2 / 0.06) + rng.uniform(-2, 2) * x
        u = (1 - 0.2 * np.exp(-r2 / 0.04)) * np.exp(1j * phi)
        out.append(np.roll(np.fft.fft2(np.fft.ifftshift(u)) / C ** 2, (3, 5), (0, 1)))
    return np.stack(out).astype(np.complex64)


def _run(ctx, nx, crops, mask):
    import torch
    import mtd_transmission_amd as m
    C, A = 2 * nx, len(crops)
    pix = nx * LAM / (NA * 8 * nx)
    g = m.geom_derive(8 * nx, nx, 4 * nx, 4 * nx, 4 * nx, NA, N0, LAM, pix, born=0, c_aber=1,
                      deroul=1)
    pos = torch.empty((2 * A,), dtype=torch.int32, device="cuda")
    fields = torch.empty((A, C, C), dtype=torch.complex64, device="cuda")
    ctx.crop_to_field(g, torch.from_numpy(crops).cuda(), mask, pos, fields)
    torch.cuda.synchronize()
    return fields.cpu().numpy(), pos.cpu().numpy()


@pytest.mark.parametrize("C", [32, 52, 64, 104, 122, 128, 160, 182, 192, 224, 250, 256, 288, 320,
                               352, 384, 512])
def test_volkov_lengths(gpu_ctx, C):
    nx, A = C // 2, 2
    print(f"volkov crop {C}", flush=True)
    crops = _crops(C, A, seed=C)
    mask = np.full((C, C), 255, np.uint8)
    mask[C // 4:-C // 4, C // 4:-C // 4] = 0
    got, pos = _run(gpu_ctx, nx, crops, mask)
    go = ref.derive_geom(8 * nx, nx, 4 * nx, 4 * nx, 4 * nx, NA, N0, LAM,
                         nx * LAM / (NA * 8 * nx), 1, 1, 1, born=0, c_aber=1, deroul=1)
    plan = ref.LsqPlan.build(mask)
    want = {}
    for prec in ("f32", "f64"):
        w = []
        for a in range(A):
            py, px = divmod(int(ref.coord_spec(crops[a], prec)), C)
            assert (px, py) == (pos[a], pos[A + a])
            w.append(ref.form_field(ref.demod(crops[a], px, py, prec), plan, go, prec, angle=a))
        want[prec] = np.stack(w)
    e, bound = rel_l2(got, want["f64"]), fp64_bound(want["f32"], want["f64"])
    print(f"  fields rel-L2 vs f64 {e:.3e} (bound {bound:.2e})", flush=True)
    assert e <= bound


@pytest.mark.parametrize("scale", [2.0 ** -70, 2.0 ** 70])
def test_volkov_amplitude_range(gpu_ctx, scale):
    """|u|^2 under- or overflows: the phase is that of the unscaled field."""
    C = 64
    crops = _crops(C, 2, seed=1)
    crops[:, 0, 0] = 0  # the specular search squares this bin
    want, _ = _run(gpu_ctx, C // 2, crops, None)
    got, _ = _run(gpu_ctx, C // 2, (crops * np.float32(scale)).astype(np.complex64), None)
    assert rel_l2(got.imag, want.imag) < 1e-5
