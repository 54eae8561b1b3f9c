"""Crops and demodulated fields at sides without a compiled FFT, bit for bit.

The angle and the logarithm of the demodulated field amplify a last-bit change
of it where the field is faint: reordered transforms moved unwrapped fields by
3e-3 of their scale at single pixels and doubled the index volume's error
against 64 bits. So the order of roundings on the way from holograms to the
demodulated field is part of the result. tests/golden/uncompiled_lengths.npz
holds the library's outputs in that order (two Stockham buffers per block, the
radices 8, 4, 2, 3, 5, 7, 11, 13 in turn, Bluestein over a power of two), for
every radix first, last and repeated, the longest lines (4096 points, direct
and Bluestein) and butterfly counts that leave a thread's last ones idle.
"""
import os

import numpy as np
import pytest

from cases import LAM, N0, NA

GOLDEN = os.path.join(os.path.dirname(__file__), "golden", "uncompiled_lengths.npz")

# (hologram side, NXMAX): direct and Bluestein holograms on direct and
# Bluestein crops
CASES = [(600, 15), (2046, 17), (552, 18), (4096, 11), (1394, 13), (338, 13), (2002, 14),
         (3000, 12), (90, 7), (768, 11), (3388, 9), (126, 10)]
A = 2


def holograms(n):
    """[A][n][n] uint16 by integer arithmetic alone: fringes and texture."""
    y, x = np.mgrid[0:n, 0:n].astype(np.uint64)
    a = np.arange(A, dtype=np.uint64)[:, None, None] + 1
    v = (x * 37 + y * 53 * a) % 251 + ((x * x * a + y * y * 3 + x * y * 7) % 1021) * 3
    return v.astype(np.uint16)


def positions(nx):
    """Speculars in the crop: all x, then all y."""
    c = 2 * nx
    return np.array([nx + 2, c - 1, nx - 3, 1], np.int32)


def geometry(m, n, nx):
    pix = nx * LAM / (NA * n)
    return m.geom_derive(n, nx, 4 * nx, n // 2 - round(0.3 * n), n // 2 + round(0.3 * n), NA, N0,
                         LAM, pix, 1.0, 1.0, 1.0, 1.0, 1, 1, 0)


def stages(m, ctx, n, nx):
    import torch
    c = 2 * nx
    pos = positions(nx)
    assert pos.min() >= 0 and pos.max() < c
    g = geometry(m, n, nx)
    crops, u = (torch.zeros((A, c, c), dtype=torch.complex64, device="cuda") for _ in range(2))
    ctx.holo_to_crop(g, torch.from_numpy(holograms(n)).cuda(), crops)
    ctx.demodulate(g, crops, torch.from_numpy(pos).cuda(), u)
    return crops.cpu().numpy(), u.cpu().numpy()


@pytest.mark.gpu
@pytest.mark.parametrize("n,nx", CASES)
def test_same_bits(gpu_ctx, n, nx):
    import mtd_transmission_amd as m
    want = np.load(GOLDEN)
    print(n, nx, flush=True)
    for name, got in zip(("crops", "u"), stages(m, gpu_ctx, n, nx)):
        ref = want["%s_%d_%d" % (name, n, nx)]
        off = np.abs(got - ref).max() / np.sqrt(np.mean(np.abs(ref) ** 2))
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32)), (name, off)


def test_stored_fields_are_the_transform():
    """The stored values are the 64-bit transforms' (a window, two 2-D FFTs) but
    for FP32 rounding: each of the at most 4 x 3 x 7 passes of both stages
    (Bluestein: three lines' worth) rounds by about 3 x 2^-24 of the rms."""
    from oracle import ref
    want = np.load(GOLDEN)
    for n, nx in ((338, 13), (90, 7), (126, 10)):
        c = 2 * nx
        x0, y0 = n // 2 - round(0.3 * n) - nx, n // 2 + round(0.3 * n) - nx
        h = holograms(n).astype(np.float64) * ref.tukey2d(n, 0.05)
        pos = positions(nx)
        for a in range(A):
            f = np.fft.fftshift(np.fft.fft2(np.fft.fftshift(h[a]))) / n ** 2
            f = f[y0:y0 + c, x0:x0 + c]
            got = want["crops_%d_%d" % (n, nx)][a]
            tol = 84 * 3 * 2.0 ** -24
            # the crop holds less than the frame: its rounding is of the frame's rms
            scale = np.sqrt(np.mean(np.abs(h[a]) ** 2) / n ** 2 * c * c)
            assert np.linalg.norm(got - f) <= tol * scale
            u = np.fft.fftshift(np.fft.ifft2(np.roll(f, (-pos[a + A], -pos[a]), (0, 1)),
                                             norm="forward"))
            got = want["u_%d_%d" % (n, nx)][a]
            assert np.linalg.norm(got - u) <= tol * scale * c
