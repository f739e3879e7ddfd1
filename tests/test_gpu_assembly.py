"""The zoomed assembly at the sizes where its y and x passes change form:
the doubled transforms with both halves in one lane and split over two
wavefronts, general zooms, lengths whose rows leave idle lanes, the
band-parallel form of small stacks and the one-plane-per-row form with and
without the phasor table.

The reference is the assembly itself in double precision from the filtered
bands that the engine holds (move_kernel's placement, an inverse transform
per band, the modulation with the float phase of cos_sin_kernel), so the fit
and the filter play no part.  A 32-bit transform of N points errs by about
eps sqrt(log2 N) = 2e-7 .. 4e-7 of its result per dimension; the bar is five
times the three dimensions' sum in quadrature."""
import numpy as np
import pytest

from cases import rel_l2, synthetic
from cudasirecon_amd import engine

pytestmark = pytest.mark.gpu

# nx, ny, nz, phases, parameters
CASES = [
    (16, 24, 1, 3, {}),                      # shortest rows; split halves with two lanes per column
    (40, 100, 1, 3, {}),                     # 10 and 7 columns per lane, idle lanes
    (80, 48, 5, 5, {}),
    (144, 160, 3, 5, dict(bDampenOrder0=0)),                    # fewer planes than the phasor table needs
    (300, 360, 1, 3, {}),
    (128, 96, 64, 5, {}),                    # phasor table, rows of several planes per workgroup
    (640, 576, 1, 5, {}),                    # 5 phases: seven bands side by side
    (1000, 720, 1, 3, {}),                   # above one wavefront per SIMD: phasors in the kernel
    (1200, 1280, 1, 3, {}),                  # both halves in one lane at 64 lanes
    (96, 64, 6, 5, dict(zoomfact=1.5)),      # general zoom
    (64, 96, 7, 5, dict(zoomfact=3.0)),
    (800, 640, 1, 3, dict(zoomfact=1.5)),
    (128, 128, 40, 5, dict(zoomfact=1.25)),  # general zoom with the phasor table
    (1024, 1600, 1, 3, dict(zoomfact=1.25)),
]


def place(full, nx, ny, nz, zdim, ydim, xdim):
    """move_kernel's placement of a spectrum [nz][ny][nx] (full x) on the zoomed grid."""
    x = np.arange(-(nx // 2 - 1), nx - nx // 2 + 1)
    y = np.arange(-(ny // 2 - 1), ny - ny // 2 + 1)
    z = np.arange(-(nz // 2 - 1), nz - nz // 2 + 1) if nz > 1 else np.zeros(1, int)
    out = np.zeros((zdim, ydim, xdim), np.complex128)
    src = full[np.ix_(z % nz, y % ny, x % nx)]
    np.add.at(out, np.ix_(z % zdim, y % ydim, x % xdim), src)
    return out


def mirrored(half, nx):
    """The full spectrum of a half-stored band [nz][ny][nx/2+1] (Hermitian in (x, y, z))."""
    nz, ny, nxh = half.shape
    out = np.zeros((nz, ny, nx), np.complex128)
    out[:, :, :nxh] = half
    m = half[(-np.arange(nz)) % nz][:, (-np.arange(ny)) % ny]
    for x in range(nxh, nx):
        out[:, :, x] = np.conj(m[:, :, nx - x])
    return out


def assembled(p, bands, fits):
    norders = p.nphases // 2 + 1
    xdim, ydim, zdim = int(round(p.zoomfact * p.nx)), int(round(p.zoomfact * p.ny)), p.z_zoom * p.nz
    f4 = np.float32
    out = np.zeros((zdim, ydim, xdim))
    n = zdim * ydim * xdim
    for d in range(p.ndirs):
        for o in range(norders):
            if o == 0:
                v = mirrored(bands[d][0], p.nx)
            else:
                v = mirrored(bands[d][2 * o - 1], p.nx) + 1j * mirrored(bands[d][2 * o], p.nx)
            r = np.fft.ifftn(place(v, p.nx, p.ny, p.nz, zdim, ydim, xdim)) * n
            if o == 0:
                out += r.real
                continue
            s1 = (np.arange(xdim) - xdim // 2).astype(f4) * (f4(fits[d].k0x) * f4(o))
            s2 = (np.arange(ydim) - ydim // 2).astype(f4) * (f4(fits[d].k0y) * f4(o))
            angle = (2.0 * np.pi * (s1[None, :] + s2[:, None]).astype(np.float64) *
                     np.float64(f4(p.dxy) / f4(p.zoomfact))).astype(f4).astype(np.float64)
            out += 2 * (r.real * np.cos(angle) - r.imag * np.sin(angle))
    return out


# zooms above two and the two forms of the phasors: the halves of a length with empty
# frequencies (1000, 1152, 1280, 2048, 2400 points; an odd height), whole lengths beside
# them (3072, 4096), the table over the output rows in parts (the last one shorter),
# phasors in the kernel with and without a remainder of their group
ZOOMS = [
    (80, 75, 4, 5, dict(zoomfact=16.0)),
    (200, 240, 1, 3, dict(zoomfact=5.0)),
    (360, 400, 3, 5, dict(zoomfact=3.2, bDampenOrder0=0)),
    (512, 48, 5, 5, dict(zoomfact=4.0)),
    (256, 300, 3, 5, dict(zoomfact=8.0, bDampenOrder0=0)),
    (384, 96, 5, 5, dict(zoomfact=8.0)),
    (400, 512, 6, 5, dict(zoomfact=4.0)),
    (512, 16, 1, 3, dict(zoomfact=8.0)),
    (240, 320, 8, 5, dict(zoomfact=4.0)),
]


@pytest.mark.parametrize("nx,ny,nz,phases,kw", CASES + ZOOMS)
def test_assembly_sizes(nx, ny, nz, phases, kw):
    print("case %dx%dx%d, %d phases, %s" % (nx, ny, nz, phases, kw), flush=True)
    p, otf, raw, _ = synthetic(nx, ny, nz, nphases=phases, seed=nx + ny, gpu=True, **kw)
    with engine.Reconstructor(p, otf) as r:
        r.set_raw(raw)
        r.load_and_rescale(0)
        r.set_time(0)
        r.process_volume()
        vol = r.result()
        fits = [r.fit(d) for d in range(p.ndirs)]
        bands = [[r.band(d, b) for b in range(p.nphases)] for d in range(p.ndirs)]
    ref = assembled(p, bands, fits)
    assert vol.shape == ref.shape and np.isfinite(vol).all()
    err = rel_l2(vol, ref)
    eps = 2.0 ** -24
    bar = 5 * eps * np.sqrt(sum(np.log2(n) for n in vol.shape))
    print("  rel-L2 %.2e, bar %.2e" % (err, bar), flush=True)
    assert err < bar
