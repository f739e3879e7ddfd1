"""Depths whose z transforms run in registers (2 to 64 planes with prime
factors up to 31), beside ones that do not, and the columns of the bands that
the forward pass leaves until somebody asks for them.

  * whole spectra: every separated band against numpy's transform of the same
    stack in double.  The bar is five times eps sqrt(log2) per dimension, in
    quadrature, of the phase images that the band is a sum of (a side band is
    a small difference of them, and each is rounded on its own);
  * the assembly's z pass at those depths, unpadded, with an axial zoom and
    with an odd height, against the double-precision assembly of
    test_gpu_assembly.py;
  * a stack whose bands are read, replaced or re-parametrised between loading
    and processing gives the result of the untouched one, bit for bit.
"""
import numpy as np
import pytest

from cases import rel_l2, synthetic
from cudasirecon_amd import engine
from test_gpu_assembly import assembled

pytestmark = pytest.mark.gpu

DEPTHS = [5, 7, 9, 11, 13, 17, 19, 21, 22, 23, 26, 29, 31, 32, 33, 37, 46, 48, 51, 58, 62, 64, 72]


def loaded(p, otf, raw):
    r = engine.Reconstructor(p, otf)
    r.set_raw(raw)
    r.load_and_rescale(0)
    r.set_time(0)
    return r


def bands_of(p, raw):
    """The separated bands' 3D spectra in double: [dir][band][z][y][nx/2+1] (no rescale, no edge blend)."""
    a = (raw.reshape(p.ndirs, p.nz, p.nphases, p.ny, p.nx).astype(np.float64) - np.float64(p.constbkgd))
    a /= p.nx * p.ny * p.nz * p.zoomfact ** 2 * p.z_zoom * p.ndirs
    phi = 2 * np.pi * np.arange(p.nphases) / p.nphases
    rows = [np.ones(p.nphases)]
    for o in range(1, p.nphases // 2 + 1):
        rows += [np.cos(o * phi), np.sin(o * phi)]
    return [[(np.fft.rfftn((a[d] * m[None, :, None, None]).sum(1), axes=(0, 1, 2)),
              np.linalg.norm(a[d] * m[None, :, None, None]) * np.sqrt(p.nx * p.ny * p.nz / 2)) for m in rows]
            for d in range(p.ndirs)]


@pytest.mark.parametrize("nz", DEPTHS)
def test_depth(nz):
    print("depth", nz, flush=True)
    p, otf, raw, _ = synthetic(48, 40, nz, seed=nz, gpu=True, do_rescale=0, napodize=0,
                               bDampenOrder0=0 if nz < 4 else 1)
    with loaded(p, otf, raw) as r:
        want = bands_of(p, raw)
        bar = 5 * 2.0 ** -24 * np.sqrt(np.log2(p.nx) + np.log2(p.ny) + np.log2(nz))
        if nz > 31 and any(nz % q == 0 for q in (37,)):
            bar *= 4  # a direct sum of nz terms
        for d in range(p.ndirs):
            for b in range(p.nphases):
                spec, size = want[d][b]  # (the norm of the terms' half spectra)
                err = np.linalg.norm(r.band(d, b) - spec) / size
                assert err < bar, (d, b, err, bar)
        r.process_volume()
        vol = r.result()
        fits = [r.fit(d) for d in range(p.ndirs)]
        got = [[r.band(d, b) for b in range(p.nphases)] for d in range(p.ndirs)]
    err = rel_l2(vol, assembled(p, got, fits))
    print("  assembly rel-L2 %.2e, bar %.2e" % (err, bar), flush=True)
    assert err < bar


@pytest.mark.parametrize("nx,ny,nz,kw", [(48, 40, 11, dict(z_zoom=2)), (48, 40, 13, dict(z_zoom=2)),
                                         (40, 48, 19, dict(z_zoom=3)), (24, 25, 8, dict(zoomfact=4.0)),
                                         (24, 25, 22, dict(zoomfact=4.0)), (48, 40, 6, dict(z_zoom=2))])
def test_padded_and_odd(nx, ny, nz, kw):
    print("case %dx%dx%d %s" % (nx, ny, nz, kw), flush=True)
    p, otf, raw, _ = synthetic(nx, ny, nz, seed=nz, gpu=True, **kw)
    with loaded(p, otf, raw) as r:
        r.process_volume()
        vol = r.result()
        fits = [r.fit(d) for d in range(p.ndirs)]
        got = [[r.band(d, b) for b in range(p.nphases)] for d in range(p.ndirs)]
    bar = 5 * 2.0 ** -24 * np.sqrt(sum(np.log2(n) for n in vol.shape))
    err = rel_l2(vol, assembled(p, got, fits))
    print("  rel-L2 %.2e, bar %.2e" % (err, bar), flush=True)
    assert err < bar


def test_left_out_columns_change_nothing():
    p, otf, raw, _ = synthetic(64, 48, 11, seed=5, gpu=True)
    with loaded(p, otf, raw) as r:
        r.process_volume()
        want = r.result()
    with loaded(p, otf, raw) as r:
        whole = [[r.band(d, b) for b in range(p.nphases)] for d in range(p.ndirs)]  # completes every direction
        r.process_volume()
        assert np.array_equal(r.result(), want)
    with loaded(p, otf, raw) as r:
        r.set_band(1, 2, whole[1][2])  # completes direction 1's other bands
        for b in range(p.nphases):
            assert np.array_equal(r.band(1, b), whole[1][b])
        r.process_volume()
        assert np.array_equal(r.result(), want)
    q = p.copy()
    q.na = p.na * 0.99  # a smaller support while the stack is loaded, and back
    with loaded(q, otf, raw) as r:
        assert engine.lib().simr_update_params(r.h, p) == 0, engine.lib().simr_last_error()
        for d in range(p.ndirs):
            for b in range(p.nphases):
                assert np.array_equal(r.band(d, b), whole[d][b])
        r.process_volume()
        assert np.array_equal(r.result(), want)
