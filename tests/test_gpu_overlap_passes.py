"""The fit's two-pass overlaps (columns formed and transformed, rows transformed
and summed over z) against the three-pass form that debug_overlaps takes: image
sizes whose plans differ (lanes of a row that swap by 4, 8, 16 or 32; an odd
number of outputs per lane; columns not a multiple of their tile; few planes, or
more than a workgroup's row pairs), the plane kz = 0 left out, a full OTF table
and a lens that excludes most columns.

The modamp is sum P e^{i phi} / sum SX; as in the modamp tests the engine's is
that sum of its own overlaps, whose two 32-bit transforms differ from the
three-pass form's by about 2e-7 of the overlaps."""
import numpy as np
import pytest

from cases import full_otf_from_ra, synthetic
from cudasirecon_amd import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz,kw", [
    (32, 48, 8, {}), (80, 64, 9, {}), (96, 96, 6, {}), (128, 40, 24, {}), (192, 128, 8, dict(bNoKz0=1)),
    (200, 100, 12, {}), (240, 360, 6, {}), (400, 48, 16, {}), (480, 400, 3, {}), (500, 64, 8, dict(bNoKz0=1)),
    (1024, 80, 8, {}), (64, 640, 8, {}), (256, 96, 9, dict(full=1)), (100, 300, 8, dict(full=1, bNoKz0=1))])
def test_fit_overlaps_in_two_passes(nx, ny, nz, kw):
    print("case %dx%dx%d %s" % (nx, ny, nz, kw), flush=True)
    kw = dict(kw)
    full = kw.pop("full", 0)
    p, otf, raw, _ = synthetic(nx, ny, nz, seed=nx + ny, gpu=True, zoomfact=2.0, **kw)
    if full:
        p, otf = full_otf_from_ra(p, otf)
    with engine.Reconstructor(p, otf) as r:
        r.set_raw(raw)
        r.load_and_rescale(0)
        r.set_time(0)
        r.find_modulation()
        for d in range(p.ndirs):
            f = r.fit(d)
            o = r.debug_overlaps(d, 0, 1, f.k0x, f.k0y)
            x = 2 * np.pi * p.dxy * (np.arange(nx) - 0.5 * nx) * f.k0x
            y = 2 * np.pi * p.dxy * (np.arange(ny) - 0.5 * ny) * f.k0y
            want = (o["P"] * np.exp(1j * (x[None, :] + y[:, None]))).sum() / o["sx"].sum()
            got = complex(f.amp_re[1], f.amp_im[1])
            cc = abs(want) * np.sqrt(o["sx"].sum() / o["sy"].sum())
            print("  direction %d: modamp off by %.1e" % (d, abs(got - want) / abs(want)), flush=True)
            assert abs(got - want) < 2e-6 * abs(want)
            assert abs(f.corr[1] - cc) < 2e-6 * cc


@pytest.mark.parametrize("nx,ny,nz,phases,kw", [(64, 64, 24, 5, {}), (200, 100, 12, 5, {}), (512, 96, 8, 5, {}),
                                                (128, 80, 1, 3, {}), (480, 48, 9, 5, dict(bNoKz0=1))])
def test_nothing_unwritten_is_read(nx, ny, nz, phases, kw):
    """The column pass leaves columns without an element unwritten and the row pass leaves them
    unread: staging memory full of NaN (a stack of NaN, whose overlap volumes go there) changes
    nothing in the next reconstruction."""
    print("case %dx%dx%d, %d phases, %s, staging full of NaN" % (nx, ny, nz, phases, kw), flush=True)
    p, otf, raw, _ = synthetic(nx, ny, nz, nphases=phases, seed=nx + ny, gpu=True, zoomfact=2.0, **kw)

    def once(r):
        r.set_raw(raw)
        r.load_and_rescale(0)
        r.set_time(0)
        r.process_volume()
        return r.result(), [r.fit(d) for d in range(p.ndirs)]

    with engine.Reconstructor(p, otf) as r, engine.Reconstructor(p, otf) as fresh:
        r.set_raw(np.full(raw.shape, np.nan, np.float32))
        r.load_and_rescale(0)
        for d in range(p.ndirs):
            ov = r.overlap_volumes(d, 0, 1, 1.0, 0.5)
        assert np.isnan(ov[0]).all() and np.isnan(ov[1]).all()
        got, fits = once(r)
        want, wfits = once(fresh)
        assert np.isfinite(want).all() and np.array_equal(got, want)
        for f, w in zip(fits, wfits):
            assert (f.k0x, f.k0y, list(f.amp_re), list(f.corr)) == (w.k0x, w.k0y, list(w.amp_re), list(w.corr))
