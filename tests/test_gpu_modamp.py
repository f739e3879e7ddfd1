"""The fit's modamps against the sums they are, at image sizes where the
modamp reduction has remainders (rows not a multiple of its row blocks,
columns not a multiple of its phasor table or of a workgroup, wider than a
workgroup) and where the overlaps take either of their forms.

The overlap pair at the fitted k0 comes from debug_overlaps (P, SX, SY per
pixel) and the modamp from numpy in double: sum P e^{i phi} / sum SX, phi as
in reductionKernel (gpuFunctionsImpl.cu:1150-1220).  The engine's value is
that sum rounded to float (6e-8); where the engine forms the overlaps in two
passes and debug_overlaps in three, the 32-bit transforms differ by about
2e-7 of the overlaps, which the sum over the image averages further down."""
import numpy as np
import pytest

from cases import synthetic
from cudasirecon_amd import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nz,kw", [(48, 40, 8, {}), (64, 100, 9, {}), (100, 120, 8, {}), (256, 256, 6, {}),
                                         (300, 200, 8, {}), (512, 256, 6, {}), (640, 500, 6, {}),
                                         (96, 80, 8, dict(fit_fp64=0))])
def test_modamps_are_the_sums(nx, ny, nz, kw):
    print("case %dx%dx%d %s" % (nx, ny, nz, kw), flush=True)
    p, otf, raw, _ = synthetic(nx, ny, nz, seed=nx + ny, gpu=True, zoomfact=2.0, **kw)
    with engine.Reconstructor(p, otf) as r:
        r.set_raw(raw)
        r.load_and_rescale(0)
        r.set_time(0)
        r.find_modulation()
        for d in range(p.ndirs):
            f = r.fit(d)
            # order 1 is fitted at the final k0 (order 2 at the start of the line search)
            o = r.debug_overlaps(d, 0, 1, f.k0x, f.k0y)
            x = 2 * np.pi * p.dxy * (np.arange(nx) - 0.5 * nx) * f.k0x
            y = 2 * np.pi * p.dxy * (np.arange(ny) - 0.5 * ny) * f.k0y
            want = (o["P"] * np.exp(1j * (x[None, :] + y[:, None]))).sum() / o["sx"].sum()
            got = complex(f.amp_re[1], f.amp_im[1])
            cc = abs(want) * np.sqrt(o["sx"].sum() / o["sy"].sum())
            err = abs(got - want) / abs(want)
            print("  direction %d: modamp off by %.1e" % (d, err), flush=True)
            assert err < (2e-6 if p.fit_fp64 else 1e-4)  # fp32: float sums and a float phase over the image
            assert abs(f.corr[1] - cc) < (2e-6 if p.fit_fp64 else 1e-4) * cc
