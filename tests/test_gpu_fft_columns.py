"""Column transforms of the lengths that the general two-pass register core
takes (no N1 | N2 split, 96 to 640 points) and of their neighbours on the other
kernels, as the y and the z axis, against numpy in double: tiles of 16 columns
with a remainder, lanes without a row, more columns than lanes in pass 1."""
import numpy as np
import pytest

from cudasirecon_amd import engine

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [96, 100, 120, 160, 200, 240, 288, 300, 360, 384, 400, 480, 500, 600, 640, 720])
@pytest.mark.parametrize("inverse", [False, True])
def test_columns(n, inverse):
    print("n", n, inverse, flush=True)
    rng = np.random.default_rng(n)
    for shape in [(2, n, 40), (n, 2, 24), (1, n, 16)]:
        if shape[0] == n and n > 512:
            continue
        a = (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)
        got = engine.fft3d(a, inverse)
        want = np.fft.ifftn(a.astype(np.complex128)) * a.size if inverse else np.fft.fftn(a.astype(np.complex128))
        err = np.linalg.norm(got - want) / np.linalg.norm(want)
        # a two-pass transform of n points rounds about log2(n) + 4 times at 6e-8 each, the other axes less
        assert err < 6e-8 * np.sqrt(3 * (np.log2(n) + 4)), (shape, err)
