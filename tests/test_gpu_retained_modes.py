"""The x product with the last retained kx at, before and after the edges of a lane's slot ranges, up to a full
Nyquist column, against the oracle."""
import math

import numpy as np
import pytest

from cdns import config
from helpers import maxrel, random_vector
import pyoracle

pytestmark = pytest.mark.gpu

# product lengths whose slots come in ranges of 12, 16, 24, 28 and 32; the last retained kx
CASES = [(48, k) for k in (1, 11, 12, 16, 23, 24)] + [(96, k) for k in (1, 15, 16, 17, 31, 32, 33, 47, 48)] + \
        [(144, k) for k in (23, 24, 47, 48, 71, 72)] + [(196, k) for k in (27, 28, 55, 56, 65, 83, 84, 97, 98)] + \
        [(384, k) for k in (31, 32, 63, 64, 127, 128, 159, 160, 191, 192)]


@pytest.mark.parametrize("nx2,nxs", CASES)
def test_cross_product_of_retained_modes(gpu, nx2, nxs):
    """The bounds of the runtime-factor lengths: FP64 at the transforms' round-off, binary32 200 units of 2^-24
    of the largest value."""
    cfg = config.make(2 * nxs, 11, 8, nxs, 9, 4, nx2, 12, 12, 4 * math.pi, 2 * math.pi, 180.0, 1e-3)
    ref = pyoracle.Oracle(cfg)
    a, b = random_vector(ref.vector(), 3), random_vector(ref.vector(), 4)
    want = ref.cross_product(a, b)
    for precision, tol in ((gpu.FP64, 1e-12), (gpu.MIXED, 200 * 2.0 ** -24)):
        dev = gpu.Channel(cfg, precision=precision)
        got = dev.cross_product(a, b)
        dev.close()
        err = max(maxrel(got[..., c], want[..., c]) for c in range(3))
        print(f"{nx2}, kx <= {nxs}, precision {precision}: {err:.2e}")
        assert np.isfinite(got).all() and err < tol
