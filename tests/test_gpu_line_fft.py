"""The x and z stages with FFT factors chosen at run time, against the oracle: every factor of the
list in both passes, odd lengths, colliding kz, lane groups that do not divide a wavefront."""
import math

import numpy as np
import pytest

from cdns import config
from helpers import maxrel, random_vector
import pyoracle

pytestmark = pytest.mark.gpu

# (NX2, NZ2, full): full keeps NXS = NX2/2 and NZS = NZ2/2 (Nyquist columns, shared slot)
LENGTHS = [(150, 126, 0), (135, 105, 0), (30, 42, 0), (40, 45, 0), (63, 56, 0), (100, 98, 0), (75, 84, 0), (12, 10, 0),
           (224, 240, 0), (162, 189, 0), (200, 216, 0), (250, 243, 0), (300, 270, 0), (324, 375, 0), (400, 360, 0),
           (14, 20, 1), (20, 14, 1), (180, 50, 1), (42, 108, 1)]


def mesh(nx2, nz2, full):
    nxs, nzs = (nx2 // 2, nz2 // 2) if full else (nx2 // 3, nz2 // 3)
    return config.make(2 * nxs, 11, 2 * nzs, nxs, 9, nzs, nx2, 13 if nx2 % 2 else 12, nz2, 4 * math.pi, 2 * math.pi,
                       180.0, 1e-3)


@pytest.mark.parametrize("nx2,nz2,full", LENGTHS)
def test_cross_product_of_runtime_factors(gpu, nx2, nz2, full):
    """FP64 at the round-off of the transforms (as the tuned lengths are held); binary32 with 9 transforms of
    a few dozen rounded operations each, products of two fields: 200 units of 2^-24 of the largest value."""
    cfg = mesh(nx2, nz2, full)
    ref = pyoracle.Oracle(cfg)
    a, b = random_vector(ref.vector(), 3), random_vector(ref.vector(), 4)
    want = ref.cross_product(a, b)
    for precision, tol in ((gpu.FP64, 1e-12), (gpu.MIXED, 200 * 2.0 ** -24)):
        dev = gpu.Channel(cfg, precision=precision)
        got = dev.cross_product(a, b)
        dev.close()
        err = max(maxrel(got[..., c], want[..., c]) for c in range(3))
        print(f"{nx2} x {nz2} precision {precision}: {err:.2e}")
        assert np.isfinite(got).all() and err < tol
