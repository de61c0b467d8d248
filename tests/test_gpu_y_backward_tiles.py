"""The y backward of whole fields where its row tiles per wavefront and its block size change, against the oracle:
3 to 12 row tiles, columns whose tables fill the LDS, one field and the six of a product, grids below and above
the device's compute units."""
import math

import numpy as np
import pytest

from cdns import config
from helpers import band_spectrum, maxrel, random_vector
import pyoracle

pytestmark = pytest.mark.gpu


def mesh(nxs, nys, nzs, ny2):
    return config.make(2 * nxs, nys + 2, 2 * nzs, nxs, nys, nzs, 3 * nxs, ny2, 3 * nzs, 4 * math.pi, 2 * math.pi, 180.0,
                       1e-3)


# 33 x 65 columns: 34 groups of 64; row tiles of the product grid's half columns
CASES = [(62, 92), (78, 116), (90, 134), (126, 188), (150, 224), (171, 255), (190, 284), (200, 300), (220, 330), (254, 380)]


@pytest.mark.parametrize("precision", ["FP64", "MIXED"])
@pytest.mark.parametrize("nys,ny2", CASES)
def test_y_backward_of_one_and_six_fields(gpu, precision, nys, ny2):
    """The bounds of the run-time factor tests: FP64 at the transforms' round-off, binary32 200 units of 2^-24."""
    cfg = mesh(32, nys, 32, ny2)
    tol = 1e-12 if precision == "FP64" else 200 * 2.0 ** -24
    dev, ref = gpu.Channel(cfg, precision=getattr(gpu, precision)), pyoracle.Oracle(cfg)
    spec = band_spectrum(cfg, 9)
    p, want = dev.fine_phys(), ref.fine_phys()
    dev.xyzfft2("B", p, spec.copy())
    ref.xyzfft2("B", want, spec.copy())
    one = maxrel(p, want)
    a, b = random_vector(ref.vector(), 3), random_vector(ref.vector(), 4)
    got, product = dev.cross_product(a, b), ref.cross_product(a, b)
    dev.close()
    six = max(maxrel(got[..., c], product[..., c]) for c in range(3))
    print(f"{nys + 1} entries, {ny2 + 1} points, {precision}: one field {one:.2e}, six {six:.2e}", flush=True)
    assert one < tol and six < tol


@pytest.mark.parametrize("precision", ["FP64", "MIXED"])
@pytest.mark.parametrize("nys", [110, 170, 254])
def test_y_backward_of_many_column_groups(gpu, precision, nys):
    """65 x 129 columns (132 groups): six fields in many rounds of blocks; every column of one entry alone."""
    cfg = mesh(64, nys, 64, 3 * nys // 2 // 2 * 2)
    tol = 1e-12 if precision == "FP64" else 64 * 2.0 ** -24
    dev, ref = gpu.Channel(cfg, precision=getattr(gpu, precision)), pyoracle.Oracle(cfg)
    spec = band_spectrum(cfg, 9)
    p, want = dev.fine_phys(), ref.fine_phys()
    dev.xyzfft2("B", p, spec.copy())
    ref.xyzfft2("B", want, spec.copy())
    a = random_vector(ref.vector(), 3)
    zero = dev.cross_product(a, a)
    other = dev.cross_product(a, 2.0 * a[..., [0, 0, 0]])
    back = dev.cross_product(2.0 * a[..., [0, 0, 0]], a)
    dev.close()
    assert maxrel(p, want) < tol
    scale = np.abs(other).max()
    assert np.abs(zero).max() < tol * scale and np.abs(other + back).max() < tol * scale
