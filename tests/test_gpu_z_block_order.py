"""The register z stages' block order: planes of 1 to 9 blocks, plane counts that are and are not whole turns over
the XCDs, one, three and six fields, against the oracle."""
import math

import numpy as np
import pytest

from cdns import config
from helpers import band_spectrum, maxrel, random_vector
import pyoracle

pytestmark = pytest.mark.gpu

# last retained kx, y intervals of the product grid, z points: 1, 1, 2, 3, 5 and 9 blocks of 16 lines a plane
CASES = [(0, 12, 32), (15, 31, 48), (16, 32, 64), (40, 33, 36), (70, 12, 96), (130, 17, 72), (33, 95, 32), (24, 21, 144),
         (20, 12, 196), (18, 14, 288)]


@pytest.mark.parametrize("nxs,ny2,nz2", CASES)
def test_z_stages_of_each_block_order(gpu, nxs, ny2, nz2):
    """The bounds of the run-time factor tests."""
    nzs = nz2 // 3
    cfg = config.make(max(2 * nxs, 2), 11, 2 * nzs, nxs, 9, nzs, max(3 * nxs // 2 * 2, 12), ny2, nz2, 4 * math.pi,
                      2 * math.pi, 180.0, 1e-3)
    cfg["NX2"] = next(n for n in (12, 48, 64, 96, 128, 196, 256, 400) if n >= cfg["NX2"])
    ref = pyoracle.Oracle(cfg)
    spec = band_spectrum(cfg, 4)
    want, back = ref.fine_phys(), ref.scalar()
    ref.xyzfft2("B", want, spec.copy())
    ref.xyzfft2("F", want.copy(), back)
    a, b = random_vector(ref.vector(), 3), random_vector(ref.vector(), 4)
    product = ref.cross_product(a, b)
    for precision, tol in ((gpu.FP64, 1e-12), (gpu.MIXED, 200 * 2.0 ** -24)):
        dev = gpu.Channel(cfg, precision=precision)
        p, s = dev.fine_phys(), dev.scalar()
        dev.xyzfft2("B", p, spec.copy())
        dev.xyzfft2("F", want.copy(), s)
        got = dev.cross_product(a, b)
        dev.close()
        errs = [maxrel(p, want), maxrel(s, back)] + [maxrel(got[..., c], product[..., c]) for c in range(3)]
        print(f"kx <= {nxs}, {ny2 + 1} x {nz2}, precision {precision}: " + " ".join(f"{e:.1e}" for e in errs), flush=True)
        assert np.isfinite(got).all() and max(errs) < tol
