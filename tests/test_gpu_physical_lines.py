"""The x stages of single physical fields against the oracle, both ways and in both precisions: FFT factors chosen
at run time up to 27, odd lengths, lengths with kernels of their own, blocks whose last one holds 1 or 15 of its
16 points, and grids of more blocks than are resident at once."""
import math

import numpy as np
import pytest

from cdns import config
from helpers import band_spectrum, maxrel
import pyoracle

pytestmark = pytest.mark.gpu

# 13 planes of 21 or 27 lines: 17 x 16 + 1 and 21 x 16 + 15 points
LENGTHS = [(30, 21, 0), (30, 27, 0), (135, 21, 0), (63, 27, 0), (12, 21, 0), (150, 126, 0), (100, 27, 0), (75, 84, 0),
           (250, 21, 0), (324, 27, 0), (375, 21, 0), (400, 27, 0), (14, 20, 1), (180, 50, 1), (42, 27, 0),
           (32, 21, 0), (48, 27, 0), (64, 20, 1), (96, 21, 0), (128, 27, 0), (160, 21, 0), (196, 27, 0), (256, 21, 0)]


def mesh(nx2, nz2, full, ny2=12):
    nxs, nzs = (nx2 // 2, nz2 // 2) if full else (nx2 // 3, nz2 // 3)
    return config.make(2 * nxs, 11, 2 * nzs, nxs, 9, nzs, nx2, ny2, nz2, 4 * math.pi, 2 * math.pi, 180.0, 1e-3)


def check(gpu, cfg):
    """FP64 at the bound of the transform parity tests; binary32 with three stages of a few dozen rounded
    operations a value each: 64 units of 2^-24 of the largest value."""
    ref = pyoracle.Oracle(cfg)
    spec = band_spectrum(cfg, 5)
    phys, back = ref.fine_phys(), ref.scalar()
    ref.xyzfft2("B", phys, spec.copy())
    ref.xyzfft2("F", phys.copy(), back)
    for precision, tol in ((gpu.FP64, 1e-13), (gpu.MIXED, 64 * 2.0 ** -24)):
        dev = gpu.Channel(cfg, precision=precision)
        p, s = dev.fine_phys(), dev.scalar()
        p[...] = s[...] = np.nan
        dev.xyzfft2("B", p, spec.copy())
        dev.xyzfft2("F", phys.copy(), s)
        dev.close()
        eb, ef = maxrel(p, phys), maxrel(s, back)
        print(f"{cfg['NX2']} x {cfg['NZ2']} precision {precision}: backward {eb:.2e} forward {ef:.2e}", flush=True)
        assert eb < tol and ef < tol


@pytest.mark.parametrize("nx2,nz2,full", LENGTHS)
def test_physical_transform_of_each_length(gpu, nx2, nz2, full):
    check(gpu, mesh(nx2, nz2, full))


@pytest.mark.parametrize("nx2", [30, 32, 64, 96])
def test_physical_transform_of_more_blocks_than_are_resident(gpu, nx2):
    """151 x 256 points: 2416 blocks."""
    check(gpu, dict(mesh(nx2, 256, 0, ny2=150)))


# 1274 (an odd number of points), 1208, 1024 and 1280 blocks of 16 points
@pytest.mark.parametrize("nx2,nz2,ny2", [(48, 135, 150), (72, 135, 150), (120, 128, 150), (128, 128, 150),
                                         (256, 128, 127), (192, 128, 159)])
def test_physical_transform_where_lengths_change_kernels(gpu, nx2, nz2, ny2):
    check(gpu, mesh(nx2, nz2, 0, ny2=ny2))


@pytest.mark.parametrize("nx2,ny2", [(500, 12), (625, 12), (625, 300)])
def test_physical_transform_of_the_longest_lines(gpu, nx2, ny2):
    """20 x 25 and 25 x 25, about the longest lengths that a context takes: a block's LDS beyond 64 KB in FP64."""
    check(gpu, mesh(nx2, 21, 0, ny2=ny2))
