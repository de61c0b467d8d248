"""set_state from every host array form it takes (contiguous ones go to the device as they are), and layout
tiles at their edges, on meshes whose kx, row and kz counts are not multiples of the tile."""
import math

import numpy as np
import pytest

from cdns import config
from helpers import random_vector

pytestmark = pytest.mark.gpu

MESHES = [(4, 4, 3), (15, 31, 4), (16, 32, 5), (33, 65, 2)]  # NXS, NYS, NZS


@pytest.mark.parametrize("nxs,nys,nzs", MESHES)
def test_state_round_trip_is_exact(gpu, nxs, nys, nzs):
    nx2, nz2 = 3 * (nxs + nxs % 2), 30
    nx2 = {12: 12, 48: 48, 102: 108}.get(nx2, nx2)
    cfg = config.make(2 * nxs, nys + 2, 2 * nzs, nxs, nys, nzs, nx2, nys + 5, nz2, 2 * math.pi, math.pi, 180.0, 1e-3)
    dev = gpu.Channel(cfg)
    v = random_vector(dev.vector(), 1)
    forms = {"contiguous": v, "fortran": np.asfortranarray(v), "strided": np.repeat(v, 2, axis=0)[::2],
             "complex64": v.astype(np.complex64), "broadcast": v[:1]}
    for name, form in forms.items():
        want = np.zeros_like(v)
        want[...] = form
        kept = form.copy()
        dev.set_state("velocity", form)
        assert np.array_equal(dev.get_state("velocity"), want), name
        assert np.array_equal(form, kept)
    for field in ("pressure", "pressure_bc", "velocity_bc"):
        want = random_vector(dev.get_state(field), 2)
        dev.set_state(field, want)
        assert np.array_equal(dev.get_state(field), want), field
    dev.close()
