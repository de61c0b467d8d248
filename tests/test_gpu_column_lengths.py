"""The step where the solve's entries per lane change: columns of 64, 128 and 192 entries and the
neighbours of each, and the longest, against the oracle."""
import math

import numpy as np
import pytest

from cdns import config, fields
import pyoracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nj", [5, 32, 63, 64, 65, 128, 129, 191, 192, 193, 256])
def test_step_at_column_length(gpu, nj):
    """Setup and three steps; the five-step bound of the long-column parity test."""
    ny = nj - 1
    cfg = config.make(16, ny + 2, 16, 6, ny, 6, 20, 3 * ny // 2 + 2, 18, 4 * math.pi, 2 * math.pi, 180.0, 1e-4)
    u0 = fields.seeded_velocity(cfg, seed=7)
    dev, ref = gpu.Channel(cfg), pyoracle.Oracle(cfg)
    dev.set_state("velocity", u0)
    ref.set_state("velocity", u0)
    dev.run(3, it_begin=1)
    ref.run(3)
    for name in ("velocity", "pressure"):
        got, want = dev.get_state(name), ref.get_state(name)
        err = fields.rel_l2(got, want)
        print(f"{nj} entries, {name}: {err:.2e}")
        assert np.isfinite(got).all() and err < 1e-10
    dev.close()
