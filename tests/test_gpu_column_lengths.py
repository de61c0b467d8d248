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


@pytest.mark.parametrize("compact", [True, False])
def test_pressure_of_a_run_is_that_of_single_steps(gpu, compact):
    """A run writes only its last step's pressure; every step of it writes the rest of the state.  Both table
    forms (u and w with wall conditions of their own have no compact one)."""
    cfg = config.make(16, 34, 16, 6, 30, 6, 20, 48, 18, 4 * math.pi, 2 * math.pi, 180.0, 1e-4,
                      **({} if compact else {"a_V": (1.0, 1.0, 0.5), "b_V": (0.0, 0.0, 0.1)}))
    u0 = fields.seeded_velocity(cfg, seed=7)
    run, steps = gpu.Channel(cfg), gpu.Channel(cfg)
    for dev in (run, steps):
        dev.set_state("velocity", u0)
    run.run(4, it_begin=1)
    for it in range(1, 5):
        steps.step(it)
    for name in ("velocity", "pressure"):
        assert np.array_equal(run.get_state(name), steps.get_state(name))
