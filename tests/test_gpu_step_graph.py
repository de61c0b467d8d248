"""Runs of a small grid, whose steady steps are replayed as a graph, against the same steps launched one by one:
every state bit for bit, with eager work, synchronisations and changed inputs between the runs."""
import numpy as np
import pytest

from cdns import config, fields

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["FP64", "MIXED"])
def test_replayed_steps_equal_launched_steps(gpu, precision):
    cfg = dict(config.channel_32(), DT=2e-4)
    u0 = fields.seeded_velocity(cfg, seed=3)
    force = 0.01 * fields.seeded_velocity(cfg, seed=7, mean="laminar", kmax=4, amplitude=1.0)
    replayed, launched = (gpu.Channel(cfg, precision=getattr(gpu, precision)) for _ in range(2))
    launched.profile(True)  # timed launches are never replayed
    both = (replayed, launched)

    def same(what):
        for name in ("velocity", "pressure"):
            a, b = (ch.get_state(name) for ch in both)
            assert np.isfinite(a).all() and np.array_equal(a, b), (what, name)
        assert replayed.time() == launched.time()

    for ch in both:
        ch.set_state("velocity", u0)
        ch.run(2, it_begin=1)
    # 45 steps before the first capture, then both plane orders (odd runs), lengths around the graph's
    for n in (45, 20, 7, 21, 6, 8, 13, 40):
        for ch in both:
            ch.run(n)
        same(n)
        assert replayed.diagnostics() == launched.diagnostics()
    for ch in both:
        ch.set_body_force(force)
    for n in (25, 50, 26):
        for ch in both:
            ch.run(n)
        same("body force")
    for ch in both:
        ch.set_state("velocity", u0)
        ch.run(30, it_begin=1)
    same("new start")
    for ch in both:
        ch.set_body_force(None)
        ch.setup(100.0)  # tables of another operator: the next step sets up its own
        ch.run(30)
    same("other tables")
    if precision == "FP64":
        for ch in both:
            ch.adjoint_run(u0, None, 5, 2)
            ch.set_state("velocity", u0)
            ch.run(40, it_begin=1)
        same("after an adjoint run")
