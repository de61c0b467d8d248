"""Coarse syntheses of a mixed context, whose workspaces hold fewer FP64 fields than one launch of an FP64 context
takes (4 and 1, or 3 and 2, of the five): the same kernels on the same FP64 planes, so the same values bit for bit."""
import numpy as np
import pytest

from cdns import config, fields

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mesh", [config.channel_32, config.reference_example])
def test_mixed_statistics_are_those_of_an_fp64_context(gpu, mesh):
    cfg = mesh()
    u = fields.seeded_velocity(cfg, seed=11, mean="laminar", kmax=4, amplitude=0.1)
    p = np.random.default_rng(5).standard_normal(u.shape[:3]) + 0j
    seen = []
    for precision in (gpu.MIXED, gpu.FP64):
        dev = gpu.Channel(cfg, precision=precision)
        dev.set_state("velocity", u)
        dev.set_state("pressure", p)
        vel, pr, finite = dev.to_physical()
        sums, planes = dev.plane_moments(higher=True)
        seen.append((vel, pr, sums, planes, finite, dev.diagnostics()))
        dev.close()
    for mixed, fp64 in zip(*seen):
        assert np.array_equal(mixed, fp64) if isinstance(mixed, np.ndarray) else mixed == fp64
    assert seen[0][4] and seen[0][5]["finite"]
