"""Storage of an adjoint horizon: checkpoints for every segment but the last, whose synthesised fields stay where the
adjoint reads them."""
import numpy as np
import pytest

from cdns import config, fields

pytestmark = pytest.mark.gpu


def _dev(torch, a):
    return torch.as_tensor(np.ascontiguousarray(a).view(np.float64), device="cuda")


def test_one_segment_needs_no_checkpoint(gpu):
    """32 x 33 x 32: 17 steps of synthesised fields are 65.3 MB of the 67.1 MB of the fixed storage; a checkpoint of
    2.6 MB or more would not fit beside them, and the eighteenth step does not fit at all."""
    import torch

    cfg = dict(config.channel_32(), DT=2e-4)
    u0 = _dev(torch, fields.seeded_velocity(cfg, seed=5))
    ch = gpu.Channel(cfg)
    want, got = torch.zeros_like(u0), torch.full_like(u0, np.nan)
    torch.cuda.synchronize()
    Jw = ch.adjoint_run_device(u0, None, 17, 4, 0, want, None)
    Jg = ch.adjoint_run_device(u0, None, 17, 17, 0, got, None, noalloc=True)
    torch.cuda.synchronize()
    err = float((got - want).abs().max() / want.abs().max())
    print(f"J {Jg!r} vs {Jw!r}, gradient {err:.1e}")
    assert abs(Jg - Jw) <= 1e-13 * abs(Jw) and err <= 1e-13
    with pytest.raises(RuntimeError, match="more than"):
        ch.adjoint_run_device(u0, None, 18, 18, 0, got, None, noalloc=True)


@pytest.mark.parametrize("nsteps,k_ckpt", [(5, 5), (6, 5), (4, 1), (10, 5)])
def test_horizons_of_each_segment_count(gpu, nsteps, k_ckpt):
    """One segment, a last segment of one step, one-step segments and whole ones: the same gradient as one segment."""
    cfg = dict(config.channel_32(), DT=2e-4)
    u0 = fields.seeded_velocity(cfg, seed=5)
    f = 0.01 * fields.seeded_velocity(cfg, seed=7, mean="laminar", kmax=4, amplitude=1.0)
    whole, parts = gpu.Channel(cfg), gpu.Channel(cfg)
    Jw, gw, fw = whole.adjoint_run(u0, f, nsteps, nsteps)
    Jp, gp, fp = parts.adjoint_run(u0, f, nsteps, k_ckpt)
    assert np.isfinite(gp).all() and Jw == Jp
    assert np.array_equal(gw, gp) and np.array_equal(fw, fp)
