"""Both products of a transposed step in one launch of the x-product kernels that the other adjoint tests do not
take (one lane per row, LDS Stockham), against the oracle on their mesh."""
import numpy as np
import pytest

from cdns import config, fields
import pyoracle

pytestmark = pytest.mark.gpu

STATE = ["velocity", "velocity_prev", "nonlinear_prev", "pressure_bc_prev"]


@pytest.mark.parametrize("knob", [("CDNS_XPRODUCT", "single"), ("CDNS_FFT", "stockham")])
def test_adjoint_step_of_each_product_kernel(gpu, monkeypatch, knob):
    """The mesh and the bound of the adjoint-step parity test."""
    monkeypatch.setenv(*knob)
    cfg = config.channel_32()
    o = pyoracle.Oracle(cfg)
    A = pyoracle.Adjoint(o)
    o.set_state("velocity", fields.seeded_velocity(cfg, seed=5))
    for it in range(1, 5):
        o.step(it)
    X = [o.get_state(n) for n in STATE]
    rng = np.random.default_rng(21)
    L = [rng.standard_normal(a.shape) + 1j * rng.standard_normal(a.shape) for a in X]
    lf0 = rng.standard_normal(X[0].shape) + 1j * rng.standard_normal(X[0].shape)
    Lr, lfr = A.adj_step(5, X, L, lf0)
    Lg, lfg = gpu.Channel(cfg).adjoint_step(5, X[0], L, lf0)
    errs = [float(np.abs(g - r).max() / max(np.abs(r).max(), np.abs(i).max()))
            for g, r, i in zip(Lg + [lfg], Lr + [lfr], L + [lf0])]
    print(f"{knob}: {errs}")
    assert max(errs) < 1e-10, errs
