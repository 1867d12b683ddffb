"""The far-field state of interior states without a real entropy, at an outflow
face, where the reference takes powers of them: NaN for a negative density (also
with a negative pressure, whose quotient is positive), and for a negative
pressure NaN or, where 1/(gamma-1) is a whole number, the power's sign. The RHS
has the oracle's NaN pattern and its values elsewhere, within 1e-13 of the
summed divergence terms (FP32: 1e-4, no more than the format's 6e-8 times the
terms' cancellation of three digits)."""
import numpy as np
import pytest

import oracle
from gocfd_amd import Euler, InputParameters2D, meshgen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("N,gamma", [(1, 1.4), (2, 1.4), (3, 1.4), (2, 1.5), (4, 1.5)])
def test_states_without_a_real_entropy(tmp_path, N, gamma, prec):
    VX, VY, E, tags = meshgen.jittered_quads(5, 5, periodic_x=False)
    path = str(tmp_path / "m.su2")
    meshgen.write_su2(path, VX, VY, E, tags)
    gpu = Euler(InputParameters2D(CFL=0.5, FluxType="Lax", InitType="Freestream", Minf=0.5, Alpha=2.0, Gamma=gamma,
                                  PolynomialOrder=N, FinalTime=1e9), path, precision=prec)
    ora = oracle.OracleSolver(path, N, flux="lax", init="freestream", CFL=0.5, FinalTime=1e9, Minf=0.5, Alpha=2.0, Gamma=gamma)
    q0 = ora.state()
    ora.rhs(q0, 0.0)
    scale = ora.rhs_term_scale().max()  # of the last evaluation
    right = [k for k in range(len(E)) if (VX[E[k]] == VX.max()).sum() == 2]
    assert len(right) == 5
    nans = 0
    for k in right:
        inverse = q0.copy()
        inverse[:, :, k] *= -1.0                     # density and pressure negative, velocity and sound speed as before
        vacuum = q0.copy()
        vacuum[3, :, k] -= 2.0 / (gamma - 1.0) * (1.0 / gamma)  # pressure -1/gamma
        for q in (inverse, vacuum):
            r, ref = gpu.rhs(q, 0.0), ora.rhs(q, 0.0)
            assert np.array_equal(np.isnan(r), np.isnan(ref))
            nans += int(np.isnan(r).any())
            ok = ~np.isnan(ref)
            assert np.abs(r[ok] - ref[ok]).max() / scale < (1e-13 if prec == "fp64" else 1e-4)
    assert nans >= len(right)
