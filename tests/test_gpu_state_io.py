"""States crossing the C ABI: what set_state is given, get_state returns bit
for bit, at sizes on both sides of the pinned-staging limit (4 MiB), odd
element counts and every order."""
import numpy as np
import pytest

from gocfd_amd import Euler, InputParameters2D, Mesh, meshgen

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,N,prec", [(3, 3, 0, "fp64"), (3, 5, 1, "fp32"), (7, 9, 2, "fp64"), (5, 13, 3, "fp32"),
                                          (66, 66, 4, "fp64"), (67, 67, 4, "fp64")])
def test_state_round_trip(nx, ny, N, prec):
    m = Mesh.from_arrays(*meshgen.jittered_quads(nx, ny))
    e = Euler(InputParameters2D(CFL=1.0, FluxType="Roe", InitType="IVortex", PolynomialOrder=N, FinalTime=1e9), m,
              precision=prec)
    rng = np.random.default_rng(nx)
    q = e.Q * (1.0 + 1e-3 * rng.standard_normal((4, e.NpInt, e.K)))
    e.Q = q
    assert np.array_equal(e.Q, q)
    e.Q = q[:, :, ::-1].copy()
    assert np.array_equal(e.Q, q[:, :, ::-1])
