"""The no-allocation RHS entry point over orders, precisions and ragged meshes."""
import numpy as np
import pytest

from gocfd_amd import Euler, InputParameters2D, meshgen
from test_zz_no_alloc import _hip, _noalloc_rhs, _perturbed

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 4, 9])  # K = 2, 32, 162: one ragged tile, half a tile, three tiles
@pytest.mark.parametrize("N,prec", [(0, "fp64"), (1, "fp64"), (2, "fp64"), (3, "fp64"), (4, "fp64"),
                                    (1, "fp32"), (2, "fp32"), (3, "fp32"), (4, "fp32")])
def test_rhs_noalloc_orders(tmp_path, n, N, prec):
    """The entry point's own launch of the state and its halo traces does
    the arithmetic of the host call's two launches: bit for bit."""
    path = str(tmp_path / "j.su2")
    VX, VY, E, tags = meshgen.jittered_quads(n, n, periodic_x=False)
    meshgen.write_su2(path, VX, VY, E, tags)
    gpu = Euler(InputParameters2D(CFL=0.5, FluxType="Roe", InitType="Freestream", Minf=0.5, Alpha=2.0,
                                  PolynomialOrder=N, FinalTime=1e9), path, precision=prec)
    q = _perturbed(gpu.Q, 10 * n + N)
    assert np.array_equal(_noalloc_rhs(_hip(), gpu, q, 0.2), gpu.rhs(q, 0.2))
