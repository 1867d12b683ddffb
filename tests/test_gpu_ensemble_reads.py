"""Reading an ensemble takes no device memory: a study that steps for hours must
not find at its first read that another program took what was left."""
import ctypes as C

import numpy as np
import pytest

from gocfd_amd import Ensemble, InputParameters2D, Mesh, _lib, meshgen

pytestmark = pytest.mark.gpu


def _free():
    _lib.load()
    hip = C.CDLL("libamdhip64.so.7")  # the runtime libgocfd_euler2d.so is linked against
    free, total = C.c_size_t(), C.c_size_t()
    assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_reads_take_no_device_memory(prec):
    # a single element pair, a case of some MB and one above the pinned-buffer limit (4 MiB), orders apart and together
    cases = [(InputParameters2D(CFL=0.5, FluxType="Roe", InitType="IVortex", PolynomialOrder=N, FinalTime=1e9),
              Mesh.from_arrays(*meshgen.jittered_quads(n, n))) for n, N in ((1, 4), (90, 2), (70, 4), (40, 4))]
    warm = Ensemble(cases, precision=prec)  # what the runtime itself allocates at the first use of a kernel or a copy
    warm.step(2)
    for i in range(len(cases)):
        warm.state(i)
    e = Ensemble(cases, precision=prec)
    e.step(2)
    before = _free()
    states = [e.state(i) for i in range(len(cases))]
    assert _free() == before
    assert all(np.isfinite(q).all() for q in states)
    # transfers leave the steps alone
    f = Ensemble(cases, precision=prec)
    f.step(4)
    e.step(2)
    for i in range(len(cases)):
        assert np.array_equal(e.state(i), f.state(i))
