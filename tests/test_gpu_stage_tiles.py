"""Tiles with more cross-tile faces than a thread prefetches: 16 copies of a
mesh laid over each other interleave along the Hilbert curve, so a tile holds
four elements of each copy and at least 96 of its faces lead out of it. The
bars are those of the parity tests: the RHS within 1e-14 of the magnitude of
the summed divergence terms, the FP32 density after a few steps within 1e-5."""
import numpy as np
import pytest

import oracle
from gocfd_amd import Euler, InputParameters2D, meshgen

pytestmark = pytest.mark.gpu

COPIES = 16


@pytest.mark.parametrize("N,prec", [(0, "fp64"), (2, "fp64"), (3, "fp64"), (4, "fp64"),
                                    (2, "fp32"), (3, "fp32"), (4, "fp32")])
def test_tiles_of_many_cross_tile_faces(tmp_path, N, prec):
    VX, VY, E, tags = meshgen.jittered_quads(8, 8, periodic_x=False)
    n = len(VX)
    path = str(tmp_path / "copies.su2")
    meshgen.write_su2(path, np.tile(VX, COPIES), np.tile(VY, COPIES), np.concatenate([E + c * n for c in range(COPIES)]),
                      {k: [(a + c * n, b + c * n) for c in range(COPIES) for a, b in v] for k, v in tags.items()})
    ip = InputParameters2D(CFL=0.5, FluxType="Roe", InitType="Freestream", Minf=0.5, Alpha=2.0, PolynomialOrder=N,
                           FinalTime=1e9)
    gpu = Euler(ip, path, precision=prec)
    ora = oracle.OracleSolver(path, N, flux="roe", init="freestream", CFL=0.5, FinalTime=1e9, Minf=0.5, Alpha=2.0)
    q = ora.state() * (1.0 + 1e-2 * np.random.default_rng(N).standard_normal(ora.state().shape))
    if prec == "fp64":
        r = gpu.rhs(q, 0.0)
        ref = ora.rhs(q, 0.0)
        assert np.abs(r - ref).max() / ora.rhs_term_scale().max() < 1e-14
        return
    gpu.Q = q
    ora.set_state(q)
    gpu.step(3)
    for _ in range(3):
        ora.step()
    assert np.linalg.norm(gpu.Q[0] - ora.state()[0]) / np.linalg.norm(ora.state()[0]) < 1e-5
