"""Tiles whose every face leads out of them: 64 copies of a mesh laid over each
other interleave along the Hilbert curve, so a tile holds one element of each
copy. At orders 1 to 4 a thread then has more cross-tile items than the two it
prefetches, and at orders 3 and 4 more items than the three whose FP64 results it
holds (both are checked on the layout). The bars are those of the parity tests:
the RHS within 1e-14 of the magnitude of the summed divergence terms (FP32 5e-6,
1e-12 where it computes in FP64), the density after a few steps within 1e-10
relative L2 of the oracle (FP32 1e-5)."""
import numpy as np
import pytest

import oracle
from gocfd_amd import Euler, InputParameters2D, meshgen

pytestmark = pytest.mark.gpu

COPIES, THREADS = 64, 256


@pytest.mark.parametrize("N", [1, 2, 3, 4])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_tiles_with_only_cross_tile_faces(tmp_path, N, prec):
    VX, VY, E, tags = meshgen.jittered_quads(6, 6, periodic_x=False)
    n = len(VX)
    path = str(tmp_path / "copies.su2")
    meshgen.write_su2(path, np.tile(VX, COPIES), np.tile(VY, COPIES), np.concatenate([E + c * n for c in range(COPIES)]),
                      {k: [(a + c * n, b + c * n) for c in range(COPIES) for a, b in v] for k, v in tags.items()})
    gpu = Euler(InputParameters2D(CFL=0.5, FluxType="Roe", InitType="Freestream", Minf=0.5, Alpha=2.0, PolynomialOrder=N,
                                  FinalTime=1e9), path, precision=prec)
    items = gpu.tiling()[2] * (N + 2)  # cross-tile items of the widest tile
    assert items > 2 * THREADS
    assert N < 3 or items > 3 * THREADS
    ora = oracle.OracleSolver(path, N, flux="roe", init="freestream", CFL=0.5, FinalTime=1e9, Minf=0.5, Alpha=2.0)
    q = ora.state() * (1.0 + 1e-2 * np.random.default_rng(N).standard_normal(ora.state().shape))
    r, ref = gpu.rhs(q, 0.0), ora.rhs(q, 0.0)
    bar = 1e-14 if prec == "fp64" else 1e-12 if N <= 1 else 5e-6
    assert np.abs(r - ref).max() / ora.rhs_term_scale().max() < bar
    gpu.Q = q
    ora.set_state(q)
    gpu.step(3)
    for _ in range(3):
        ora.step()
    err = np.linalg.norm(gpu.Q[0] - ora.state()[0]) / np.linalg.norm(ora.state()[0])
    assert err < (1e-10 if prec == "fp64" else 1e-5)
