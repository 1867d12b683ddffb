"""Solvers and ensembles with a ratio of specific heats other than 1.4: the
kernels whose boundary states take powers. The bars are those of the same tests
at 1.4: the RHS within 1e-14 of the summed divergence terms (FP32 5e-6, or 1e-12
where it computes in FP64), densities after steps within 1e-10 relative L2 of the
oracle (FP32 1e-5), transposes within 1e-10."""
import numpy as np
import pytest

import oracle
from gocfd_amd import Ensemble, Euler, InputParameters2D, Mesh, meshgen

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def meshes(tmp_path_factory):
    d = tmp_path_factory.mktemp("gamma")
    VX, VY, E, tags = meshgen.jittered_quads(9, 7, periodic_x=False)
    box = str(d / "box.su2")
    meshgen.write_su2(box, VX, VY, E, tags)
    return dict(box=box, foil=meshgen.airfoil_mesh(str(d / "foil.su2"), n_around=60, n_radial=12, radius=8.0, seed=2),
                wedge=meshgen.wedge_mesh(str(d / "wedge.su2"), 700))


def _pair(mesh, N, flux, gamma, prec, M=0.5, alpha=2.0, **kw):
    gpu = Euler(InputParameters2D(CFL=0.5, FluxType=flux, InitType="Freestream", Minf=M, Alpha=alpha, Gamma=gamma,
                                  PolynomialOrder=N, FinalTime=1e9, **kw), mesh, precision=prec)
    ora = oracle.OracleSolver(mesh, N, flux=flux.lower(), init="freestream", CFL=0.5, FinalTime=1e9, Minf=M, Alpha=alpha,
                              Gamma=gamma, **{k.replace("Limiter", "limiter"): v for k, v in kw.items()})
    return gpu, ora


def _start(gpu, ora, seed, amp=1e-2):
    q = ora.state() * (1.0 + amp * np.random.default_rng(seed).standard_normal(ora.state().shape))
    gpu.Q = q
    ora.set_state(q)
    return q


def _density_error(gpu, ora, steps):
    gpu.step(steps)
    for _ in range(steps):
        ora.step()
    return np.linalg.norm(gpu.Q[0] - ora.state()[0]) / np.linalg.norm(ora.state()[0])


@pytest.mark.parametrize("N,flux", [(0, "Lax"), (1, "Average"), (1, "Roe"), (2, "Lax"), (2, "Roe"), (3, "Roe-ER"), (3, "Roe"),
                                    (4, "Average"), (4, "Lax"), (4, "Roe"), (4, "Roe-ER")])
@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_rhs_and_steps(meshes, N, flux, prec):
    gpu, ora = _pair(meshes["box"], N, flux, 1.3, prec)
    q = _start(gpu, ora, 20 + N)
    r, ref = gpu.rhs(q, 0.0), ora.rhs(q, 0.0)
    bar = 1e-14 if prec == "fp64" else 1e-12 if N <= 1 else 5e-6
    assert np.abs(r - ref).max() / ora.rhs_term_scale().max() < bar
    assert _density_error(gpu, ora, 10) < (1e-10 if prec == "fp64" else 1e-5)


@pytest.mark.parametrize("gamma", [1.4 + 1e-9, 1.4 - 1e-9, 5.0 / 3.0, 1.1])
def test_rhs_over_gamma(meshes, gamma):
    gpu, ora = _pair(meshes["foil"], 2, "Roe", gamma, "fp64")
    q = _start(gpu, ora, 3)
    r, ref = gpu.rhs(q, 0.0), ora.rhs(q, 0.0)
    assert np.abs(r - ref).max() / ora.rhs_term_scale().max() < 1e-14


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("N,lts", [(2, False), (3, False), (2, True)])
def test_shock_capturing(meshes, N, lts, prec):
    gpu, ora = _pair(meshes["wedge"], N, "Roe", 1.3, prec, M=2.0, alpha=0.0, Limiter="PerssonC0", Kappa=10.0,
                     LocalTimeStepping=lts)
    _start(gpu, ora, 11, amp=0.02)
    assert _density_error(gpu, ora, 20) < (1e-10 if prec == "fp64" else 1e-5)
    assert (ora.shock()[1] > 0).any()


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_local_time_stepping(meshes, prec):
    gpu, ora = _pair(meshes["foil"], 2, "Lax", 1.3, prec, LocalTimeStepping=True)
    _start(gpu, ora, 12, amp=1e-3)
    assert _density_error(gpu, ora, 20) < (1e-10 if prec == "fp64" else 1e-5)


@pytest.mark.parametrize("par,prec", [(0, "fp64"), (1, "fp64"), (2, "fp64"), (0, "fp32"), (1, "fp32")])
def test_gammas_mixed_in_an_ensemble(par, prec):
    """Cases of both kinds in one order group: each is bit for bit its own run."""
    cases = [(InputParameters2D(CFL=0.5, FluxType="Roe", InitType="Freestream", Minf=0.5, Alpha=2.0, Gamma=g, PolynomialOrder=N,
                                FinalTime=1e9), Mesh.from_arrays(*meshgen.jittered_quads(n, n, seed=n)))
             for n, N, g in ((7, 2, 1.4), (9, 2, 1.3), (8, 4, 1.3), (6, 4, 1.4), (10, 1, 1.4))]
    ens = Ensemble(cases, precision=prec)
    ens.set_launch(par, 6, True)
    ens.step(14)
    for i, (ip, mesh) in enumerate(cases):
        one = Euler(ip, mesh, precision=prec)
        one.step(14)
        assert np.array_equal(ens.state(i), one.Q), i
        assert ens.time_info(i) == one.time_info(), i


@pytest.mark.parametrize("N,flux,lts", [(2, "Roe", False), (3, "Lax", False), (2, "Roe", True)])
def test_derivatives(meshes, N, flux, lts):
    e = Euler(InputParameters2D(CFL=0.5, FluxType=flux, InitType="Freestream", Minf=0.5, Alpha=2.0, Gamma=1.3, PolynomialOrder=N,
                                FinalTime=1e9, LocalTimeStepping=lts), meshes["foil"])
    e.step(3)
    rng = np.random.default_rng(N)
    v = rng.standard_normal(e.Q.shape) * np.abs(e.Q)
    w, s = rng.standard_normal(4), rng.standard_normal(e.Q.shape)
    qn, jv = e.jvp(4, v, w)
    d0, dfar = e.vjp(4, s)
    lhs = float(np.sum(s * jv))
    assert abs(lhs - float(np.sum(d0 * v) + dfar @ w)) <= 1e-10 * abs(lhs)
    e.step(4)
    assert np.abs(qn - e.Q).max() / np.abs(e.Q).max() < 1e-12
