"""Reverse sweeps short of device memory (refused by a host-side hook, no kernel
is affected): with room for some blocks of records the others are recomputed,
with none the call fails and the next one is whole. Every schedule runs the same
kernels on the same values: bit for bit."""
import numpy as np
import pytest

from gocfd_amd import Euler, InputParameters2D, meshgen
from gocfd_amd._lib import GocfdError

pytestmark = pytest.mark.gpu

STEPS = 16  # four blocks of four steps


@pytest.fixture(scope="module")
def foil(tmp_path_factory):
    path = str(tmp_path_factory.mktemp("foil") / "foil.su2")
    meshgen.airfoil_mesh(path, n_around=60, n_radial=12, radius=8.0, seed=2)
    return path


def _solver(path, lts):
    """A solver a few steps into the run (a non-uniform state)."""
    e = Euler(InputParameters2D(CFL=1.0, FluxType="Roe", InitType="Freestream", PolynomialOrder=2, Minf=0.5, Alpha=2.0,
                                FinalTime=1e9, LocalTimeStepping=lts), path)
    e.step(3)
    return e


@pytest.mark.parametrize("lts", [False, True])
@pytest.mark.parametrize("room", [8, 4, 0])  # steps: two blocks, one, none
def test_records_of_some_blocks(foil, monkeypatch, lts, room):
    e = _solver(foil, lts)
    v = np.random.default_rng(1).standard_normal(e.Q.shape)
    whole = e.vjp(STEPS, v)
    assert np.isfinite(whole[0]).all()
    monkeypatch.setenv("GOCFD_TEST_RECORD_STEPS", str(room))
    for got in (e.vjp(STEPS, v), _solver(foil, lts).vjp(STEPS, v)):
        assert all(np.array_equal(a, b) for a, b in zip(whole, got))


def test_a_call_after_a_failed_one(foil, monkeypatch):
    v = np.random.default_rng(2).standard_normal(_solver(foil, False).Q.shape)
    whole = _solver(foil, False).vjp(STEPS, v)
    e = _solver(foil, False)
    monkeypatch.setenv("GOCFD_TEST_RECORD_STEPS", "-1")
    with pytest.raises(GocfdError, match="no device memory"):
        e.vjp(STEPS, v)
    monkeypatch.delenv("GOCFD_TEST_RECORD_STEPS")
    assert all(np.array_equal(a, b) for a, b in zip(whole, e.vjp(STEPS, v)))
