"""One launch per Jacobi pass (cg_one_kernel, systems whose rows fit an XCD's
L2) against the two-kernel passes of a learned context's collection solves:
the same recurrences, so the same iteration counts and fields to the rounding
of the reductions (1e-9 relative L2 in fp64: the 60 solves stop at 1e-8 of
their warm-start residuals and differ by rounding only), and every solve at
its tolerance."""
import numpy as np
import pytest

from tetfit_amd import Model, configs
from tetfit_amd.device import Simulation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layout", ["one_base", "win", "col32"])
@pytest.mark.parametrize("n,prec,tol", [(2, "fp64", 1e-9), (9, "fp64", 1e-9), (12, "fp32", 1e-5)])
def test_one_launch_passes(workdir, monkeypatch, n, prec, tol, layout):
    """2^3: one slice, partly empty; 9^3 and 12^3: rows of more than one batch
    of eight entries, a partial last slice; the three column layouts."""
    if layout != "one_base":
        monkeypatch.setenv({"win": "TETFIT_SELL_WIN", "col32": "TETFIT_SELL_COL32"}[layout], "1")
    b = Model(configs.kuhn_cavity(str(workdir), n=n, method="gfdtd", n_steps=80, n_probes=1, block=2, seed=n,
                                  name=f"one{n}")).build(1)
    out = []
    for opts in ({}, dict(precond="learned", learn_steps=1000)):
        sim = Simulation(b, prec, output=False)
        st = sim.run(n=60, **opts)
        assert st["cg_not_converged"] == 0 and st["cg_max_relres"] <= b.cg_tol
        out.append((st["cg_iters_total"], sim.state(), sim.poynting()))
        sim.close()
    (it1, f1, p1), (it2, f2, p2) = out
    assert abs(it1 - it2) <= (0 if prec == "fp64" else 2)
    for a, e in zip(f1, f2):
        assert np.linalg.norm(a - e) <= tol * np.linalg.norm(e) and np.linalg.norm(e) > 0
    np.testing.assert_allclose(p1, p2, rtol=10 * tol, atol=10 * tol * np.abs(p2).max())


def test_one_launch_maxiter_and_guess(workdir):
    """The stop at maxiter and the extrapolated start (stop test relative to
    the warm-start residual) on the same kernel."""
    b = Model(configs.kuhn_cavity(str(workdir), n=8, method="gfdtd", n_steps=60, n_probes=1, block=2,
                                  name="one_mx")).build(1)
    sim = Simulation(b, "fp64", output=False)
    st = sim.run(n=4, cg_maxiter=3)
    assert st["cg_iters_max"] == 3 and st["cg_not_converged"] >= 3
    sim.close()
    its = {}
    for guess in (0, 2):
        sim = Simulation(b, "fp64", output=False)
        st = sim.run(n=50, guess=guess)
        assert st["cg_not_converged"] == 0
        its[guess] = st["cg_iters_total"]
        sim.close()
    assert its[2] < its[0]
