"""State reads and writes go through a device staging buffer (permutation and
conversion on the device): written fields come back bit for bit (rounded to
fp32 where the context holds fp32) in every layout, and a batch instance's
read equals the single simulation's fields."""
import numpy as np
import pytest

from tetfit_amd import Model, configs
from tetfit_amd.device import BatchSimulation, Simulation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("case", ["grid", "indexed", "relabeled", "numbering"])
def test_state_round_trip(workdir, monkeypatch, case, prec):
    """A grid whose fields take the staging buffer's 2^20 values and a part of
    them once more, and a tet mesh, in both of their layouts."""
    if case in ("grid", "indexed"):
        monkeypatch.setenv("TETFIT_FIT_INDEXED", "1" if case == "indexed" else "0")
        b = Model(configs.fit_cavity(str(workdir), n=72, step=0.1, n_steps=4, n_probes=1, name="io_fit")).build(1)
    else:
        if case == "numbering":
            monkeypatch.setenv("TETFIT_TET_ORDER", "numbering")
        b = Model(configs.kuhn_cavity(str(workdir), n=5, method="dga", n_steps=4, n_probes=1, block=2,
                                      name="io_dga")).build(1)
    assert case not in ("grid", "indexed") or (1 << 20) < min(b.n_edges, b.n_faces) < (2 << 20)
    rng = np.random.default_rng(3)
    put = [rng.standard_normal(k) for k in (b.n_edges, b.n_faces, b.n_faces)]
    sim = Simulation(b, prec, output=False)
    sim.set_state(*put)
    got = sim.state()
    sim.set_state(U=2 * put[0])  # the other fields stay
    again = sim.state()
    sim.close()
    as_held = (lambda v: v) if prec == "fp64" else (lambda v: v.astype(np.float32).astype(np.float64))
    for g, p in zip(got, put):
        np.testing.assert_array_equal(g, as_held(p))
    for g, p in zip(again, (2 * put[0], put[1], put[2])):
        np.testing.assert_array_equal(g, as_held(p))


@pytest.mark.parametrize("method", ["dga", "gfdtd"])
def test_batch_instance_state(workdir, method):
    builds = [Model(configs.kuhn_cavity(str(workdir), n=n, method=method, n_steps=40, n_probes=1, block=2, seed=n,
                                        name=f"io_{method}{n}")).build(1) for n in (3, 5, 4)]
    sim = BatchSimulation(builds, "fp64")
    sim.run(20)
    for k, b in enumerate(builds):
        one = Simulation(b, "fp64", output=False)
        one.run(n=20)
        for got, ref in zip(sim.state(k), one.state()):
            assert np.linalg.norm(got - ref) <= 1e-10 * np.linalg.norm(ref) and np.linalg.norm(ref) > 0
        one.close()
    sim.close()
