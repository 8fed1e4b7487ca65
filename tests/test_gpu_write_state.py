"""tf_write_state in the caller's numbering: the values written on Dirichlet
edges reach the first solve of a run that continues from the written state
(a run from step 1 sets them itself, D:1434-1453), whatever layout the context
keeps its edges in."""
import numpy as np
import pytest

from tetfit_amd import Model, configs
from tetfit_amd.device import Simulation

from test_gpu_parity import rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method", ["gfdtd", "fem"])
def test_written_wall_value_reaches_the_solve(workdir, monkeypatch, method):
    """U is 1000 on one wall edge and 0 elsewhere. The edge is one that the
    mass matrix couples to a free one and whose number is no wall edge's label
    in the locality layout, so a check of the written values by label sees none
    of it; in the problem's own numbering labels and numbers are the same.
    Solves stop at 1e-12 of their warm-start residual and cond(A) of the mesh
    is below 1e3, so the two layouts agree within 1e-9."""
    b = Model(configs.kuhn_cavity(str(workdir), n=5, method=method, n_steps=20, n_probes=1, block=2,
                                  name=f"ws_{method}")).build(1)
    rank, free, M = b.edge_rank(), b.dga_ops()["free_edges"], b.dga_ops()["E"]
    wall = np.setdiff1d(np.arange(b.n_edges), free)
    row = np.repeat(np.arange(b.n_edges), np.diff(M["rowptr"]))
    coupled = M["col"][np.isin(row, free) & (M["val"] != 0)]
    e = np.setdiff1d(np.intersect1d(wall, coupled), rank[wall])[0]
    z = np.zeros(b.n_faces)

    def run(order, value):
        monkeypatch.setenv("TETFIT_TET_ORDER", order)
        U = np.zeros(b.n_edges)
        U[e] = value
        sim = Simulation(b, "fp64", output=False)
        sim.set_state(U, z, z)
        st = sim.run(first=5, n=1, cg_tol=1e-12)
        got = sim.state()
        sim.close()
        assert st["cg_not_converged"] == 0
        return got[0], got[2]

    ref = run("numbering", 1000.0)
    assert rel_l2(run("numbering", 0.0)[0][free], ref[0][free]) > 1e-2
    for a, r in zip(run("rank", 1000.0), ref):
        assert rel_l2(a, r) <= 1e-9
