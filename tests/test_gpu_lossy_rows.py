"""Lossy dga rows too long for one lane (the mirror entries in row 0 of H and
of Mp, D:9180-9481), F stepped in place without magnetic loss, and the lossy
loop in HIP graphs, against the CPU checker (fp64: 1e-10 relative L2 of the
final fields, the bar of test_gpu_parity)."""
import numpy as np
import pytest

from tetfit_amd.device import Simulation

import pyoracle
from test_gpu_parity import rel_l2
from test_lossy_dga import lossy_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("chi_frac", [0.0, 0.4])
def test_long_rows_and_graph_parity(workdir, chi_frac):
    """10^3 mesh: row 0 of H holds several hundred entries, over two passes of
    a workgroup. 1 + 130 + 65 steps: an odd start (the other ping-pong
    buffer), replays and remainders, with and without graphs bit for bit."""
    _, b = lossy_case(workdir, n=10, n_steps=196, name=f"long_{chi_frac}", chi_frac=chi_frac)
    length = np.diff(b.frac_ops()["Ku"]["rowptr"])
    assert length.max() > 512 and (length > 128).sum() == 2
    out = []
    for graphs in (True, False):
        sim = Simulation(b, "fp64", output=False)
        sim.set_graphs(graphs)
        for n in (1, 130, 65):
            sim.run(n=n)
        out.append((*sim.state(), sim.poynting()))
        sim.close()
    for a, e in zip(*out):
        np.testing.assert_array_equal(a, e)
    r = pyoracle.run(b, n=196, output=False)
    for got, ref in zip(out[0], (r["U"], r["F"], r["B"])):
        assert rel_l2(got, ref) <= 1e-10
    np.testing.assert_allclose(out[0][3], r["poynting"], rtol=1e-9, atol=1e-12 * np.abs(r["poynting"]).max())
