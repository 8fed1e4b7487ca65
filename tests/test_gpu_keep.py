"""The wide-mesh kernels load part of an operator's slices to stay in cache
(SellView::keep) and the rest non-temporally: the loads' kind changes no bit."""
import numpy as np
import pytest

from tetfit_amd import Model, configs
from tetfit_amd.device import Simulation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("method", ["dga", "gfdtd"])
def test_resident_share_bitwise(workdir, monkeypatch, method, prec):
    """A small mesh forced into the wide-mesh kernels (every slice resident:
    the operators fit) against the ordinary kernels; 9^3 gives slices past the
    first eight and a partial last one."""
    b = Model(configs.kuhn_cavity(str(workdir), n=9, method=method, n_steps=60, n_probes=2, block=3,
                                  name=f"keep_{method}")).build(1)
    out = []
    for wide in ("0", "1"):
        monkeypatch.setenv("TETFIT_SELL_WIDE", wide)
        sim = Simulation(b, prec)
        sim.run(n=20)
        out.append((*sim.state(), sim.probes()[1], sim.poynting()))
        sim.close()
    for a, e in zip(*out):
        np.testing.assert_array_equal(a, e)
    assert np.abs(out[0][0]).max() > 0
