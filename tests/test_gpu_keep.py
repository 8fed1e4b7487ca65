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
    """A small mesh forced into the wide-mesh kernels, with none, three eighths
    and all of an operator's slices loaded to stay, against the ordinary
    kernels; 9^3 gives slices past the first eight and a partial last one.
    gfdtd in the two-kernel CG passes, whose A has a share."""
    b = Model(configs.kuhn_cavity(str(workdir), n=9, method=method, n_steps=60, n_probes=2, block=3,
                                  name=f"keep_{method}")).build(1)
    monkeypatch.setenv("TETFIT_CG_ONE", "0")
    out = []
    for wide, keep in (("0", "0"), ("1", "0"), ("1", "3"), ("1", "8")):
        monkeypatch.setenv("TETFIT_SELL_WIDE", wide)
        monkeypatch.setenv("TETFIT_SELL_KEEP", keep)
        print(f"case: {method} {prec} wide={wide} keep={keep}", flush=True)
        sim = Simulation(b, prec)
        sim.set_profiling(True)
        sim.run(n=20)
        assert ("cg_w_kernel" if method == "gfdtd" else "sell_h_kernel") in sim.kernel_times()
        out.append((*sim.state(), sim.probes()[1], sim.poynting()))
        sim.close()
    for other in out[1:]:
        for a, e in zip(other, out[0]):
            np.testing.assert_array_equal(a, e)
    assert np.abs(out[0][0]).max() > 0
