"""Every form of the grid-order FIT kernels (items per thread, palettes, plain
coefficients loaded either way), bit for bit against the index-table layout. The
grids are not cubes and no direction's item count is a multiple of 4 x 256, so
each form has a partial last block in each direction."""
import re

import numpy as np
import pytest

from tetfit_amd import Model, configs
from tetfit_amd.device import Simulation

pytestmark = pytest.mark.gpu


def brick(path, y, z):
    """The unit-box input cut at y and z (step 1/n)."""
    text = open(path).read()
    for ax, stop in (("y", y), ("z", z)):
        text = re.sub(r"SET %sgrid \{0,([^,]+),[^}]+\}" % ax, r"SET %sgrid {0,\1,%r}" % (ax, stop), text)
    open(path, "w").write(text)
    return Model(path).build(1)


def build(workdir, media):
    n = 22
    if media == "uniform":
        return brick(configs.fit_cavity(str(workdir), n=n, step=1.0 / n, n_steps=400, n_probes=5, name="ker_u",
                                        pml={"+x": 0.2}), 0.8, 0.7)
    return brick(configs.fit_random_media(str(workdir), n=n, n_steps=400, n_probes=5, name="ker_r"), 0.8, 0.7)


@pytest.mark.parametrize("prec,items", [("fp64", 1), ("fp64", 2), ("fp32", 1), ("fp32", 2), ("fp32", 4)])
@pytest.mark.parametrize("media,nt", [("uniform", 0), ("random", 0), ("random", 1)])
def test_forms_bitwise(workdir, monkeypatch, media, nt, prec, items):
    b = build(workdir, media)
    o = b.fit_ops()
    nx, ny, nz = o["cells"]
    counts = [nx * (ny + 1) * (nz + 1), (nx + 1) * ny * (nz + 1), (nx + 1) * (ny + 1) * nz, (nx + 1) * ny * nz,
              nx * (ny + 1) * nz, nx * ny * (nz + 1)]
    assert len({nx, ny, nz}) == 3 and all(c % 1024 for c in counts)
    monkeypatch.setenv("TETFIT_FIT_ITEMS", str(items))
    monkeypatch.setenv("TETFIT_FIT_NT", str(nt))
    rng = np.random.default_rng(7)
    state = [rng.standard_normal(m) for m in (b.n_edges, b.n_faces, b.n_faces)]
    got = []
    for indexed in ("0", "1"):
        monkeypatch.setenv("TETFIT_FIT_INDEXED", indexed)
        print(f"case: {media} {prec} items={items} nt={nt} indexed={indexed} E={b.n_edges}", flush=True)
        sim = Simulation(b, prec)
        assert sim.fit_grid_order() == (indexed == "0")
        sim.set_state(*state)
        sim.run(n=67)
        got.append([*sim.state(), *sim.probes(), sim.poynting()])
        sim.close()
    for a, e in zip(*got):
        np.testing.assert_array_equal(a, e)
    assert np.abs(got[0][0]).max() > 0
