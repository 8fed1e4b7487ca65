"""FIT coefficient palettes and the stores of B they allow, bit for bit against
the index-table layout (which keeps plain coefficient arrays and stores B
every step)."""
import numpy as np
import pytest

from tetfit_amd import Model, _ffi, configs
from tetfit_amd.device import Simulation

pytestmark = pytest.mark.gpu


def _build(workdir, media):
    if media == "uniform":
        return Model(configs.fit_cavity(str(workdir), n=13, step=0.1, n_steps=400, n_probes=5, name="pal_u",
                                        pml={"+x": 0.35})).build(1)
    # 24^3: more distinct E coefficients than a palette holds (plain arrays), H in a palette
    return Model(configs.fit_random_media(str(workdir), n=24, n_steps=400, n_probes=5, name="pal_r")).build(1)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("media", ["uniform", "random"])
def test_palette_bitwise(workdir, monkeypatch, media, prec):
    """Runs of 64 (a replay and nothing after it), 1 and 70 steps without
    sampling: B is whole after each. Then the probes change between sampled
    runs (replays of other sample counts among them): a face that was probed,
    one that stays probed, new ones. Last an output period that skips steps."""
    b = _build(workdir, media)
    got = {}
    for indexed in ("0", "1"):
        monkeypatch.setenv("TETFIT_FIT_INDEXED", indexed)
        print(f"case: {media} {prec} indexed={indexed} E={b.n_edges}", flush=True)
        out = []
        sim = Simulation(b, prec, output=False)
        for n in (64, 1, 70):
            sim.run(n=n)
            out += list(sim.state())
        _ffi.hip_lib().tf_set_output(sim._h, 0.0, 0.0)
        p, _, npr = b.probes_raw()
        for lo, n, steps in ((0, npr, 133), (1, 2, 5), (0, 0, 70), (2, npr - 2, 65), (0, npr, 64)):
            part = (_ffi.tf_probe * max(n, 1))(*[p[lo + k] for k in range(n)])
            assert _ffi.hip_lib().tf_set_probes(sim._h, part, n) == 0
            sim.n_probes = n
            sim.run(n=steps)
            out += [*sim.probes(), *sim.state()]
        _ffi.hip_lib().tf_set_output(sim._h, sim.next_step * b.dt, 2.5 * b.dt)
        sim.run(n=70)
        out += [*sim.probes(), *sim.state()]
        out.append(sim.poynting())
        sim.close()
        got[indexed] = out
    for a, e in zip(got["0"], got["1"]):
        np.testing.assert_array_equal(a, e)
    assert np.abs(got["0"][2]).max() > 0
