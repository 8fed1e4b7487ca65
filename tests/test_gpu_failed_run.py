"""A run that ends with an error after some of its steps: the probe records hold
the samples of the steps that were done and no others."""
import ctypes as C

import numpy as np
import pytest

from tetfit_amd import Model, _ffi, configs
from tetfit_amd.device import DeviceError, Simulation

pytestmark = pytest.mark.gpu


class OneSided:
    """A gfdtd build whose A lacks one off-diagonal entry (its mirror stays)."""

    def __init__(self, build):
        self._build = build
        A = build.dga_ops()["A"]
        row = np.repeat(np.arange(A["nrows"]), np.diff(A["rowptr"]))
        off = np.flatnonzero(row != A["col"])
        q = off[np.argmin(np.abs(A["val"][off]))]  # the smallest: the solves stay close to the full A's
        ptr = A["rowptr"].copy().astype(np.int64)
        ptr[row[q] + 1:] -= 1
        self._keep = [ptr, np.delete(A["col"], q).astype(np.int32), np.delete(A["val"], q)]
        p = _ffi.tf_problem.from_buffer_copy(build.problem_ptr.contents)
        p.dga.A.rowptr = self._keep[0].ctypes.data_as(_ffi.i64p)
        p.dga.A.col = self._keep[1].ctypes.data_as(_ffi.i32p)
        p.dga.A.val = self._keep[2].ctypes.data_as(_ffi.f64p)
        p.dga.A.nnz -= 1
        self.problem_ptr = C.pointer(p)

    def __getattr__(self, name):
        return getattr(self._build, name)


def test_samples_of_a_failed_run(workdir, monkeypatch):
    """The learned preconditioner needs a symmetric pattern, which is noticed
    when training starts, after 10 collection solves of a 40-step run. The
    collection's Jacobi solves are those of a plain run (two-kernel passes), so
    its samples are the same bits."""
    b = OneSided(Model(configs.kuhn_cavity(str(workdir), n=5, method="gfdtd", n_steps=60, n_probes=2, block=2,
                                           name="failed")).build(1))
    monkeypatch.setenv("TETFIT_CG_ONE", "0")
    sim = Simulation(b, "fp64")
    with pytest.raises(DeviceError, match="not symmetric"):
        sim.run(n=40, precond="learned", learn_steps=10)
    times, vals = sim.probes()
    sim.close()
    ref = Simulation(b, "fp64")
    ref.run(n=12)
    rt, rv = ref.probes()
    ref.close()
    assert 10 <= len(times) <= 11 and np.abs(rv[:10]).max() > 0
    np.testing.assert_array_equal(times, rt[:len(times)])
    np.testing.assert_array_equal(vals, rv[:len(times)])
