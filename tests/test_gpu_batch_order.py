"""Batches in their instances' locality order (each instance's block of the
stacked problem relabeled by its own ranks). Rows keep their entries' order
and the dga step has no reductions, so a dga batch is bitwise the one in the
instances' numbering (tolerance 0). A gfdtd batch sums its CG scalars in
another row order, so its solves, each stopped at relative residual
tol = 1e-10, agree within steps x tol x cond(A) / 2 per field; cond(A) of these
meshes (epsilon contrast 10, jitter 0.2) is below 1e3: 12 steps -> 6e-7."""

import ctypes as C

import numpy as np
import pytest

from tetfit_amd import _ffi, configs
from tetfit_amd.host import Model

pytestmark = pytest.mark.gpu

STEPS = 12


def instances(tmp_path, method):
    """Sizes around the 64-row slice: a block of 1 cube, ragged ones, and one
    whose rows span several slices."""
    out = []
    for k, (n, seed, f) in enumerate([(2, 1, 2e8), (5, 2, 3e8), (3, 3, 1.5e8), (9, 4, 4e8)]):
        p = configs.kuhn_cavity(str(tmp_path), n=n, method=method, n_steps=STEPS, n_probes=3, block=2, seed=seed,
                                eps_range=(1.0, 10.0), freq=f, name=f"o{method}{k}",
                                **({"tol": 1e-10} if method == "gfdtd" else {}))
        out.append(Model(p).build(1))
    return out


@pytest.mark.parametrize("method,prec", [("dga", "fp64"), ("dga", "fp32"), ("gfdtd", "fp64")])
def test_batch_locality_order(tmp_path, monkeypatch, method, prec):
    from tetfit_amd.device import BatchSimulation
    bs = instances(tmp_path, method)
    runs = {}
    for order in ("numbering", "rank"):
        if order == "numbering":
            monkeypatch.setenv("TETFIT_TET_ORDER", "numbering")
        else:
            monkeypatch.delenv("TETFIT_TET_ORDER")
        print(f"case: batch {method} {prec} {order}", flush=True)
        sim = BatchSimulation(bs, prec, sample_every=1)
        sim.run(STEPS)
        runs[order] = [sim.probes(k)[1:] + tuple(sim.state(k)) for k in range(len(bs))]
        sim.close()
    for k, (a, b) in enumerate(zip(runs["numbering"], runs["rank"])):
        assert np.abs(a[1]).max() > 0, k
        for x, y in zip(a, b):
            if method == "dga":
                np.testing.assert_array_equal(x, y)
            else:
                assert np.linalg.norm(np.asarray(x) - y) <= 6e-7 * np.linalg.norm(x), k


class Altered:
    """A build whose problem carries other locality ranks."""

    def __init__(self, build, edge_rank, face_rank):
        self._build = build
        self._keep = [np.ascontiguousarray(r, np.int32) for r in (edge_rank, face_rank)]
        p = _ffi.tf_problem.from_buffer_copy(build.problem_ptr.contents)
        p.dga.edge_rank, p.dga.face_rank = (r.ctypes.data_as(_ffi.i32p) for r in self._keep)
        self.problem_ptr = C.pointer(p)

    def __getattr__(self, name):
        return getattr(self._build, name)


@pytest.mark.parametrize("method", ["dga", "gfdtd"])
def test_batch_with_unusable_ranks(tmp_path, monkeypatch, method):
    """Ranks that are no permutation of an instance's own entities (repeated
    ones, and ones past its block of the stacked problem) are not used for that
    instance, as in a batch in the instances' numbering; the others keep their
    order."""
    from tetfit_amd.device import BatchSimulation
    good = instances(tmp_path, method)
    bad = list(good)
    bad[0] = Altered(good[0], np.zeros(good[0].n_edges), good[0].face_rank())
    bad[2] = Altered(good[2], good[2].edge_rank() + 1, good[2].face_rank())
    runs = []
    for order, bs in (("numbering", good), ("rank", bad)):
        monkeypatch.setenv("TETFIT_TET_ORDER", order)
        sim = BatchSimulation(bs, "fp64", sample_every=1)
        sim.run(STEPS)
        runs.append([sim.probes(k)[1:] + tuple(sim.state(k)) for k in range(len(bs))])
        sim.close()
    for k, (a, b) in enumerate(zip(*runs)):
        assert np.abs(a[1]).max() > 0, k
        for x, y in zip(a, b):
            if method == "dga":
                np.testing.assert_array_equal(x, y)
            else:
                assert np.linalg.norm(np.asarray(x) - y) <= 6e-7 * np.linalg.norm(x), k
