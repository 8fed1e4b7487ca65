"""FIT problems whose entities are not numbered the way the mesher does it, bit
for bit against the index-table layout (every item with its own faces, edges and
signs)."""
import ctypes as C

import numpy as np
import pytest

from tetfit_amd import Model, _ffi, configs
from tetfit_amd.device import Simulation

pytestmark = pytest.mark.gpu


class Altered:
    """A build with some arrays of its FIT operators replaced."""

    def __init__(self, build, **arrays):
        self._build, self._keep = build, []
        p = _ffi.tf_problem.from_buffer_copy(build.problem_ptr.contents)
        kinds = {np.dtype(np.int64): _ffi.i64p, np.dtype(np.int32): _ffi.i32p, np.dtype(np.int8): _ffi.i8p}
        for k, v in arrays.items():
            if np.isscalar(v):
                setattr(p.fit, k, v)
            else:
                v = np.ascontiguousarray(v)
                self._keep.append(v)
                setattr(p.fit, k, v.ctypes.data_as(kinds[v.dtype]))
        self.problem_ptr = C.pointer(p)

    def __getattr__(self, name):
        return getattr(self._build, name)


def small_cavity(workdir):
    return Model(configs.fit_cavity(str(workdir), n=7, step=0.1, n_steps=400, n_probes=4, name="ord7")).build(1)


def both_layouts(b, monkeypatch, prec, state, runs=(64, 1, 70)):
    """(grid order used, fields and probes) of the two layouts."""
    out = []
    for indexed in ("0", "1"):
        monkeypatch.setenv("TETFIT_FIT_INDEXED", indexed)
        print(f"case: E={b.n_edges} {prec} indexed={indexed}", flush=True)
        sim = Simulation(b, prec)
        sim.set_state(*state)
        got = []
        for n in runs:
            sim.run(n=n)
            got += [*sim.state(), *sim.probes()]
        got.append(sim.poynting())
        out.append((sim.fit_grid_order(), got))
        sim.close()
    return out


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
def test_common_edge_on_the_boundary(workdir, monkeypatch, prec):
    """A y edge of the x = 1 wall updated from four faces, one of them at the
    position that its missing neighbour's indices wrap around to."""
    b = small_cavity(workdir)
    o, n = b.fit_ops(), 7
    i, j, k = n, 3, 3
    e = int(np.flatnonzero(o["edge_sid"] == n * (n + 1) * (n + 1) + (k * n + j) * (n + 1) + i)[0])
    assert e in o["bc_edges"]
    xf = lambda c: (c * n + j) * (n + 1) + i
    zf = lambda a: (n + 1) * n * n + n * (n + 1) * n + (k * n + j) * n + a
    faces = [int(np.flatnonzero(o["face_sid"] == s)[0]) for s in (xf(k - 1), zf(i - 1), zf(i), xf(k))]
    ptr, face, sgn = o["ct_ptr"].copy(), o["ct_face"], o["ct_sgn"]
    a, z = ptr[e], ptr[e + 1]
    ptr[e + 1:] += 4 - (z - a)
    alt = Altered(b, ct_ptr=ptr, ct_face=np.concatenate([face[:a], faces, face[z:]]).astype(np.int32),
                  ct_sgn=np.concatenate([sgn[:a], [1, -1, 1, -1], sgn[z:]]).astype(np.int8),
                  common_edges=np.append(o["common_edges"], np.int32(e)), n_common=len(o["common_edges"]) + 1,
                  bc_edges=o["bc_edges"][o["bc_edges"] != e].astype(np.int32),
                  n_bc=int((o["bc_edges"] != e).sum()))
    rng = np.random.default_rng(5)
    state = [rng.standard_normal(m) for m in (b.n_edges, b.n_faces, b.n_faces)]
    (_, got), (indexed, ref) = both_layouts(alt, monkeypatch, prec, state)
    assert not indexed and not np.array_equal(ref[0][e], state[0][e])
    for x, y in zip(got, ref):
        np.testing.assert_array_equal(x, y)


def reordered(b, rng):
    """The same updates in other words: for a third of the common edges and of
    the faces the four entries are rotated by one and the sign turned round, for
    another third the first and third entry change places (both '+')."""
    o = b.fit_ops()
    face, curl, dual = o["ct_face"].copy(), o["curl"].copy(), o["dual_curl"].copy()
    edges = o["c_edge"].copy()

    def change(rows, get, put, sign):
        for r, how in zip(rows, rng.integers(0, 3, len(rows))):
            q = get(r)
            if how == 1:
                put(r, np.roll(q, 1))
                sign[r] *= -1
            elif how == 2:
                put(r, q[[2, 1, 0, 3]])

    def put_face(e, q):
        face[o["ct_ptr"][e]:o["ct_ptr"][e] + 4] = q

    def put_edge(f, q):
        edges[f] = q

    change(o["common_edges"], lambda e: face[o["ct_ptr"][e]:o["ct_ptr"][e] + 4].copy(), put_face, dual)
    change(o["tbc_faces"], lambda f: edges[f].copy(), put_edge, curl)
    return Altered(b, ct_face=face, dual_curl=dual, c_edge=edges.reshape(-1), curl=curl)


@pytest.mark.parametrize("prec", ["fp64", "fp32"])
@pytest.mark.parametrize("media", ["uniform", "random"])
def test_entities_in_another_order(workdir, monkeypatch, media, prec):
    """Orders and signs of their own keep the grid layout (a code per item),
    with probes and sources; bitwise the index tables, which sum in the same
    order."""
    rng = np.random.default_rng(6)
    if media == "uniform":
        b = reordered(small_cavity(workdir), rng)
    else:
        b = reordered(Model(configs.fit_random_media(str(workdir), n=12, n_steps=400, n_probes=4, name="ord12")).build(1),
                      rng)
    state = [rng.standard_normal(m) for m in (b.n_edges, b.n_faces, b.n_faces)]
    (grid, got), (indexed, ref) = both_layouts(b, monkeypatch, prec, state)
    assert grid and not indexed
    for x, y in zip(got, ref):
        np.testing.assert_array_equal(x, y)
