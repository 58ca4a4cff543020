"""Edges of many faces with more cells in their rows than twice the faces (cells elsewhere, of weight zero, between the
edge's own): the heavy blocks of the products hold a row of any length up to 2048 cells, and a longer one is refused.  The
sums are the same terms in the same order beside exact zeros, so the product is the oracle's bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class _Padded:
    """The mesh with `times` as many cells in the rows of its edges of more than 32 faces."""

    def __init__(self, mesh, times):
        from mpcns_uns_amd._lib import MeshDesc

        self.n_cells, self.n_faces, self.n_edges, self._mesh = mesh.n_cells, mesh.n_faces, mesh.n_edges, mesh
        self.array = mesh.array
        p, cell, w = mesh.array("ec_ptr"), mesh.array("ec_cell"), mesh.array("ec_weight")
        rng = np.random.default_rng(1)
        cells, weights, ptr = [], [], [0]
        for e, n in enumerate(np.diff(mesh.array("e2f.ptr"))):
            c, v = cell[p[e] : p[e + 1]], w[p[e] : p[e + 1]]
            if n > 32:
                others = np.setdiff1d(np.arange(mesh.n_cells, dtype=np.int32), c)
                more = (times - 1) * c.size
                more = rng.choice(others, more, replace=more > others.size)
                c, v = np.concatenate([c, more]), np.concatenate([v, np.zeros(more.size)])
                order = np.argsort(c, kind="stable")
                c, v = c[order], v[order]
            cells.append(c)
            weights.append(v)
            ptr.append(ptr[-1] + c.size)
        self._ptr, self._cell, self._w = np.array(ptr, np.int64), np.concatenate(cells).astype(np.int32), np.concatenate(weights)
        d, self._desc = mesh.desc(), MeshDesc()
        for name, _ in MeshDesc._fields_:
            setattr(self._desc, name, getattr(d, name))
        for name, a in (("ec_ptr", self._ptr), ("ec_cell", self._cell), ("ec_weight", self._w)):
            setattr(self._desc, name, a.ctypes.data_as(dict(MeshDesc._fields_)[name]))

    def desc(self):
        return self._desc


def _shell():
    from mpcns_uns_amd import Mesh, workloads

    return Mesh.shell(4, 40, 2, seed=3).boundary({1: "wall", 2: "farfield"}, u_inf=workloads.U_INF)


@pytest.mark.parametrize("times", [1, 3, 7])
def test_products_hold_the_longer_rows(times):
    from mpcns_uns_amd import Device, workloads
    from oracle.oracle import Oracle

    mesh = _Padded(_shell(), times)
    valence = int(np.max(np.diff(mesh.array("e2f.ptr"))))
    assert valence > 32 and (times < 3 or int(np.max(np.diff(mesh._ptr))) > 2 * valence)
    cfg = workloads.physics_config(True, ind_rtol=1e-12, ind_restart=40)
    dev, orc = Device(mesh, cfg), Oracle(mesh, cfg)
    rng = np.random.default_rng(5)
    B0, ne = rng.normal(size=3 * mesh.n_cells), 1.0 + 0.1 * rng.random(mesh.n_cells)
    phi, E = rng.normal(size=mesh.n_faces), rng.normal(size=mesh.n_edges) * mesh.array("edge_len")
    for x in (dev, orc):
        x.ind_set_frozen(B0, ne)
    assert np.array_equal(dev.ind_apply_F(phi), orc.ind_apply_F(phi))
    dt = 0.1 * float(np.min(mesh.array("edge_len"))) ** 2
    d = mesh.array("edge_mode") != 0
    a, b = dev.ind_solve(phi, E, d, dt, 0)[0], orc.ind_solve(phi, E, d, dt)[0]
    assert np.linalg.norm(a - b) <= 1e-10 * np.linalg.norm(b)


def test_too_long_a_row_is_refused():
    from mpcns_uns_amd import Device, workloads

    with pytest.raises(RuntimeError, match="cells around an edge"):
        Device(_Padded(_shell(), 60), workloads.physics_config(True))
