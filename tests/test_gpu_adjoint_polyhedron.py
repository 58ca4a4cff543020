"""The reverse sweep on a cell of more faces than a machine word has bits: a polyhedron of 72 triangles inside a layer of
72 prisms, against the tangent (per input, as in test_gpu_adjoint_branches).  Every primitive grows away from one face and
is nearly flat towards it, so that face sets the limiter, by its neighbours' extreme or by the relative limit; it is given on
both sides of number 64."""
import numpy as np
import pytest

from meshes import polyhedron
from test_gpu_adjoint_branches import _check

pytestmark = pytest.mark.gpu


def _state(cfg, mesh, face):
    """Conservative states of both ions and the entry of the polyhedron's row that limits its gradients."""
    c2f = mesh.array("c2f.idx")[: 72]
    xc, fc = mesh.array("cell_center").reshape(-1, 3), mesh.array("face_center").reshape(-1, 3)
    away = lambda x: (x - xc[0]) / np.linalg.norm(x - xc[0], axis=-1, keepdims=True)
    cosine = away(xc[1:]) @ -away(fc[c2f[face]])
    shape = np.concatenate([[0.0], np.where(cosine > 0, 0.4 * cosine, 0.002 * cosine)])[:, None]
    U = []
    for s in range(2):
        w = np.array([cfg.fs[s][m] for m in range(5)]) + np.array([0, 0, 0.1, -0.1, 0])
        w = w * (1 + shape) + 0.001 * np.random.default_rng(s).random((mesh.n_cells, 5)) * w
        u = np.column_stack([w[:, 0], w[:, :1] * w[:, 1:4], w[:, 4] / (cfg.gamma - 1) + 0.5 * w[:, 0] * (w[:, 1:4] ** 2).sum(1)])
        U.append(u.ravel())
    return U


@pytest.mark.parametrize("rel_limit", [0.0, 0.002])
@pytest.mark.parametrize("second_order", [1, 0])
@pytest.mark.parametrize("face", [3, 66, 70])
def test_adjoint_is_the_tangent_transposed(face, second_order, rel_limit):
    from mpcns_uns_amd import Device, Mesh, workloads

    xyz, cells, tags = polyhedron()
    assert len(cells[0]) == 72
    mesh = Mesh.from_cells(xyz, cells, tags=tags).boundary({1: "wall", 2: "inflow"}, default="outflow", u_inf=workloads.U_INF)
    cfg = workloads.physics_config(False, second_order=second_order, recon_rel_limit=rel_limit)
    dev = Device(mesh, cfg)
    PhiAdd, Badd = mesh.background(workloads.B_IMF, workloads.DIPOLE_M, (0.0, 0.0, 0.0), 1e-3)
    dev.set_background(PhiAdd, Badd)
    rng = np.random.default_rng(5)
    Phi = 0.01 * rng.normal(size=mesh.n_edges)[mesh.array("f2e.idx")] * mesh.array("f2e.sgn")
    U = _state(cfg, mesh, face)
    dev.set_state(U[0], U[1], np.add.reduceat(Phi, mesh.array("f2e.ptr")[:-1]))
    _check(mesh, dev, steps=2)
