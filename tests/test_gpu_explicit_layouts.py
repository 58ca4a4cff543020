"""The fused step's explicit stage over the shapes its kernels are instantiated for: rows of four faces (tetrahedra), of
six (hexahedra) and of varying length (hexahedra and pyramids), two ions and more (record rows with and without padding,
blocks whose last threads hold no ion), first and second order, meshes that end inside a block, solid cells.  The
kernels keep the order of every sum, so the oracle's step is matched bit for bit.
"""
import numpy as np
import pytest

from meshes import box_cells, pyramid_split

pytestmark = pytest.mark.gpu


def _mesh(kind):
    from mpcns_uns_amd import Mesh, workloads

    if kind == "tets":
        return Mesh.shell(7, 13, 2, seed=3).boundary({1: "wall", 2: "farfield"}, u_inf=workloads.U_INF)
    xyz, cells, tags = box_cells(5, 4, 3, (1.5, -1.0, -1.0), (3.5, 1.0, 1.0))
    if kind == "mixed":
        xyz, cells = pyramid_split(xyz, cells)
    material = None
    if kind == "solid":
        material = np.zeros(len(cells), np.int32)
        material[[0, 7, 31]] = 1
    mesh = Mesh.from_cells(xyz, cells, material=material, tags=tags)
    return mesh.boundary({1: "wall", 2: "inflow"}, default="outflow", u_inf=workloads.U_INF)


@pytest.mark.parametrize("second_order", [1, 0])
@pytest.mark.parametrize("ions", [2, 3, 4, 7, 10])
@pytest.mark.parametrize("kind", ["tets", "hexes", "solid", "mixed"])
def test_explicit_step_bitwise(kind, ions, second_order):
    from mpcns_uns_amd import Device, workloads
    from oracle.oracle import Oracle

    mesh = _mesh(kind)
    if ions == 2:
        cfg = workloads.physics_config(False, second_order=second_order)
        fs = [tuple(cfg.fs[s][m] for m in range(5)) for s in range(2)]
    else:
        cfg = workloads.mars_config(False, n_species=ions, second_order=second_order)
        fs = [tuple(cfg.ion_fs[s][m] for m in range(5)) for s in range(ions)]
    PhiAdd, Badd = mesh.background(workloads.B_IMF, workloads.DIPOLE_M, (0.0, 0.0, 0.0), 1e-3)
    U, Phi = mesh.seeded_species_state(cfg, fs, 0.05, 17, Badd)
    dev, orc = Device(mesh, cfg), Oracle(mesh, cfg)
    for x in (dev, orc):
        x.set_background(PhiAdd, Badd)
        x.set_state(U[0], U[1], Phi)
        for s in range(2, ions):
            x.set_species_state(s, U[s])
    for _ in range(2):
        assert dev.step_explicit() == orc.step()[0]
    for s in range(ions):
        assert np.array_equal(dev.get_species_state(s), orc.get_species_state(s)), s
        assert np.array_equal(dev.get_species_prim(s), orc.get_species_prim(s)), s
    assert np.array_equal(dev.get_state()[2], orc.get_state()[2])
    for n in ("W_H", "W_Na", "B_ind", "B_tot", "J", "u_plus", "E"):
        assert np.array_equal(dev.derived(n), orc.derived(n)), n
    dev.prepare()
    orc.prepare()
    for n in ("W_H", "W_Na", "B_ind", "B_tot", "J", "u_plus"):
        assert np.array_equal(dev.derived(n), orc.derived(n)), n
