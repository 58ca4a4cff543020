"""The product's first launch (face fluxes and cell fields together) on the shapes it serves: tetrahedra and hexahedra with
solid cells and boundary faces, against the oracle's step; and the meshes it does not serve, which keep the separate launches.
Bounds: 1e-12 of each field for the reference iteration (the kernel keeps the order of every sum), 1e-7 for the others,
which stop elsewhere below the same residual of 1e-8 of the right-hand side."""
import numpy as np
import pytest

from test_gpu_explicit_layouts import _mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1, 3])
@pytest.mark.parametrize("kind", ["tets", "hexes", "solid", "mixed"])
def test_hall_step_matches_the_oracle(kind, precision):
    from mpcns_uns_amd import Device, workloads
    from oracle.oracle import Oracle

    mesh = _mesh(kind)
    cfg = workloads.physics_config(True)
    fs = [tuple(cfg.fs[s][m] for m in range(5)) for s in range(2)]
    PhiAdd, Badd = mesh.background(workloads.B_IMF, workloads.DIPOLE_M, (0.0, 0.0, 0.0), 1e-3)
    U, Phi = mesh.seeded_species_state(cfg, fs, 0.05, 17, Badd)
    dev, orc = Device(mesh, cfg), Oracle(mesh, cfg)
    for x in (dev, orc):
        x.set_background(PhiAdd, Badd)
        x.set_state(U[0], U[1], Phi)
    for _ in range(2):
        dev.step(precision=precision)
        orc.step()
    dev.profile(True)
    dev.step(precision=precision)
    orc.step()
    names = {k for k in dev.profile_report()}
    fused = {"flux_cell", "flux_cell_f32"} & names
    assert bool(fused) == (kind != "mixed"), names
    tol = 1e-12 if precision == 0 else 1e-7
    for a, b in zip(dev.get_state(), orc.get_state()):
        assert np.linalg.norm(a - b) <= tol * np.linalg.norm(b)
