"""mhdg_prepare forms the derived fields of the resident state and nothing a step would need beside them: two launches, on
every shape of row, the fields the oracle's bit for bit."""
import numpy as np
import pytest

from test_gpu_explicit_layouts import _mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ions", [2, 10])
@pytest.mark.parametrize("kind", ["tets", "hexes", "solid", "mixed"])
def test_prepare_forms_the_fields_only(kind, ions):
    from mpcns_uns_amd import Device, workloads
    from oracle.oracle import Oracle

    mesh = _mesh(kind)
    cfg = workloads.physics_config(False) if ions == 2 else workloads.mars_config(False, n_species=ions)
    fs = [tuple((cfg.fs if ions == 2 else cfg.ion_fs)[s][m] for m in range(5)) for s in range(ions)]
    PhiAdd, Badd = mesh.background(workloads.B_IMF, workloads.DIPOLE_M, (0.0, 0.0, 0.0), 1e-3)
    U, Phi = mesh.seeded_species_state(cfg, fs, 0.05, 17, Badd)
    dev, orc = Device(mesh, cfg), Oracle(mesh, cfg)
    for x in (dev, orc):
        x.set_background(PhiAdd, Badd)
        x.set_state(U[0], U[1], Phi)
        for s in range(2, ions):
            x.set_species_state(s, U[s])
    dev.profile(True)
    dev.prepare()
    assert {k: v[0] for k, v in dev.profile_report().items()} == {"prepare": 1, "current": 1}
    orc.prepare()
    for n in ("W_H", "W_Na", "B_ind", "B_tot", "J", "u_plus"):
        assert np.array_equal(dev.derived(n), orc.derived(n)), n
