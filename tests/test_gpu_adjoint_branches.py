"""The reverse sweep over the shapes and branches its kernels are instantiated for, against the tangent: <grad J, v> = dJ[v] per
input.  Rows of four faces (tetrahedra), six (hexahedra) and of varying length, solid cells, wall, inflow and outflow
faces, edges of valence up to 6 (registers), up to 32 (one thread) and above (one block), meshes that end inside a block,
first and second order, cells at the pressure floor, and a time step set by dt_max instead of a cell.

The tangent takes the branch of the same values and both sum about 1e2 terms per output in FP64: 1e-9 of the sum of the
inputs' parts is far above their rounding and far below a missing term."""
import numpy as np
import pytest

from test_gpu_explicit_layouts import _mesh

pytestmark = pytest.mark.gpu
R0, R1 = 1.2, 3.2


def _case(kind, second_order=1, seed=17, **kw):
    from mpcns_uns_amd import Device, workloads

    mesh = workloads.build(net=(4, 40, 2), hall=False)["mesh"] if kind == "poles" else _mesh(kind)
    cfg = workloads.physics_config(False, second_order=second_order, **kw)
    fs = [tuple(cfg.fs[s][m] for m in range(5)) for s in range(2)]
    PhiAdd, Badd = mesh.background(workloads.B_IMF, workloads.DIPOLE_M, (0.0, 0.0, 0.0), 1e-3)
    U, Phi = mesh.seeded_species_state(cfg, fs, 0.05, seed, Badd)
    dev = Device(mesh, cfg)
    dev.set_background(PhiAdd, Badd)
    dev.set_state(U[0], U[1], Phi)
    return mesh, dev


def _check(mesh, dev, steps=3, dt_max=1e9):
    J, g = dev.step_vjp(steps, R0, R1, dt_max=dt_max)
    rng = np.random.default_rng(5)
    seeds = {k: rng.normal(size=np.size(g[k])) * (1e-6 if k == "U_Na" else 1e-3) for k in ("U_H", "U_Na", "Phi", "PhiAdd", "Badd", "fs", "E_inf")}
    parts = {k: float(np.ravel(g[k]) @ seeds[k]) for k in seeds}
    scale = sum(abs(v) for v in parts.values())
    assert J > 0 and scale > 0 and all(np.isfinite(v) for v in parts.values())
    for k in seeds:
        Jt, dJ = dev.explicit_tangent(steps, R0, R1, dt_max=dt_max, **{"d" + k: seeds[k]})
        assert J == Jt
        assert abs(parts[k] - dJ) <= 1e-9 * scale, (k, parts[k], dJ)
    return parts


@pytest.mark.parametrize("second_order", [1, 0])
@pytest.mark.parametrize("kind", ["tets", "poles", "hexes", "solid", "mixed"])
def test_adjoint_is_the_tangent_transposed(kind, second_order):
    parts = _check(*_case(kind, second_order))
    assert parts["fs"] != 0.0


@pytest.mark.parametrize("kind", ["tets", "mixed"])
def test_cells_at_the_pressure_floor(kind):
    """Half of the Na+ cells start below the floor: recovery and update both take their clamped branches."""
    _check(*_case(kind, p_floor=1e-4), steps=2)


@pytest.mark.parametrize("kind", ["tets", "hexes"])
def test_step_set_by_the_caller(kind):
    mesh, dev = _case(kind)
    _check(mesh, dev, dt_max=0.25 * dev.step_explicit())


def test_repeated_and_longer_sweeps():
    """A sweep leaves the state alone and repeats bit for bit, also after a shorter one and on a context that keeps its
    work arrays; no step at all is the gradient of the energy itself."""
    _, dev = _case("tets")
    a, b, c = dev.step_vjp(4, R0, R1), dev.step_vjp(1, R0, R1), dev.step_vjp(4, R0, R1)
    assert a[0] == c[0] and a[0] != b[0]
    for k in a[1]:
        assert np.array_equal(a[1][k], c[1][k]), k
    J, g = dev.step_vjp(0, R0, R1)
    assert J == dev.shell_energy(R0, R1) and not np.any(g["U_H"]) and not np.any(g["PhiAdd"]) and np.any(g["Phi"])
