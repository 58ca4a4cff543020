"""A descriptor with one face more, which no cell and no edge has: the step, the EMF entry and the gradient are those of the
mesh without it, bit for bit, and the face keeps its flux."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class _OneFaceMore:
    def __init__(self, mesh):
        from mpcns_uns_amd._lib import Incidence, MeshDesc

        self.n_cells, self.n_faces, self.n_edges, self._mesh = mesh.n_cells, mesh.n_faces + 1, mesh.n_edges, mesh
        d, self._desc, self._keep = mesh.desc(), MeshDesc(), []
        fields = dict(MeshDesc._fields_)
        for name in fields:
            setattr(self._desc, name, getattr(d, name))
        self._desc.n_faces = self.n_faces

        def give(a, kind):
            self._keep.append(a)
            return a.ctypes.data_as(kind)

        for name in ("f2e", "f2c"):
            p = mesh.array(name + ".ptr")
            inc = Incidence()
            inc.idx, inc.sgn = getattr(d, name).idx, getattr(d, name).sgn
            inc.ptr = give(np.append(p, p[-1]), dict(Incidence._fields_)["ptr"])
            setattr(self._desc, name, inc)
        more = dict(face_kind=np.zeros(1, np.int8), face_area=np.array([0.0, 1.0, 0.0]), face_center=np.full(3, 2.0),
                    face_area_mag=np.ones(1), star2=np.ones(1))
        for name, x in more.items():
            setattr(self._desc, name, give(np.concatenate([mesh.array(name), x]), fields[name]))

    def desc(self):
        return self._desc


@pytest.mark.parametrize("kind", ["tets", "mixed"])
def test_same_as_without_it(kind):
    from mpcns_uns_amd import Device, workloads
    from test_gpu_explicit_layouts import _mesh

    mesh = _mesh(kind)
    cfg = workloads.physics_config(True)
    fs = [tuple(cfg.fs[s][m] for m in range(5)) for s in range(2)]
    PhiAdd, Badd = mesh.background(workloads.B_IMF, workloads.DIPOLE_M, (0.0, 0.0, 0.0), 1e-3)
    U, Phi = mesh.seeded_species_state(cfg, fs, 0.05, 17, Badd)
    more = lambda x: np.append(x, 0.25)
    out = []
    for m, f in ((mesh, lambda x: x), (_OneFaceMore(mesh), more)):
        dev = Device(m, cfg)
        dev.set_background(f(PhiAdd), Badd)
        dev.set_state(U[0], U[1], f(Phi))
        J, g = dev.step_vjp(2, 1.2, 3.2)
        dev.step_explicit()
        dev.step(precision=0)
        UH, UNa, B = dev.get_state()
        emf = dev.ideal_emf(dev.derived("u_plus"), dev.derived("B_tot"), dev.derived("B_ind"), f(Phi), f(Phi))
        out.append((J, g["U_H"], g["Phi"][: mesh.n_faces], UH, UNa, B[: mesh.n_faces], emf))
    assert B[-1] == 0.25 and g["Phi"][-1] == 0.0
    for a, b in zip(*out):
        assert np.array_equal(a, b)
