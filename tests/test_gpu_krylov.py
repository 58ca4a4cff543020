"""The Krylov vector kernels through the implicit solve: edge counts on both sides of the limit up to which the update sums
the dot products' partials itself, with and without a remainder of the 16-byte packs; more basis vectors than one
dot-product pass takes; a step so small that A P is nearly the identity, where classical Gram-Schmidt projects twice.
"""
import numpy as np
import pytest

from conftest import maxrel
from meshes import hex_workload

pytestmark = pytest.mark.gpu

# 12,678 edges (both precisions fold), 72,882 (FP32 folds, FP64 does not), 1,022 (two left over of packs of four), and a box
# of hexahedra with 523 (an odd count)
NETS = [(12, 48, 3), (24, 48, 9), (7, 17, 1), "box"]


def _systems(net):
    from mpcns_uns_amd import Device, workloads
    from oracle.oracle import Oracle

    kw = dict(ind_rtol=1e-12, ind_restart=40)
    w = hex_workload(True, **kw) if net == "box" else workloads.build(net=net, hall=True, **kw)
    m, cfg = w["mesh"], w["cfg"]
    dev, orc = Device(m, cfg), Oracle(m, cfg)
    rng = np.random.default_rng(5)
    B0 = w["background"][1] + 0.02 * rng.normal(size=3 * m.n_cells)
    ne = 1.0 + 0.1 * rng.random(m.n_cells)
    for x in (dev, orc):
        x.ind_set_frozen(B0, ne)
    E = rng.normal(size=m.n_edges) * m.array("edge_len")
    return w, dev, orc, E, m.array("edge_mode") != 0


@pytest.mark.parametrize("net", NETS)
@pytest.mark.parametrize("scale", [1e-4, 8.0, 200.0])
def test_solves_agree_with_the_oracle(net, scale):
    w, dev, orc, E, dirichlet = _systems(net)
    dt = scale * 0.1 * float(np.min(w["mesh"].array("edge_len"))) ** 2
    ref, it_ref, res_ref = orc.ind_solve(w["state"][2], E, dirichlet, dt)
    assert res_ref <= 1e-12
    for precision in (0, 3, 1):
        # each solve from a cold start: the warm start of the one before is dropped with the state
        dev.set_state(*w["state"])
        dev.profile(None)
        dev.profile(True)
        got, it, res = dev.ind_solve(w["state"][2], E, dirichlet, dt, precision)
        dev.profile(False)
        passes = dev.profile_report()[{0: "mgs_dots", 3: "multidot64", 1: "multidot"}[precision]][0]
        if scale == 200.0 and net != "box":
            assert it > 16  # one pass takes 16 vectors, a cycle has up to 40
        assert passes > it if precision == 3 and scale == 1e-4 else passes >= it  # a second projection is a pass of its own
        # both stop at a residual of 1e-12 |b|, A = I + dt F d1 with dt |F d1| of order `scale`
        assert res <= 1e-12 and maxrel(got, ref) < 1e-10, precision
        if precision == 0:
            assert abs(it - it_ref) <= 1
