"""The reverse sweep keeps every operation and every sum of forward-mode columns in their order.

Over a shell of four layers the inflow boundary is further from the objective (1.2 <= r <= 1.5) than a few steps reach, so
the gradients with respect to the inflow EMF and the free stream are what cancelling sums leave (1e-60 to 1e-35 beside
gradients of 1e-1): another order of a sum anywhere in the sweep changes their leading digits.  The values below are those
of the sweep that formed every column as a pass of Dual arithmetic over the whole operation, one kernel per operation;
the other gradients are compared by a checksum of their bytes.  Rows of four faces, of six and of varying length,
a valence above the one-thread limit, the first order, cells at the pressure floor and dt_max setting the step.
"""
import zlib

import numpy as np
import pytest

from test_gpu_explicit_layouts import _mesh

pytestmark = pytest.mark.gpu

# case: (net or mesh kind, configuration, steps, dt_max over the CFL step or 0)
CASES = {
    "layers4": ((12, 24, 4), {}, 4, 0),
    "layers4_poles": ((9, 80, 4), {}, 5, 0),
    "layers4_first_order": ((12, 24, 4), dict(second_order=0), 4, 0),
    "tets_floor": ("tets", dict(p_floor=1e-4), 2, 0),
    "hexes": ("hexes", {}, 3, 0),
    "mixed": ("mixed", {}, 3, 0.25),
    "solid": ("solid", dict(recon_rel_limit=0.05), 3, 0),
}


def gradient(case):
    from mpcns_uns_amd import Device, Mesh, workloads

    mesh, kw, steps, dt = CASES[case]
    if isinstance(mesh, tuple):
        mesh = Mesh.shell(*mesh, seed=5).boundary({1: "wall", 2: "farfield"}, u_inf=workloads.U_INF)
        r = (1.2, 1.5)
    else:
        mesh, r = _mesh(mesh), (1.2, 3.2)
    cfg = workloads.physics_config(False, **kw)
    fs = [tuple(cfg.fs[s][m] for m in range(5)) for s in range(2)]
    PhiAdd, Badd = mesh.background(workloads.B_IMF, workloads.DIPOLE_M, (0.0, 0.0, 0.0), 1e-3)
    U, Phi = mesh.seeded_species_state(cfg, fs, 0.05, 17, Badd)
    dev = Device(mesh, cfg)
    dev.set_background(PhiAdd, Badd)
    dev.set_state(U[0], U[1], Phi)
    dt_max = 1e9
    if dt:
        dt_max = dt * dev.step_explicit()
        dev.set_state(U[0], U[1], Phi)
    J, g = dev.step_vjp(steps, *r, dt_max=dt_max)
    return J, g


def digest(J, g):
    """J, E_inf and fs in hexadecimal, and the checksum of the other gradients' bytes (a zero counts as +0)."""
    small = [float(v).hex() for v in (J, *g["E_inf"], *np.ravel(g["fs"]))]
    crc = 0
    for k in ("U_H", "U_Na", "Phi", "PhiAdd", "Badd"):
        crc = zlib.crc32((np.asarray(g[k]) + 0.0).tobytes(), crc)
    return small, crc


EXPECTED = {
    "layers4": (
        [
            "0x1.ecb96333e2bc7p-4", "-0x1.89a2364bed528p-200", "0x1.4c54771e15de2p-201", "-0x1.73cdfd5fc23c8p-207",
            "0x1.52e567c09f491p-160", "-0x1.1f2541c9ec96cp-154", "0x1.e6fc8da2f1f73p-159", "0x1.caa603f7440eap-156",
            "-0x1.f85f1a07a29cfp-159", "0x1.3b8d3d130f6a3p-162", "0x1.923cbfe913c10p-167", "-0x1.916a8234e534fp-169",
            "-0x1.afaf622b3316cp-172", "0x1.687a82cbc3d22p-156",
        ],
        0xc981c8e3,
    ),
    "layers4_poles": (
        [
            "0x1.0b312b5925b37p-3", "-0x1.64328bf6b0250p-109", "-0x1.52ca4140e1f87p-108", "0x1.446c7caa9eeebp-112",
            "0x1.486924fd6527dp-57", "-0x1.a914d2b6fdc20p-53", "-0x1.02d6f31337e65p-63", "0x1.751f89a6d7accp-59",
            "-0x1.7e38f6db565b4p-57", "-0x1.fb744cfea1aeap-66", "-0x1.29fd43140a375p-69", "0x1.bd9292498761cp-73",
            "-0x1.c2f661e66af96p-73", "0x1.250532df0d276p-62",
        ],
        0x38e67756,
    ),
    "layers4_first_order": (
        [
            "0x1.ecb99d928432ap-4", "-0x1.2b833508cb549p-198", "-0x1.61c7ce8f3ad53p-201", "-0x1.ec76923dee70ep-200",
            "0x0.0p+0", "0x0.0p+0", "0x0.0p+0", "0x0.0p+0",
            "0x0.0p+0", "0x0.0p+0", "0x0.0p+0", "0x0.0p+0",
            "0x0.0p+0", "0x0.0p+0",
        ],
        0xb0a2d768,
    ),
    "tets_floor": (
        [
            "0x1.124c3341c7fb0p+0", "0x1.e2b77ef2bef92p-12", "0x1.88a08aafc00cdp-7", "0x1.52569354840e6p-12",
            "-0x1.3b137018f7999p-24", "-0x1.9bb36fe2759b7p-19", "0x1.0924f8ab35553p-24", "0x1.2c606c95804fap-24",
            "0x1.2fe8805f85c9cp-19", "-0x1.57cf354f00c43p-29", "-0x1.1d3cb2fb36c9cp-33", "0x1.08245f0128a78p-37",
            "0x1.334a153d9b5d7p-39", "0x1.a3d378838b17fp-24",
        ],
        0xc9ff28c0,
    ),
    "hexes": (
        [
            "0x1.71ffe4168d28fp-7", "0x0.0p+0", "0x1.82cdbb8914f10p-9", "-0x1.4940f71aac03ep-17",
            "0x1.b381aedab6f8ep-23", "-0x1.584ca6c05a23dp-14", "0x1.b291fbf595751p-22", "-0x1.1d9c11e62ee2ep-22",
            "0x1.60d7c820f4264p-15", "-0x1.0d374901a8e30p-32", "-0x1.ed9a6dc806d3ap-29", "0x1.13606422c187cp-35",
            "-0x1.3bc9d8012f1fdp-37", "0x1.dfb69daef4059p-20",
        ],
        0xb01e17d9,
    ),
    "mixed": (
        [
            "0x1.4face7cbb5117p-7", "0x0.0p+0", "0x1.a1d88d0e344f6p-18", "0x1.e67889e0b2ae5p-26",
            "-0x1.b6a370119a3cep-31", "-0x1.887561c48c7b4p-24", "-0x1.11177cc3c5672p-30", "-0x1.5dd48bd687540p-34",
            "0x1.ed839917641b2p-26", "0x1.5e1c9d1165123p-34", "-0x1.07c4741685757p-38", "0x1.4720a047b2c6ep-45",
            "-0x1.61a9629307a34p-46", "0x1.014a966cd1de7p-29",
        ],
        0xad00ab6e,
    ),
    "solid": (
        [
            "0x1.63da2b1288a88p-7", "0x0.0p+0", "0x1.8f5ee65a56ee1p-9", "-0x1.ab4ab554323edp-17",
            "0x1.2e9b4b1afebf7p-24", "-0x1.5b19b992c058ap-14", "0x1.5c14b1363ac38p-22", "-0x1.27b238663ad53p-22",
            "0x1.649aaaf7c11d7p-15", "0x1.6389d99159cecp-30", "-0x1.f2bd40b622960p-29", "0x1.5e09bb81734bfp-35",
            "-0x1.8217379ac2e2ap-37", "0x1.e641632195584p-20",
        ],
        0x7e6c42e6,
    ),
}


@pytest.mark.parametrize("case", CASES)
def test_bits_of_the_gradient(case):
    J, g = gradient(case)
    small, crc = digest(J, g)
    expected, expected_crc = EXPECTED[case]
    assert [float.fromhex(v) for v in small] == [float.fromhex(v) for v in expected]
    assert crc == expected_crc
