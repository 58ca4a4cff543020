"""Kernels whose XCDs take one range of blocks each (near_block): grids of fewer than eight blocks, of eight, with every
kind of remainder, against the oracle.  Explicit steps and the FP64 Hall step's explicit part are the oracle's bit for
bit; the solve is held to the 1e-12 of the other FP64 solve tests."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# cells per net: 216, 1296, 2160, 3780, 4608, 9504 (1 to 38 blocks of 256 cells, 2 to 75 of 128)
NETS = [(4, 12, 1), (6, 24, 2), (10, 20, 2), (9, 20, 4), (8, 48, 2), (12, 48, 3)]


@pytest.mark.parametrize("net", NETS)
@pytest.mark.parametrize("hall", [False, True])
def test_steps_match_the_oracle(net, hall):
    from mpcns_uns_amd import Device, workloads
    from oracle.oracle import Oracle

    w = workloads.build(net=net, hall=hall)
    dev, orc = Device(w["mesh"], w["cfg"]), Oracle(w["mesh"], w["cfg"])
    for x in (dev, orc):
        x.set_background(*w["background"])
        x.set_state(*w["state"])
    for _ in range(2):
        dt = dev.step(precision=0)[0] if hall else dev.step_explicit()
        assert dt == orc.step()[0] or hall
    UH, UNa, Phi = dev.get_state()
    oH, oNa, oPhi = orc.get_state()
    if not hall:
        assert np.array_equal(UH, oH) and np.array_equal(UNa, oNa) and np.array_equal(Phi, oPhi)
        return
    for a, b in ((UH, oH), (UNa, oNa), (Phi, oPhi)):
        assert np.linalg.norm(a - b) <= 1e-12 * np.linalg.norm(b)
