"""Kernels that do the work of several simpler ones: a step's functions sharing
launches (des_step against the entry points called one by one) and the force
contributions that a wave stores in slot order through LDS (per-pass launches)
against those that every lane stores for itself (the persistent launch).  The
same operations on the same values: bitwise equal, so no tolerance."""
import numpy as np
import pytest

import scenarios as SC
from dynearthsol_amd import abi

pytestmark = pytest.mark.gpu


def _same(a, b):
    assert a.keys() == b.keys()
    for k in a:
        assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("name", ["evp3", "bc3", "bc2", "dynmat3", "psevp2", "viscous2"])
def test_step_equals_its_functions_one_by_one(name):
    from dynearthsol_amd.lib import DesModel
    m = SC.build(name, nelem=1500)
    print(name, m.nelem, "elements", flush=True)
    g, h = DesModel(m), DesModel(m)
    for _ in range(3):
        g.step(1)
        if m.params.has_thermal_diffusion:
            assert h.lib.des_update_temperature(h.ctx) == 0
        for f in ("update_strain_rate", "compute_dvoldt", "compute_edvoldt", "update_stress", "nmd_stress",
                  "update_force", "update_velocity", "apply_vbcs", "update_mesh"):
            assert getattr(h.lib, "des_" + f)(h.ctx) == 0, f
        if m.params.rheol_type & abi.RH_ELASTIC:
            assert h.lib.des_rotate_stress(h.ctx) == 0
    _same(g.download(), h.download())


# element counts whose last block ends in a full wave, a part of one or a single element
@pytest.mark.parametrize("name,nelem", [("evp3", 300), ("evp3", 900), ("mat3", 1500), ("evp3", 2400), ("evp2", 250),
                                        ("mat2", 700), ("maxwell2", 1300)])
@pytest.mark.parametrize("mixed", [False, True])
def test_force_slots_stored_by_waves_and_by_lanes(name, nelem, mixed):
    from dynearthsol_amd.lib import DesModel
    m = SC.build(name, nelem=nelem)
    print(name, m.nelem, "elements:", m.nelem % 256, "in the last block", flush=True)
    out = []
    for mode in (0, 1):
        g = DesModel(m)
        g.set_launch_mode(mode)
        g.run(8, abi.DES_MIXED if mixed else abi.DES_FP64)
        out.append(g.download())
        g.close()
    _same(*out)
