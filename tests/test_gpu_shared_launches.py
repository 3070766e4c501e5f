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


# above 65,536 elements the waves store (batches count all their models), below
# it the lanes; the last block of each model ends in a full wave or in a part
# of one
@pytest.mark.parametrize("name,nelem", [("evp3", 900), ("evp2", 700), ("evp3", 66000), ("mat3", 70000), ("evp2", 66000),
                                        ("mat2", 68000), ("maxwell3", 68500)])
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


@pytest.mark.parametrize("mixed", [False, True])
def test_force_slots_of_a_batch_with_part_blocks(mixed):
    from dynearthsol_amd.lib import DesBatch
    models = [SC.build("evp3", nelem=n) for n in (66000, 300, 900, 1500)]
    print([m.nelem % 256 for m in models], "in the last blocks", flush=True)
    out = []
    for mode in (0, 1):
        b = DesBatch(models)
        b.set_launch_mode(mode)
        b.run(8, abi.DES_MIXED if mixed else abi.DES_FP64)
        out.append([b.download(k) for k in range(len(models))])
        b.close()
    for a, c in zip(*out):
        _same(a, c)
