"""des_step past its tenth step against the entry points called one by one: the
time step that compute_dt gives there, the time and the step count that the
merged kernels keep, and geometry, masses and shape functions from their own
kernels (des_update_mesh shares des_step's).  Bitwise: the same operations on
the same values."""
import numpy as np
import pytest

import scenarios as SC
from dynearthsol_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["evp3", "dynmat3", "psevp2", "viscous2"])
def test_step_scalars_and_own_geometry_kernels(name):
    from dynearthsol_amd.lib import DesModel
    m = SC.build(name, nelem=1500)
    print(name, m.nelem, "elements", flush=True)
    g, h = DesModel(m), DesModel(m)
    dt, time = g.scalars()[0], 0.0
    for k in range(1, 13):
        g.step(1)
        if m.params.has_thermal_diffusion:
            h.call("update_temperature")
        for f in ("update_strain_rate", "compute_dvoldt", "compute_edvoldt", "update_stress", "nmd_stress",
                  "update_force", "update_velocity", "apply_vbcs", "update_mesh"):
            h.call(f)
        before = h.download(["volume", "mass", "tmass", "volume_n", "shpdx", "shpdz"])
        for f in ("compute_volume", "compute_mass", "compute_shape_fn"):
            h.call(f)
        after = h.download(list(before))
        for n in before:
            assert np.array_equal(before[n], after[n]), (k, n)
        if m.params.rheol_type & abi.RH_ELASTIC:
            h.call("rotate_stress")
        time += dt
        if k % 10 == 0:
            dt = h.compute_dt()
        assert g.scalars() == (dt, time, k)
    a, b = g.download(), h.download()
    for n in a:
        assert np.array_equal(a[n], b[n]), n
