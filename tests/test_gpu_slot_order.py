"""Every variant of pass E above 65,536 elements, where full waves store their
force contributions in slot order through LDS: staged and gathered node
records, the slots found by one-byte ranks and (force layout 2) by their full
positions.  Against the persistent launch, in which every lane stores its own:
the same operations on the same values, so bitwise equal and no tolerance."""
import numpy as np
import pytest

import scenarios as SC
from dynearthsol_amd import abi

pytestmark = pytest.mark.gpu

VARIANTS = {abi.DES_FP64: 3, abi.DES_MIXED: 2}


@pytest.mark.parametrize("name,nelem", [("mat3", 70000), ("evp2", 67000)])
@pytest.mark.parametrize("precision", sorted(VARIANTS))
def test_pass_e_variants_in_slot_order(name, nelem, precision):
    from dynearthsol_amd.lib import DesModel, set_force_layout
    m = SC.build(name, nelem=nelem)
    assert m.nelem > 65536 and m.nelem % 64, "the last wave has to be a partial one"
    print(name, m.nelem, "elements:", m.nelem % 256, "in the last block", flush=True)

    def run(launch, layout, variant):
        print("launch mode", launch, "layout", layout, "variant", variant, flush=True)
        set_force_layout(layout)
        try:
            g = DesModel(m)
            g.set_launch_mode(launch)
            g.set_tuning_all(precision, [0, 1 if precision == abi.DES_FP64 else 0, 0, variant, 0, 0])
            g.run(8, precision)
            out = g.download()
            g.close()
            return out
        finally:
            set_force_layout(0)

    ref = run(1, 0, 0)
    for layout in (0, 2):
        for variant in range(VARIANTS[precision]):
            got = run(0, layout, variant)
            for k in ref:
                assert np.array_equal(got[k], ref[k]), (layout, variant, k)
