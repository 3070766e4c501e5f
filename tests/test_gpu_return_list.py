"""Pass C's deferred Mohr-Coulomb returns with more listed than a wavefront
takes at once: at most 2048 wavefronts walk the list, each over segments of 64
elements, up to 64 segments a round.  200 k yielding elements leave some of
them over 64 entries (a second round over the entries); 8.4 M elements have
more segments than 64 rounds of 2048 (a second round over the segments).
Against the per-function step, which returns every element where it is
updated: the same operations on the same values, so bitwise equal."""
import math

import numpy as np
import pytest

import scenarios as SC
from dynearthsol_amd import abi

pytestmark = pytest.mark.gpu

FIELDS = ["stress", "plstrain", "delta_plstrain", "coord"]


def _yielding(m):
    """A horizontal stress beyond the yield surface: at least that at which
    sigma_z = n sigma_x - 2 c sqrt(n) for the cohesion c times 1.2."""
    P = m.params
    phi = math.radians(P.friction_angle0[0])
    n = (1 + math.sin(phi)) / (1 - math.sin(phi))
    st = m.stress0.copy()
    s1 = np.minimum(st[:, 2], -1e6)
    st[:, 2] = s1
    st[:, 0] = (s1 + 2 * 1.2 * P.cohesion0[0] * math.sqrt(n)) / n
    st[:, 1] = 0.5 * (st[:, 0] + s1)
    st[:, 3:] = 1e4          # never isotropic to the bit
    return st


@pytest.mark.parametrize("nelem,segments", [(200_000, None), (8_450_000, 64 * 2048)])
def test_long_return_lists_equal_returns_in_place(nelem, segments):
    from dynearthsol_amd.lib import DesModel
    m = SC.build("ep3", nelem=nelem)
    print(m.nelem, "elements", flush=True)
    assert segments is None or m.nelem > 64 * segments
    st = _yielding(m)
    out = []
    for fused in (False, True):
        g = DesModel(m)
        g.upload(stress=st)
        for _ in range(2):
            g.run(1) if fused else g.step(1)
        out.append(g.download(FIELDS))
        g.close()
        print("fused" if fused else "in place", "done", flush=True)
    a, b = out
    yields = int((a["delta_plstrain"] > 0).sum())
    print(yields, "elements yield", flush=True)
    assert yields > 64 * 2048        # some wavefront has more than 64
    for k in FIELDS:
        assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("precision", [abi.DES_FP64, abi.DES_MIXED])
def test_returns_come_and_go(mode, precision):
    """Steps in which nothing yields before and after steps in which all does:
    the lists fill and empty each time.  FP64 against the per-function step,
    mixed against the other launch mode."""
    from dynearthsol_amd.lib import DesModel
    m = SC.build("ep3", nelem=1500)
    print(m.nelem, "elements, launch mode", mode, "precision", precision, flush=True)
    high = _yielding(m)
    low = high.copy()
    low[:, :2] = high[:, 2:3]          # isotropic but for a little shear: far from the yield surface
    g, h = DesModel(m), DesModel(m)
    g.set_launch_mode(mode)
    h.set_launch_mode(1 - mode)
    for st, yields in ((low, False), (high, True), (low, False), (high, True)):
        for a in (g, h):
            a.upload(stress=st, plstrain=np.zeros(m.nelem), delta_plstrain=np.zeros(m.nelem))
        g.run(1, precision)
        h.step(1) if precision == abi.DES_FP64 else h.run(1, precision)
        a, b = g.download(FIELDS), h.download(FIELDS)
        assert bool((a["plstrain"] > 0).any()) == yields
        for k in FIELDS:
            assert np.array_equal(a[k], b[k]), k
