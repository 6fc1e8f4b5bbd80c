"""Calls of odd and even lengths in any order on the steps whose graph covers two steps: steps with the turbulence
closure, and level counts the fused kernels do not take.  A step exchanges the current and the forecast buffer, so a
graph recorded before an odd call must not serve after it."""
import numpy as np
import pytest

from model_amd import configs, ids

pytestmark = pytest.mark.gpu

CALLS = (3, 2, 1, 4, 3, 3, 2)


def _same(a, b, moist):
    for g in (a, b):
        g.sync()
    for f in ids.PROGNOSTIC if moist else (ids.U, ids.V, ids.W, ids.TH):
        for role in (ids.ROLE_M, ids.ROLE_CUR, ids.ROLE_P):
            x, y = a.get_field(f, role), b.get_field(f, role)
            assert np.isfinite(x).all()
            assert np.array_equal(x, y), (ids.FIELD_NAMES[f], role)


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32"])
@pytest.mark.parametrize("moist", [0, 1], ids=["dry", "moist"])
@pytest.mark.parametrize("nz,turbulence", [(12, True), (65, True), (65, False)])
def test_mixed_call_lengths_match_per_operator_bitwise(precision, moist, nz, turbulence):
    from model_amd.core import DynCore
    c = configs.small_case(nx=14, ny=16, nz=nz, microphysics=moist, amplitude=0.2, rayleigh_level=nz - 3)
    a, b = DynCore(c, precision=precision), DynCore(c, precision=precision)
    if turbulence:
        for g in (a, b):
            g.set_turbulence(True)
    for n in CALLS:
        a.step_reference(n)
        b.step(n)
        _same(a, b, moist)
    a.close()
    b.close()
