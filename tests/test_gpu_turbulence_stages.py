"""Turbulent steps in the fused stage kernels (dyn_step) against the per-operator sequence, bit for bit: the
tendencies are added to the same expressions at the same places, inside the advected box by the stage kernels and
on the rows beside it by the boundary epilogue.  Packed rows and one wavefront per row, one wavefront and two per
column in the epilogue, sponge rows wider and narrower than the ghost rows, steps replayed from the graph and an
eager one after them."""
import numpy as np
import pytest

from model_amd import configs, ids

pytestmark = pytest.mark.gpu

ROLES = (ids.ROLE_M, ids.ROLE_CUR, ids.ROLE_P)


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32"])
@pytest.mark.parametrize("moist", [0, 1], ids=["dry", "moist"])
@pytest.mark.parametrize("nx,ny,nz", [(13, 16, 12), (40, 23, 21), (17, 37, 33), (14, 18, 57), (12, 16, 66), (22, 25, 67)])
def test_turbulent_steps_match_per_operator_bitwise(precision, moist, nx, ny, nz):
    from model_amd.core import DynCore
    c = configs.small_case(nx=nx, ny=ny, nz=nz, microphysics=moist, amplitude=0.2, rayleigh_level=max(1, nz - 3))
    ls = np.ones((c.nx, c.ny))
    ls[:, : c.ny // 3] = 0.0
    a, b = DynCore(c, precision=precision), DynCore(c, precision=precision)
    for g in (a, b):
        g.set_turbulence(True, ls)
    for n in (2, 4, 3):
        a.step_reference(n)
        b.step(n)
    a.sync()
    b.sync()
    assert (a.get_turbulence(0) > 0).any()  # the closure is active
    for f in ids.PROGNOSTIC if moist else (ids.U, ids.V, ids.W, ids.TH):
        for role in ROLES:
            x, y = a.get_field(f, role), b.get_field(f, role)
            assert np.isfinite(x).all()
            assert np.array_equal(x, y), (ids.FIELD_NAMES[f], role)
    for which in range(10 if moist else 6):
        assert np.array_equal(a.get_turbulence(which), b.get_turbulence(which)), which
    if moist:
        assert np.array_equal(a.get_field(ids.ACCRAIN), b.get_field(ids.ACCRAIN))
    a.close()
    b.close()
