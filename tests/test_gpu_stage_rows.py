"""The stage kernels' packed rows (levels of a block's rows one after another over its lanes) against the
per-operator kernels: the level counts where wavefront edges fall at a column's ends, at the lid's source
levels and inside it, and the counts beside those that take one wavefront per row."""
import numpy as np
import pytest

from model_amd import configs, ids

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32"])
@pytest.mark.parametrize("nx,ny,nz", [(13, 16, 5), (9, 37, 12), (40, 23, 21), (17, 16, 32), (21, 30, 33), (31, 19, 56), (14, 18, 57),
                                      (12, 16, 66), (22, 25, 67), (11, 26, 127), (200, 61, 21)])
def test_packed_rows_match_per_operator_bitwise(precision, nx, ny, nz):
    """Same expression trees in both forms, so every buffer of every role agrees to the last bit."""
    from model_amd.core import DynCore
    c = configs.small_case(nx=nx, ny=ny, nz=nz, microphysics=1, amplitude=0.5, rayleigh_level=max(1, nz - 3))
    a, b = DynCore(c, precision=precision), DynCore(c, precision=precision)
    a.step_reference(3)
    b.step_fused(3)
    a.sync()
    b.sync()
    for f in ids.PROGNOSTIC:
        for role in (ids.ROLE_M, ids.ROLE_CUR, ids.ROLE_P):
            assert np.array_equal(a.get_field(f, role), b.get_field(f, role)), (ids.FIELD_NAMES[f], role)
    assert np.array_equal(a.get_field(ids.VT, 0), b.get_field(ids.VT, 0))
    assert np.array_equal(a.get_field(ids.ACCRAIN), b.get_field(ids.ACCRAIN))


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32"])
@pytest.mark.parametrize("moist", [0, 1], ids=["dry", "moist"])
@pytest.mark.parametrize("nx,ny,nz", [(13, 16, 5), (9, 37, 12), (31, 30, 33), (48, 48, 40), (14, 18, 57), (16, 16, 64), (12, 16, 66)])
def test_one_launch_stages_match_two_streams_bitwise(precision, moist, nx, ny, nz):
    """Small grids run both halves of a stage, and the boundary updates after it, in one launch each; asked for
    two streams they run the two halves apart.  The same tiles, so the same bits, from graphs of each length and
    eagerly."""
    from model_amd.core import DynCore
    c = configs.small_case(nx=nx, ny=ny, nz=nz, microphysics=moist, amplitude=0.5, rayleigh_level=max(1, nz - 3))
    a, b = DynCore(c, precision=precision), DynCore(c, precision=precision)
    b.tune_set(5, 4)
    for n in (7, 1, 6, 2):
        a.step(n)
        b.step(n)
    a.sync()
    b.sync()
    for f in ids.PROGNOSTIC if moist else (ids.U, ids.V, ids.W, ids.TH):
        assert np.isfinite(a.get_field(f, ids.ROLE_CUR)).all()
        for role in (ids.ROLE_M, ids.ROLE_CUR):
            assert np.array_equal(a.get_field(f, role), b.get_field(f, role)), (ids.FIELD_NAMES[f], role)
    assert np.array_equal(a.get_field(ids.PI, 0), b.get_field(ids.PI, 0))
