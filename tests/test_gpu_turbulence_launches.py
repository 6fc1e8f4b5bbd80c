"""Steps with the turbulence closure in every launch form of a stage (both halves in one launch, and two launches on
one stream and on two with each fork), against the per-operator sequence, bit for bit.  The timing records say which
form ran."""
import ctypes

import numpy as np
import pytest

from model_amd import configs, core, ids

pytestmark = pytest.mark.gpu


def _records(g, run):
    g.timing(1)
    run()
    g.sync()
    buf = ctypes.create_string_buffer(1 << 16)
    g.timing_report(buf, len(buf))
    g.timing(0)
    return {line.split()[0] for line in buf.value.decode().splitlines()}


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32"])
@pytest.mark.parametrize("moist", [0, 1], ids=["dry", "moist"])
@pytest.mark.parametrize("nx,ny,nz,streams,one", [(40, 23, 21, 0, True), (40, 23, 21, 1, False), (40, 23, 21, 2, False),
                                                  (40, 23, 21, 3, False), (40, 23, 21, 4, False), (14, 18, 57, 2, False),
                                                  (22, 25, 67, 3, False), (150, 126, 50, 0, False)])
def test_launch_forms_match_per_operator_bitwise(precision, moist, nx, ny, nz, streams, one):
    c = configs.small_case(nx=nx, ny=ny, nz=nz, microphysics=moist, amplitude=0.2, rayleigh_level=nz - 3)
    ls = np.ones((c.nx, c.ny))
    ls[:, : c.ny // 3] = 0.0
    a, b = core.DynCore(c, precision=precision), core.DynCore(c, precision=precision)
    for g in (a, b):
        g.set_turbulence(True, ls)
    b.tune_set(core.DYN_TUNE_STAGE_STREAMS, streams)
    assert ("adv_stage" in _records(b, lambda: b.step(1))) == one  # a single step runs eagerly
    b.step(4)
    a.step_reference(5)
    a.sync()
    b.sync()
    assert (a.get_turbulence(0) > 0).any()  # the closure is active
    for f in ids.PROGNOSTIC if moist else (ids.U, ids.V, ids.W, ids.TH):
        for role in (ids.ROLE_M, ids.ROLE_CUR, ids.ROLE_P):
            x, y = a.get_field(f, role), b.get_field(f, role)
            assert np.isfinite(x).all()
            assert np.array_equal(x, y), (ids.FIELD_NAMES[f], role)
    a.close()
    b.close()
