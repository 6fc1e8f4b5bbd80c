"""The launch parameters in force: what the size rules choose while the knobs are unset, against what the timing
records of a step name, and the values set."""
import ctypes

import pytest

from model_amd import configs, core
from model_amd.core import DynCore, DynError

pytestmark = pytest.mark.gpu

SHAPE = (core.DYN_TUNE_MOMENTUM_TJ, core.DYN_TUNE_MOMENTUM_TI, core.DYN_TUNE_SCALAR_TJ, core.DYN_TUNE_SCALAR_TI)


def _records(g):
    g.timing(1)
    g.step_fused(1)
    g.sync()
    buf = ctypes.create_string_buffer(1 << 16)
    g.timing_report(buf, len(buf))
    g.timing(0)
    return {line.split()[0]: line.split() for line in buf.value.decode().splitlines()}


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32"])
@pytest.mark.parametrize("nx,ny,nz,one", [(24, 24, 20, True), (200, 200, 40, False), (160, 120, 60, False), (96, 96, 80, False)])
def test_what_is_in_force_is_what_runs(precision, nx, ny, nz, one):
    g = DynCore(configs.supercell(nx=nx, ny=ny, nz=nz), precision=precision)
    assert ("adv_stage" in _records(g)) == one
    streams = g.tune_in_force(core.DYN_TUNE_STAGE_STREAMS)
    assert streams == 1 if one else streams > 1
    for p in SHAPE:
        assert g.tune_in_force(p) >= 2
    for p, v in zip(SHAPE, (2, 9, 2, 7)):  # set: in force, and the stage in two launches
        g.tune_set(p, v)
        assert g.tune_in_force(p) == g.tune_get(p) == v
    assert "adv_stage" not in _records(g)
    for p in SHAPE:
        g.tune_set(p, 0)
    assert ("adv_stage" in _records(g)) == one
    for v in (1, 2, 3, 4):
        g.tune_set(core.DYN_TUNE_STAGE_STREAMS, v)
        assert g.tune_in_force(core.DYN_TUNE_STAGE_STREAMS) == v
    with pytest.raises(DynError):
        g.tune_in_force(core.DYN_TUNE_STAGE_STREAMS + 1)
    g.close()


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32"])
def test_j_pass_in_force(precision):
    """Three launches where the timing records show them: lengths by products with more tiles than a slab takes, and the
    full complex spectrum of an i length that is too long for them."""
    for nx, ny, nz in ((96, 96, 48), (32, 32, 20), (521, 14, 20)):
        g = DynCore(configs.supercell(nx=nx, ny=ny, nz=nz), precision=precision)
        assert ("p3_thomas" in _records(g)) == (g.tune_in_force(core.DYN_TUNE_PRESSURE_JPASS) == 2)
        g.close()
