"""Launch shapes of an ensemble's stage kernels: the autotuner and the shapes a caller sets."""
import numpy as np
import pytest

from model_amd import configs, ids
from model_amd.core import DYN_FP32, DynCore, Ensemble

pytestmark = pytest.mark.gpu

SIZES = [(48, 64), (64, 48), (80, 80)]


def _cases(nz=20):
    return [configs.vortex_in_shear(nx=n, ny=m, nz=nz, seed_offset=70 + k) for k, (n, m) in enumerate(SIZES)]


def _same(alone, members):
    for a, b in zip(alone, members):
        a.sync()
        for f in (ids.U, ids.V, ids.W, ids.TH):
            for role in (ids.ROLE_M, ids.ROLE_CUR):
                assert np.array_equal(a.get_field(f, role), b.get_field(f, role)), (ids.FIELD_NAMES[f], role)


@pytest.mark.parametrize("precision", [0, DYN_FP32], ids=["fp64", "fp32"])
def test_autotune_behind_queued_steps(precision):
    """The autotuner rewrites the tables that queued steps read: it waits for them."""
    cases = _cases()
    alone = [DynCore(c, precision=precision) for c in cases]
    members = [DynCore(c, precision=precision) for c in cases]
    ens = Ensemble(members)
    ens.step(40)
    ens.autotune()
    ens.step(3)
    ens.sync()
    for a in alone:
        a.step(43)
    _same(alone, members)
    ens.close()
