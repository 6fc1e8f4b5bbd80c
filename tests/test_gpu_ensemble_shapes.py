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


def test_shape_in_force_can_be_set_again():
    """The shape a batch starts with is one that a caller can read and set; the autotuner leaves each kernel that shape
    or the one it reports."""
    ens = Ensemble([DynCore(c, precision=DYN_FP32) for c in _cases()])
    own = ens.shape
    ens.set_shape(own)
    best = ens.autotune()
    now = ens.shape
    for k in (0, 2):
        assert now[k:k + 2] in (own[k:k + 2], best[k:k + 2])
    ens.set_shape(own)
    assert ens.shape == own
    ens.close()


@pytest.mark.parametrize("precision", [0, DYN_FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("nz,shape,refused", [(20, (3, 5, 25, 2), (26, 8, 4, 8)), (40, (12, 13, 6, 14), (13, 8, 4, 8)),
                                              (56, (9, 16, 5, 3), (4, 8, 10, 8)), (57, (2, 9, 8, 7), (6, 8, 4, 8))])
def test_any_shape_gives_the_same_bits(precision, nz, shape, refused):
    """Rows of packed levels up to 512 lanes (nz 20, 40, 56), and one wavefront per row (nz 57); one row more, and rows
    the instances do not have, are refused and leave the shape as it was."""
    from model_amd.core import DynError
    cases = _cases(nz)[:2]
    alone = [DynCore(c, precision=precision) for c in cases]
    members = [DynCore(c, precision=precision) for c in cases]
    ens = Ensemble(members)
    ens.set_shape(shape)
    for bad in (refused, (1, 8, 4, 8), (4, 1, 4, 8), (4, 8, 4, 513)):
        with pytest.raises(DynError):
            ens.set_shape(bad)
        assert ens.shape == shape
    ens.step(2)
    ens.sync()
    for a in alone:
        a.step(2)
    _same(alone, members)
    ens.close()
