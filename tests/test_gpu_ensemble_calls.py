"""Ensemble calls of odd and even lengths in any order, graph and eager: a step exchanges the members' current and
forecast buffers, so a graph recorded before an odd call must not serve after it."""
import numpy as np
import pytest

from model_amd import configs, ids

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32"])
def test_mixed_call_lengths_match_members_alone(precision):
    from model_amd.core import DynCore, Ensemble
    cases = [configs.vortex_in_shear(nx=n, ny=m, nz=20, seed_offset=50 + k) for k, (n, m) in enumerate([(24, 32), (40, 24)])]
    alone = [DynCore(c, precision=precision) for c in cases]
    members = [DynCore(c, precision=precision) for c in cases]
    ens = Ensemble(members)
    for n, graph in ((3, True), (2, True), (1, False), (4, True), (3, True), (3, True)):
        ens.step(n, graph=graph)
        ens.sync()
        for a, b in zip(alone, members):
            a.step(n)
            a.sync()
            for f in (ids.U, ids.V, ids.W, ids.TH):
                for role in (ids.ROLE_M, ids.ROLE_CUR, ids.ROLE_P):
                    assert np.array_equal(a.get_field(f, role), b.get_field(f, role)), (n, ids.FIELD_NAMES[f], role)
    ens.close()


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32"])
def test_members_stepped_on_their_own_between_calls(precision):
    """An odd number of steps of one member alone exchanges its buffers; the ensemble follows."""
    from model_amd.core import DynCore, Ensemble
    cases = [configs.vortex_in_shear(nx=n, ny=m, nz=20, seed_offset=60 + k) for k, (n, m) in enumerate([(24, 32), (40, 24), (32, 32)])]
    alone = [DynCore(c, precision=precision) for c in cases]
    members = [DynCore(c, precision=precision) for c in cases]
    ens = Ensemble(members)
    for turn, (n, graph) in enumerate(((2, True), (3, True), (1, False), (4, True))):
        ens.step(n, graph=graph)
        ens.sync()
        members[turn % 3].step(turn + 1)
        members[turn % 3].sync()
        for m, a in enumerate(alone):
            a.step(n + (turn + 1 if m == turn % 3 else 0))
            a.sync()
    ens.autotune()
    ens.step(2)
    ens.sync()
    for a, b in zip(alone, members):
        a.step(2)
        a.sync()
        for f in (ids.U, ids.V, ids.W, ids.TH):
            for role in (ids.ROLE_M, ids.ROLE_CUR):
                assert np.array_equal(a.get_field(f, role), b.get_field(f, role)), (ids.FIELD_NAMES[f], role)
    ens.close()
