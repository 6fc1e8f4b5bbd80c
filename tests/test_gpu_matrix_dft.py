"""Pressure solves on lengths with prime factors above 5 (products with the transform's matrices) and on odd
lengths of factors 3 and 5 (half-spectrum passes), against the oracle."""
import ctypes

import numpy as np
import pytest

from model_amd import configs, ids

pytestmark = pytest.mark.gpu

# rows n/2+1 of the matrices at the edges of 4-row steps and 16-row tiles, the longest length of the products
# and the first one past it, odd smooth lengths, and level counts that leave partial column tiles
SIZES = [(7, 22, 9), (11, 29, 12), (13, 31, 11), (31, 14, 18), (33, 62, 10), (46, 35, 7), (61, 63, 13), (97, 11, 24), (15, 21, 33),
         (25, 28, 10), (45, 33, 21), (509, 14, 5), (14, 509, 6), (521, 14, 5)]


@pytest.mark.parametrize("nx,ny,nz", SIZES)
@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32"])
def test_solve_against_oracle(nx, ny, nz, precision):
    """FP64 to 1e-12 of the pressure's largest value (sums of up to 509 terms, and the vertical solve's
    amplification of their rounding, against a factored transform); FP32 to 2e-4 (storage rounding of the
    divergence, a small difference of large terms in this random state, amplified by the solve)."""
    from model_amd.core import DynCore
    from oracle.pyoracle import Oracle
    c = configs.small_case(nx=nx, ny=ny, nz=nz, microphysics=0, amplitude=0.3)
    o, g = Oracle(c), DynCore(c, precision=precision)
    o.solve_pressure(ctypes.c_double(0.5))
    g.solve_pressure(ctypes.c_double(0.5))
    g.sync()
    a, b = g.get_field(ids.PI, 0), o.get_field(ids.PI)
    assert np.abs(a - b).max() <= (2e-4 if precision else 1e-12) * np.abs(b).max()


# the longest smooth lengths that take the products and the next ones that don't, along i and along j, one and
# both sides by products, and j lengths on either side of the fused j pass
SMOOTH = [(192, 12, 9), (200, 12, 9), (384, 12, 6), (400, 12, 6), (16, 192, 9), (16, 200, 9), (18, 112, 7), (18, 120, 7), (200, 100, 8)]


@pytest.mark.parametrize("nx,ny,nz", SMOOTH)
@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32"])
def test_smooth_lengths_against_oracle(nx, ny, nz, precision):
    test_solve_against_oracle(nx, ny, nz, precision)


@pytest.mark.parametrize("precision", [0, 1], ids=["fp64", "fp32"])
def test_ensemble_members_match_solo_runs_bitwise(precision):
    """A batch keeps slabs in one launch that a solo run takes through three: the same bits."""
    from model_amd.core import DynCore, Ensemble
    sizes = [(96, 104), (112, 96), (48, 48), (31, 29), (200, 100)]
    cases = [configs.small_case(nx=nx, ny=ny, nz=20, microphysics=0, amplitude=0.3, seed=n) for n, (nx, ny) in enumerate(sizes)]
    solo = [DynCore(c, precision=precision) for c in cases]
    members = [DynCore(c, precision=precision) for c in cases]
    e = Ensemble(members)
    e.step(2)
    e.sync()
    for s, m in zip(solo, members):
        s.step(2)
        s.sync()
        m.sync()
        for f in (ids.U, ids.V, ids.W, ids.TH):
            assert np.array_equal(s.get_field(f), m.get_field(f)), ids.FIELD_NAMES[f]
        assert np.array_equal(s.get_field(ids.PI, 0), m.get_field(ids.PI, 0))
    e.close()
