"""FP32 pressure solves by matrix products: the one-slab form, the three launches with the 64-bit spectrum between
them, blocks of one, two and four column tiles along i and along j, and the lengths past the limits.  Every case
asserts the form it ran, from the timing records."""
import ctypes

import numpy as np
import pytest

from model_amd import configs, core, ids

pytestmark = pytest.mark.gpu

FIELDS = (ids.U, ids.V, ids.W, ids.TH)


def _records(g, run):
    g.timing(1)
    run()
    g.sync()
    buf = ctypes.create_string_buffer(1 << 16)
    g.timing_report(buf, len(buf))
    g.timing(0)
    return {line.split()[0] for line in buf.value.decode().splitlines()}


def _form(records):
    x = "dft" if {"p1_div_dft_x", "adj_dft_x"} & records else "fft"
    if "p2_ypass_dft" in records or "adj_ypass_dft" in records:
        return x, "slab"
    return x, "three" if "p2_dft_y" in records or "adj_dft_y" in records else "fft"


# lengths with a prime factor above 5 (tile edges, the longest length of the products and the next one) and odd ones
FACTORS = [(7, 22, 9, "dft", "slab"), (11, 29, 12, "dft", "slab"), (13, 31, 11, "dft", "slab"), (31, 14, 18, "dft", "slab"),
           (33, 62, 10, "dft", "slab"), (46, 35, 7, "dft", "slab"), (61, 63, 13, "dft", "slab"), (97, 11, 24, "dft", "slab"),
           (15, 21, 33, "dft", "slab"), (25, 28, 10, "dft", "slab"), (45, 33, 21, "dft", "slab"), (509, 14, 5, "dft", "slab"),
           (14, 509, 6, "dft", "slab"), (14, 509, 12, "dft", "three"), (20, 67, 64, "dft", "three"), (521, 14, 5, "fft", "fft")]
# two and four column tiles a block: along j, along i, both
TILES = [(257, 67, 52, "dft", "three"), (257, 131, 40, "dft", "three"), (61, 257, 66, "dft", "three"), (131, 131, 66, "dft", "three")]
# smooth lengths as deep as the FP32 rule asks for: the longest that take the products, and the next
SMOOTH = [(192, 12, 96, "dft", "slab"), (200, 12, 100, "fft", "fft"), (16, 192, 96, "dft", "three"), (16, 200, 100, "fft", "fft"),
          (18, 112, 56, "dft", "three"), (18, 120, 60, "fft", "fft"), (64, 48, 40, "dft", "slab")]


@pytest.mark.parametrize("nx,ny,nz,x,y", FACTORS + TILES + SMOOTH)
def test_moist_solve_against_oracle(nx, ny, nz, x, y):
    """To 2e-4 of the pressure's largest value: FP32 winds and an FP32 spectrum after the i pass, 6e-8 of each value; the
    horizontal cancellation in the longest waves (up to 509 points: 80) and the vertical one between the fluxes of
    neighbouring levels (five times the horizontal terms) raise that to 3e-5, factored transforms round more."""
    from oracle.pyoracle import Oracle
    c = configs.small_case(nx=nx, ny=ny, nz=nz, microphysics=1, amplitude=0.3)
    o, g = Oracle(c, variant="omp"), core.DynCore(c, precision=core.DYN_FP32)
    o.solve_pressure(ctypes.c_double(0.5))
    assert _form(_records(g, lambda: g.solve_pressure(ctypes.c_double(0.5)))) == (x, y)
    a, b = g.get_field(ids.PI, 0), o.get_field(ids.PI)
    assert np.abs(a - b).max() <= 2e-4 * np.abs(b).max()


@pytest.mark.parametrize("nx,ny,nz,jpass,form", [(18, 22, 11, 0, ("dft", "slab")), (18, 22, 11, 2, ("dft", "three")),
                                                 (18, 94, 50, 0, ("dft", "three"))])
def test_gradient_by_products(nx, ny, nz, jpass, form):
    """The transposed solve in FP32 by products (sweeps of the 64-bit spectrum in the three launches), against the FP64
    gradient: two steps' worth of FP32 rounding, with the solve's cancellations 1e-5, and the odd flipped upwind sign,
    within 1e-3 of the norm."""
    from model_amd.adjoint import backward, record, vorticity_weights
    c = configs.vortex_in_shear(nx=nx, ny=ny, nz=nz)
    Wu, Wv = vorticity_weights(c)
    out = []
    for precision in (0, core.DYN_FP32):
        g = core.DynCore(c, precision=precision)
        g.tune_set(core.DYN_TUNE_PRESSURE_JPASS, jpass)
        record(g, 2, 2)
        names = _records(g, lambda: out.append(backward(g, [Wu, Wv, None, None])))
        if precision == core.DYN_FP32:
            assert _form(names) == form
        g.close()
    for f, a, b in zip(FIELDS, *out):
        assert np.isfinite(b).all()
        assert np.linalg.norm(a - b) <= 1e-3 * np.linalg.norm(a), ids.FIELD_NAMES[f]


def test_batch_keeps_slabs_that_solo_runs_split_bitwise():
    """A batch solves in one launch what a member with 24 tile pairs takes through three on its own: the same bits."""
    sizes = [((20, 67), ("dft", "three")), ((48, 48), ("dft", "slab")), ((62, 61), ("dft", "slab"))]
    cases = [configs.small_case(nx=nx, ny=ny, nz=64, microphysics=0, amplitude=0.3, seed=n) for n, ((nx, ny), _) in enumerate(sizes)]
    solo = [core.DynCore(c, precision=core.DYN_FP32) for c in cases]
    members = [core.DynCore(c, precision=core.DYN_FP32) for c in cases]
    for s, (_, form) in zip(solo, sizes):
        assert _form(_records(s, lambda: s.step_fused(2))) == form
    e = core.Ensemble(members)
    assert "ens_p2_ypass" in _records(members[0], lambda: e.step(2, graph=False))
    e.sync()
    for s, m in zip(solo, members):
        m.sync()
        for f in FIELDS:
            assert np.array_equal(s.get_field(f), m.get_field(f)), ids.FIELD_NAMES[f]
        assert np.array_equal(s.get_field(ids.PI, 0), m.get_field(ids.PI, 0))
    e.close()
