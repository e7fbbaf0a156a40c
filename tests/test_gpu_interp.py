"""The coarse-to-fine interpolation and its transpose at the geometries where
their windows can go wrong: refinements 1, 2, 3 and 8, zooms that touch or
cross the box's edge, a zoom as large as the box (its stencils fall on a
coarse cell twice), nested zooms whose stencils clamp, and grids smaller than
a block's rows -- the forward map against the oracle's level combination and
the transpose against the forward map."""
import os

import numpy as np
import pytest
import torch

import pyoracle as po
from genetic_amd import gic

pytestmark = pytest.mark.gpu

EH_TABLE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..", "genetic_amd", "data", "eh_nowiggle_512.dat")
COSMO = dict(Om=0.31, Ol=0.69, hubble=0.677, s8=0.81, ns=0.967, z=99)

LEVELS = {
    "ratio1": [(50.0, 32), (5, 9, 2, 2, 16)],
    "ratio3": [(50.0, 32), (3, 7, 11, 3, 32)],
    "ratio8": [(50.0, 16), (2, 5, 9, 4, 32)],
    "box edge": [(50.0, 32), (0, 24, 23, 4, 16)],
    "across the edge": [(50.0, 32), (26, 30, 5, 4, 16)],
    "whole box": [(50.0, 16), (0, 0, 0, 1, 32)],
    "nested, clamped": [(50.0, 32), (8, 8, 8, 2, 32), (0, 16, 7, 2, 32)],
    "tiny": [(50.0, 8), (2, 2, 2, 2, 4)],
}


def _gen(levels, precision):
    g = gic.ICGenerator(precision=precision)
    g.set_cosmology(**COSMO)
    g.set_camb(EH_TABLE)
    g.init_base_grid(*levels[0])
    for z in levels[1:]:
        g.init_zoom_grid_with_origin_at(*z)
    return g


@pytest.mark.parametrize("name", sorted(LEVELS))
def test_level_combination_matches_the_oracle(name):
    levels = LEVELS[name]
    g = _gen(levels, gic.FLOAT64)
    o = po.OracleIC()
    o.set_cosmology(**COSMO)
    o.set_camb(*po.read_camb(EH_TABLE))
    o.init_base_grid(*levels[0])
    for z in levels[1:]:
        o.init_zoom_grid_at(*z)
    for x in (g, o):
        (x.set_seed if x is g else x.seed)(31)
        x.draw()
        x.apply_power_spectrum()
        x.zeldovich()
    for l in range(len(levels)):
        for which in range(4):
            a, b = g.field(which, l), o.field(which, l)
            np.testing.assert_allclose(a, b, rtol=0, atol=1e-10 * np.abs(b).max(), err_msg="%d %d" % (l, which))
    g.close()


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("name", sorted(LEVELS))
def test_transpose(name, precision):
    """<Psi w, g> = <w, Psi^T g> to rounding over sums of the fields' length."""
    levels = LEVELS[name]
    gen = _gen(levels, precision)
    dt = torch.float32 if precision == 32 else torch.float64
    rng = np.random.default_rng(len(name))
    draw = lambda n: torch.tensor(rng.standard_normal((n, n, n)), dtype=dt, device="cuda")
    w = [draw(n) for n in gen.sizes]
    bar = [draw(n) for n in gen.sizes for _ in range(3)]
    psi = [torch.empty_like(w[l]) for l in range(len(w)) for _ in range(3)]
    wbar = [torch.empty_like(t) for t in w]
    torch.cuda.synchronize()
    gen.displacement_forward([t.data_ptr() for t in w], [t.data_ptr() for t in psi])
    gen.displacement_adjoint([t.data_ptr() for t in bar], [t.data_ptr() for t in wbar])
    dots = lambda a, b: sum(float((x.double() * y.double()).sum()) for x, y in zip(a, b))
    size = sum(float((x.double() ** 2).sum()) for x in psi) ** 0.5 * sum(float((x.double() ** 2).sum()) for x in bar) ** 0.5
    assert abs(dots(psi, bar) - dots(w, wbar)) < (2e-5 if precision == 32 else 1e-12) * size
    gen.close()
