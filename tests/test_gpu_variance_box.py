"""The variance operator on the box of the flagged cells: sets of cells whose
box wraps, reaches the largest box that takes the cut transforms or just
passes it, against the oracle's variance of the same field; the gradient
against the value, which is quadratic in the field."""
import os

import numpy as np
import pytest
import torch

import pyoracle as po
from genetic_amd import gic
from helpers import golden

pytestmark = pytest.mark.gpu

N, BOX, SCALE = 16, 50.0, 12.5
COSMO = dict(Om=0.31, Ol=0.69, hubble=0.677, s8=0.81, ns=0.967, z=99)


def _cells(name):
    x, y, z = np.meshgrid(*[np.arange(N)] * 3, indexing="ij")
    r2 = sum(np.minimum(q, N - q) ** 2 for q in (x, y, z))
    m = {"pair": (x == 5) & (y == 9) & (z <= 1),
         "corner_ball": r2 <= 10,
         "far_apart": (x % 15 == 3) & (y % 7 == 1) & (z % 15 == 0),
         "half": x >= N // 2,
         "past_half": (x >= N // 2 - 1) & (y < 3),
         "thin_x": (x == 15) & (y != 4),
         "all": x >= 0}[name]
    return np.flatnonzero(m.ravel()).astype(np.uint64)


def _gpu(levels, precision):
    ic = gic.ICGenerator(precision=precision)
    ic.set_cosmology(**COSMO)
    ic.set_camb(golden("camb_transfer_kmax40_z0.dat"))
    ic.init_base_grid(*levels[0])
    for z in levels[1:]:
        ic.init_zoom_grid_with_origin_at(*z)
    return ic


def _oracle(levels):
    o = po.OracleIC()
    o.set_cosmology(**COSMO)
    tab, _ = po.read_camb(golden("camb_transfer_kmax40_z0.dat"))
    o.set_camb(tab, _)
    o.init_base_grid(*levels[0])
    for z in levels[1:]:
        o.init_zoom_grid_at(*z)
    return o


@pytest.mark.parametrize("level", [0, 1])
@pytest.mark.parametrize("name", ["pair", "corner_ball", "far_apart", "half", "past_half", "thin_x", "all"])
def test_variance_of_cells_matches_oracle(name, level):
    print("variance of", name, "level", level, flush=True)
    levels = [(BOX, N)] + ([(4, 4, 4, 2, N)] if level else [])
    ic, o = _gpu(levels, gic.FLOAT64), _oracle(levels)
    for g in (ic, o):
        (g.set_seed if g is ic else g.seed)(77)
        g.set_flags(level, _cells(name))
    ic.set_variance_filter_scale(SCALE)
    o.set_variance_scale(SCALE)
    want = o.calculate("variance")
    # FP64 throughout, other orders of the sums: 12 transforms of 4096 values
    assert abs(ic.calculate("variance") - want) <= 1e-11 * abs(want)


@pytest.mark.parametrize("precision,tol", [(gic.FLOAT64, 1e-11), (gic.FLOAT32, 2e-5)])
@pytest.mark.parametrize("name", ["pair", "corner_ball", "half", "past_half", "thin_x"])
def test_gradient_belongs_to_the_value(name, precision, tol):
    """V(w + d) - V(w - d) = 2 <dV/dw, d> exactly, V being quadratic."""
    print("variance gradient", name, precision, flush=True)
    ic = _gpu([(BOX, N)], precision)
    ic.set_flags(0, _cells(name))
    ic.set_variance_filter_scale(SCALE)
    rng = np.random.default_rng(3)
    dt = torch.float64 if precision == gic.FLOAT64 else torch.float32
    w, d = (torch.tensor(rng.standard_normal((N, N, N)), dtype=dt, device="cuda") for _ in range(2))
    grad = torch.empty_like(w)

    def value(t, g=None):
        t = t.contiguous()
        torch.cuda.synchronize()
        return ic.variance_gradient([t.data_ptr()], None if g is None else [g.data_ptr()])

    v0 = value(w, grad)
    vp, vm = value(w + d), value(w - d)
    assert abs((vp - vm) - 2 * float((grad.double() * d.double()).sum())) <= tol * (vp + vm + v0)
    # and V(w) = <dV/dw, w> / 2
    assert abs(v0 - 0.5 * float((grad.double() * w.double()).sum())) <= tol * v0


def _many_cells(name, n):
    x, y, z = np.meshgrid(*[np.arange(n)] * 3, indexing="ij")
    dx, dy, dz = (np.minimum((q - c) % n, (c - q) % n) for q, c in ((x, 1), (y, 30), (z, 60)))
    m = {"ellipsoid": (dx / 15) ** 2 + (dy / 20) ** 2 + (dz / 20) ** 2 <= 1,
         "wrapped slab": ((x >= 50) | (x < 10)) & (y != 4) & (z > 2),
         "planes apart": (x % 16 == 3) & (y < 50),
         "half": (x >= 32) & (y % 5 == 2),
         "past half": x >= 31}[name]
    return np.flatnonzero(m.ravel()).astype(np.uint64)


@pytest.mark.parametrize("name", ["ellipsoid", "wrapped slab", "planes apart", "half", "past half"])
def test_variance_of_many_cells_matches_oracle(name):
    """Sets whose axes are marked on the device, and two that span too many
    planes."""
    print("variance of many cells", name, flush=True)
    n, cells = 64, _many_cells(name, 64)
    assert cells.size > 16384 or name == "planes apart"
    ic, o = _gpu([(BOX, n)], gic.FLOAT64), _oracle([(BOX, n)])
    for g in (ic, o):
        (g.set_seed if g is ic else g.seed)(77)
        g.set_flags(0, cells)
    ic.set_variance_filter_scale(SCALE)
    o.set_variance_scale(SCALE)
    want = o.calculate("variance")
    assert abs(ic.calculate("variance") - want) <= 1e-11 * abs(want)


@pytest.mark.parametrize("n", [64, 128, 256])
def test_cut_transforms_of_larger_grids(n):
    """A wrapping ball's variance and gradient: in FP64 the gradient belongs to
    the value (V is quadratic), in FP32 both are the FP64 ones to float
    rounding."""
    print("variance box at", n, flush=True)
    q = np.minimum(np.arange(n), n - np.arange(n))
    r2 = q[:, None, None] ** 2 + q[None, :, None] ** 2 + q[None, None, :] ** 2
    cells = np.flatnonzero((r2 <= (n // 10) ** 2).ravel()).astype(np.uint64)
    rng = torch.Generator(device="cuda").manual_seed(n)
    w, d = (torch.randn((n, n, n), generator=rng, device="cuda", dtype=torch.float64) for _ in range(2))
    got = {}
    for precision, dt in ((gic.FLOAT64, torch.float64), (gic.FLOAT32, torch.float32)):
        ic = _gpu([(BOX, n)], precision)
        ic.set_flags(0, cells)
        ic.set_variance_filter_scale(BOX / n * 4)

        def value(t, g=None):
            t = t.to(dt)
            torch.cuda.synchronize()
            return ic.variance_gradient([t.data_ptr()], None if g is None else [g.data_ptr()])

        grad = torch.empty_like(w, dtype=dt)
        got[precision] = value(w, grad), grad.double()
        if precision == gic.FLOAT64:
            vp, vm = value(w + d), value(w - d)
            assert abs((vp - vm) - 2 * float((grad * d).sum())) <= 1e-11 * (vp + vm)
        ic.close()
    (v, g), (v32, g32) = got[gic.FLOAT64], got[gic.FLOAT32]
    assert abs(v32 - v) <= 2e-5 * v
    assert float((g32 - g).norm()) <= 2e-5 * float(g.norm())
