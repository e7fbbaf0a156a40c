"""The sum of |psi|^2 over a mask's cells and its gradient, formed on the box
around the mask, against the full displacement fields multiplied by the mask
as weights (which take the general route)."""
import os

import pytest
import torch

from genetic_amd import autodiff, gic

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
EH_TABLE = os.path.join(HERE, "..", "genetic_amd", "data", "eh_nowiggle_512.dat")


def _gen(n, precision):
    g = gic.ICGenerator(precision=precision)
    g.set_cosmology(Om=0.31, Ol=0.69, hubble=0.677, s8=0.81, ns=0.967, z=99)
    g.set_camb(EH_TABLE)
    g.init_base_grid(50.0, n)
    g.set_flags(0, [5, 6, n * n + 5])
    g.set_variance_filter_scale(25.0)
    return g


def _mask(name, n):
    q = torch.arange(n, device="cuda")
    x, y, z = torch.meshgrid(q, q, q, indexing="ij")
    d = lambda v: torch.minimum(v, n - v)
    return {"corner_ball": d(x) ** 2 + d(y) ** 2 + d(z) ** 2 <= (n // 4) ** 2,
            "one_cell": (x == n - 1) & (y == 0) & (z == n - 1),
            "last_plane": x == n - 1,
            "two_gaps": (x % (n - 1) == 1) & (y % 3 == 0) & (z == 2),
            "all": x >= 0,
            "none": x < 0}[name]


# FP64: the same sums in other orders.  FP32: float rounding of the transforms,
# as in the other displacement tests.
@pytest.mark.parametrize("precision,tol", [(gic.FLOAT64, 1e-12), (gic.FLOAT32, 1e-5)])
@pytest.mark.parametrize("n", [8, 64, 128, 256])
@pytest.mark.parametrize("name", ["corner_ball", "one_cell", "last_plane", "two_gaps", "all", "none"])
def test_loss_of_a_mask_matches_weights(name, n, precision, tol):
    print("masked displacement", name, n, precision, flush=True)
    g = _gen(n, precision)
    dt = torch.float64 if precision == gic.FLOAT64 else torch.float32
    w = torch.randn((n, n, n), dtype=torch.float64, generator=torch.Generator().manual_seed(n)).to("cuda", dt)
    mask = _mask(name, n)
    out = []
    for m in (mask, mask.to(dt)):
        x = w.clone().requires_grad_(True)
        loss = autodiff.sphere_loss(g, x, m, 0.0)
        loss.backward()
        out.append((float(loss.detach()), x.grad.double()))
    (a, ga), (b, gb) = out
    assert abs(a - b) <= tol * abs(b)
    assert float((ga - gb).norm()) <= tol * float(gb.norm())


def test_value_without_gradient_and_refusals():
    print("masked displacement: value alone, refusals", flush=True)
    g = _gen(16, gic.FLOAT64)
    w = torch.randn((16, 16, 16), dtype=torch.float64, device="cuda")
    mask = _mask("corner_ball", 16)
    torch.cuda.synchronize()
    grad = torch.empty_like(w)
    v = g.masked_displacement(w.data_ptr(), mask.data_ptr())
    odd = torch.cat([mask.new_zeros(1), mask.ravel()])[1:]   # not aligned to words
    torch.cuda.synchronize()
    assert v == g.masked_displacement(w.data_ptr(), odd.data_ptr())
    assert v == g.masked_displacement(w.data_ptr(), mask.data_ptr(), grad.data_ptr())
    with pytest.raises(gic.GICError):
        g.masked_displacement(0, mask.data_ptr())
    with pytest.raises(ValueError):
        autodiff.sphere_loss(g, w.float(), mask, 0.0)
    g = _gen(16, gic.FLOAT64)
    g.init_zoom_grid_with_origin_at(4, 4, 4, 2, 16)
    with pytest.raises(gic.GICError):
        g.masked_displacement(w.data_ptr(), mask.data_ptr())
