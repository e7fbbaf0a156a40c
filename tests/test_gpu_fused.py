"""The fused transform passes at every grid size: the displacement map, its
transpose and the second-order displacements of one level against the same
in plain torch at 64 bits (a power-law spectrum, so that the reference needs
no table)."""
import math

import numpy as np
import pytest
import torch

from genetic_amd import gic

pytestmark = pytest.mark.gpu

BOX, NS = 50.0, 0.9
SIZES = [4, 8, 16, 32, 64, 128, 256, 512]
# rounding of a few transforms of 3 log2 n stages, relative to the field's rms
TOL = {32: 2e-6, 64: 1e-13}


def _gen(n, precision, lpt=1):
    g = gic.ICGenerator(precision=precision)
    g.set_cosmology(Om=0.3, Ol=0.7, s8=0.8, ns=NS, z=0.0)
    g.set_power_law(1.0)
    g.init_base_grid(BOX, n)
    g.set_lpt_order(lpt)
    return g


def _modes(n):
    """Signed wavenumbers per axis, those without +Nyquist, and delta / k^2 = table * w."""
    kmin = 2 * math.pi / BOX
    i = torch.arange(n, device="cuda")
    i = torch.where(i > n // 2, i - n, i)
    ks = [i.view(-1, 1, 1), i.view(1, -1, 1), torch.arange(n // 2 + 1, device="cuda").view(1, 1, -1)]
    ks = [k.double() * kmin for k in ks]
    k2 = sum(k ** 2 for k in ks)
    p = torch.where(k2 > 0, k2, 1.0) ** (NS / 2) * (n / BOX) ** 3
    root = torch.where(k2 > 0, p.sqrt(), 0.0)
    odd = [torch.where(k > kmin * (n // 2 - 0.5), 0.0, k) for k in ks]
    return ks, odd, root, torch.where(k2 > 0, 1 / torch.where(k2 > 0, k2, 1.0), 0.0)


def _fwd(x):
    return torch.fft.rfftn(x, norm="ortho")


def _inv(x, n):
    return torch.fft.irfftn(x, s=(n, n, n), norm="ortho")


def _near(got, want, precision, factor=1.0):
    scale = float((want.double() ** 2).mean().sqrt())
    err = float((got.double() - want).abs().max())
    assert err < factor * 50 * TOL[precision] * scale, (err, scale)


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("n", SIZES)
def test_displacement_and_transpose(n, precision):
    dt = torch.float32 if precision == 32 else torch.float64
    rng = torch.Generator(device="cuda").manual_seed(n)
    w = torch.randn((n, n, n), generator=rng, device="cuda", dtype=dt)
    bar = [torch.randn((n, n, n), generator=rng, device="cuda", dtype=dt) for _ in range(3)]
    psi = [torch.empty_like(w) for _ in range(3)]
    wbar = torch.empty_like(w)
    g = _gen(n, precision)
    torch.cuda.synchronize()
    g.displacement_forward([w.data_ptr()], [p.data_ptr() for p in psi])
    g.displacement_adjoint([b.data_ptr() for b in bar], [wbar.data_ptr()])
    _, odd, root, inv2 = _modes(n)
    x = w.double().requires_grad_(True)
    ref = [_inv(_fwd(x) * root * inv2 * (1j * k), n) for k in odd]
    for p, r in zip(psi, ref):
        _near(p, r.detach(), precision)
    _near(wbar, torch.autograd.grad(ref, x, [b.double() for b in bar])[0], precision)
    # the overdensity is left behind as the forward map's field
    delta = torch.from_numpy(g.field(gic.FIELD_OVERDENSITY, 0)).cuda()
    _near(delta, _inv(_fwd(w.double()) * root, n), precision)
    g.close()


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("n", SIZES)
def test_second_order(n, precision):
    rng = np.random.default_rng(n)
    w = rng.standard_normal((n, n, n)).astype(np.float32 if precision == 32 else np.float64)
    g = _gen(n, precision, lpt=2)
    g.set_field(0, w)
    g.apply_power_spectrum()
    g.zeldovich()
    ks, odd, root, inv2 = _modes(n)
    m = _fwd(torch.from_numpy(w).cuda().double()) * root * inv2

    def phi(a, b):
        return _inv(m * (ks[a] * ks[b] if a == b else odd[a] * odd[b]), n)

    S = sum(phi(a, a) * phi(b, b) - phi(a, b) ** 2 for a, b in ((0, 1), (0, 2), (1, 2)))
    s = _fwd(S)
    for a in range(3):
        _near(torch.from_numpy(g.field(1 + a, 0)).cuda(), _inv(m * (1j * odd[a]), n), precision)
        # S sums products of phi that cancel: a few times the error of one
        _near(torch.from_numpy(g.field(4 + a, 0)).cuda(), _inv(s * inv2 * (3.0 / 7.0) * (1j * odd[a]), n), precision, 10)
    g.close()


# 1024: what the grids above check cell by cell, on one component, without the
# fields' way through the host where there is another

@pytest.mark.parametrize("precision", [32, 64])
def test_displacement_and_transpose_at_1024(precision):
    n = 1024
    print("displacement at 1024, precision", precision, flush=True)
    dt = torch.float32 if precision == 32 else torch.float64
    rng = torch.Generator(device="cuda").manual_seed(n)
    w = torch.randn((n, n, n), generator=rng, device="cuda", dtype=dt)
    bar = [torch.randn((n, n, n), generator=rng, device="cuda", dtype=dt) for _ in range(3)]
    psi = [torch.empty_like(w) for _ in range(3)]
    wbar = torch.empty_like(w)
    g = _gen(n, precision)
    torch.cuda.synchronize()
    g.displacement_forward([w.data_ptr()], [p.data_ptr() for p in psi])
    g.displacement_adjoint([b.data_ptr() for b in bar], [wbar.data_ptr()])
    g.close()

    def dot(a, b):
        return sum(float((x[i].double() * y[i].double()).sum()) for x, y in zip(a, b) for i in range(n))

    size = (dot(psi, psi) * dot(bar, bar)) ** 0.5
    assert abs(dot(psi, bar) - dot([w], [wbar])) < (2e-5 if precision == 32 else 1e-12) * size
    del bar, wbar
    _, odd, root, inv2 = _modes(n)
    m = _fwd(w.double()) * root * inv2
    del root, inv2
    for a in (0, 2):
        _near(psi[a], _inv(m * (1j * odd[a]), n), precision)


@pytest.mark.parametrize("precision", [32, 64])
def test_second_order_at_1024(precision):
    n = 1024
    print("second order at 1024, precision", precision, flush=True)
    g = _gen(n, precision, lpt=2)
    g.set_seed(1024)
    g.zeldovich()
    real = np.float32 if precision == 32 else np.float64
    delta = torch.from_numpy(g.field(gic.FIELD_OVERDENSITY, 0, dtype=real)).cuda()
    got = torch.from_numpy(g.field(5, 0, dtype=real)).cuda()   # psi2_y
    g.close()
    ks, odd, _, inv2 = _modes(n)
    m = _fwd(delta.double()) * inv2
    del delta

    def phi(a, b):
        return _inv(m * (ks[a] * ks[b] if a == b else odd[a] * odd[b]), n)

    S = phi(0, 0)
    trace = S.clone()
    for a, first in ((1, True), (2, False)):
        p = phi(a, a)
        S = S * p if first else S + trace * p
        trace += p
    del trace, p
    for a, b in ((0, 1), (0, 2), (1, 2)):
        S -= phi(a, b) ** 2
    del m
    s = _fwd(S)
    del S
    _near(got, _inv(s * inv2 * (3.0 / 7.0) * (1j * odd[1]), n), precision, 10)
