"""The torch functions whose gradient the library returns beside the value,
with a stand-in for the library: first derivatives, that a second one with
respect to the noise is refused, not left without the gradient's own
dependence on it, and that derivatives of the gradient with respect to other
parameters stay."""
import ctypes
import types

import numpy as np
import pytest
import torch

from genetic_amd import autodiff, gic

N = 4


class _Gen:
    """value = sum of w^2 over the mask (all cells for the variance)"""
    precision = gic.FLOAT64
    sizes = [N]

    def _quadratic(self, noise, mask, grad):
        w = np.ctypeslib.as_array((ctypes.c_double * N ** 3).from_address(noise))
        if grad is not None:
            np.ctypeslib.as_array((ctypes.c_double * N ** 3).from_address(grad))[:] = 2 * w * mask
        return float((w * w * mask).sum())

    def masked_displacement(self, noise, mask, grad=None):
        m = np.ctypeslib.as_array((ctypes.c_uint8 * N ** 3).from_address(mask))
        return self._quadratic(noise, m != 0, grad)

    def variance_gradient(self, noise, grad=None):
        return self._quadratic(noise[0], np.ones(N ** 3), grad and grad[0])


@pytest.fixture
def on_cpu(monkeypatch):
    monkeypatch.setattr(autodiff, "_check_levels", lambda *a: None)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(synchronize=lambda: None))


def _loss(name, w):
    gen, mask = _Gen(), torch.arange(N ** 3).view(N, N, N) % 3 == 0
    if name == "masked":
        return autodiff.MaskedSquares.apply(gen, w, mask), 2 * w.detach() * mask
    if name == "variance":
        return autodiff.filtered_variance(gen, w), 2 * w.detach()
    v = float((w.detach() ** 2).sum())
    return autodiff.sphere_loss(gen, w, mask, 0.5), 2 * w.detach() * mask + 2 * (v - 0.5) * 2 * w.detach()


@pytest.mark.parametrize("name", ["masked", "variance", "sphere_loss"])
def test_first_derivative_and_no_second(on_cpu, name):
    w = torch.randn((N, N, N), dtype=torch.float64, generator=torch.Generator().manual_seed(3)).requires_grad_(True)
    value, want = _loss(name, w)
    (g,) = torch.autograd.grad(value, w, retain_graph=True)
    torch.testing.assert_close(g, want, rtol=1e-13, atol=0)
    (g,) = torch.autograd.grad(value ** 2, w, create_graph=True)
    torch.testing.assert_close(g.detach(), 2 * value.detach() * want, rtol=1e-13, atol=0)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(g.sum(), w)
    # ... but the gradient's derivative with respect to a factor of the loss is its own
    (value, _), a = _loss(name, w), torch.tensor(3.0, dtype=torch.float64, requires_grad=True)
    (g,) = torch.autograd.grad(a * value ** 2, w, create_graph=True)
    (da,) = torch.autograd.grad((g * w.detach()).sum(), a)
    torch.testing.assert_close(da, (2 * value.detach() * want * w.detach()).sum(), rtol=1e-12, atol=0)
    with torch.no_grad():
        assert float(_loss(name, w)[0]) == float(value)
