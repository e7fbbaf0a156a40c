"""The Gram matrices of batched realisations, formed in blocks of 16
covectors: one block, a full one, and one covector more, against the
one-at-a-time path."""
import numpy as np
import pytest
import torch

from genetic_amd import gic
from helpers import cosmology_from_paramfile, golden, select_sphere_cells

pytestmark = pytest.mark.gpu

BOX, N = 50.0, 32


@pytest.mark.parametrize("precision,tol", [(gic.FLOAT64, 1e-9), (gic.FLOAT32, 2e-4)])   # as the batch tests'
@pytest.mark.parametrize("ncons", [1, 4, 15, 16, 17, 32])
def test_constraints_in_blocks(ncons, precision, tol):
    print("gram", ncons, precision, flush=True)
    ic = gic.ICGenerator(precision=precision)
    ic.set_cosmology(**cosmology_from_paramfile(golden("test_11_import", "paramfile.txt")))
    ic.set_camb(golden("camb_transfer_kmax40_z0.dat"))
    ic.init_base_grid(BOX, N)
    rng = np.random.default_rng(ncons)
    # spheres around different points of a lattice, so that they are independent
    pts = np.stack(np.meshgrid(*[np.arange(4) * 12.5 + 3] * 3, indexing="ij"), -1).reshape(-1, 3)
    cons = np.empty((2, ncons, 5))
    for r in range(2):
        cons[r, :, :3] = pts[rng.permutation(64)[:ncons]] + rng.uniform(0, 2, (ncons, 3))
    cons[..., 3] = rng.uniform(2.5, 4.0, (2, ncons))
    cons[..., 4] = rng.normal(0, 1.5, (2, ncons))
    dt = torch.float64 if precision == gic.FLOAT64 else torch.float32
    out = torch.empty((2, 4, N, N, N), dtype=dt, device="cuda")
    torch.cuda.synchronize()
    ic.batch_constrained([31, 32], cons, out.data_ptr())
    got = out.cpu().numpy().astype(np.float64)
    for r, seed in enumerate([31, 32]):
        ic.reseed(seed)
        ic.draw()
        ic.clear_modifications()
        for x, y, z, rad, t in cons[r]:
            ic.set_flags(0, select_sphere_cells(N, BOX, (x, y, z), rad))
            ic.modify("overdensity", False, float(t))
        ic.apply_modifications()
        ic.apply_power_spectrum()
        want = ic.field(gic.FIELD_OVERDENSITY, 0)
        assert np.abs(got[r, 0] - want).max() <= tol * np.abs(want).max()
    ic.close()
