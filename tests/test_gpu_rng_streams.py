"""The parse and the stores of the device RNG where they can go wrong: draws
of a few values, chunks of one, two and four ranlxs2 blocks, rows shorter
than the four values stored at a time, and targets that end inside them --
against the oracle's serial stream."""
import numpy as np
import pytest

import pyoracle as po
from genetic_amd import gic

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 11, 12, 13, 767, 768, 769, 20011, 700_001, 1_428_013, 1_428_017,
                               1_500_001, 2_857_889, 2_857_893, 3_000_001])
def test_stream_of_any_length(n):
    """One block per chunk up to 1 428 014 values, two up to 2 857 890, then
    four; the values past the first are the same numbers in the same order."""
    seed = 4099 + n
    ic = gic.ICGenerator(precision=gic.FLOAT64)
    got = ic.gaussian_stream(seed, n)
    ic.close()
    want, _ = po.gaussians(seed, n)
    np.testing.assert_allclose(got, want, rtol=0, atol=1e-13)


@pytest.mark.parametrize("precision", [32, 64])
@pytest.mark.parametrize("sizes", [(4, 4), (8, 4), (4, 32), (16, 8)])
def test_rows_and_levels_shorter_than_a_store(precision, sizes):
    """The stream runs on over rows and from the base level into the zoom."""
    n0, n1 = sizes
    ic = gic.ICGenerator(precision=precision)
    ic.set_cosmology(Om=0.279, Ol=0.721, s8=0.817, ns=0.96, z=99.0)
    ic.set_power_law(1.0)
    ic.init_base_grid(50.0, n0)
    ic.init_zoom_grid_with_origin_at(0, 0, 0, 2, n1)
    ic.set_seed(77)
    ic.draw()
    want, _ = po.gaussians(77, n0 ** 3 + n1 ** 3)
    # the first read of a level removes its mean (the k = 0 mode's real part)
    for level, w in ((0, want[:n0 ** 3].reshape((n0,) * 3)), (1, want[n0 ** 3:].reshape((n1,) * 3))):
        tol = 1e-5 if precision == 32 else 1e-12
        np.testing.assert_allclose(ic.field(gic.FIELD_OVERDENSITY, level), w - w.mean(), rtol=0, atol=tol)
    ic.close()
