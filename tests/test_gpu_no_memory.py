"""The differentiable entry points where device memory runs out after the
caller's noise has begun to replace the context's: the call fails, the context
has no half-made field afterwards, and works again once there is memory."""
import os

import numpy as np
import pytest
import torch

from genetic_amd import gic

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
EH_TABLE = os.path.join(HERE, "..", "genetic_amd", "data", "eh_nowiggle_512.dat")
N = 512
FIELD = 8 * N * N * (N + 2)


def _gen():
    g = gic.ICGenerator(precision=gic.FLOAT64)
    g.set_cosmology(Om=0.31, Ol=0.69, hubble=0.677, s8=0.81, ns=0.967, z=99)
    g.set_camb(EH_TABLE)
    g.init_base_grid(200.0, N)
    return g


@pytest.mark.parametrize("entry", ["forward", "masked"])
def test_failed_call_leaves_no_half_made_field(entry):
    print("no memory in", entry, flush=True)
    g = _gen()
    w = torch.randn((N, N, N), dtype=torch.float64, device="cuda")
    psi = [torch.empty_like(w) for _ in range(3)]
    mask = torch.ones((N, N, N), dtype=torch.bool, device="cuda")   # its box is the level: scratch of 8 fields

    def call():
        torch.cuda.synchronize()
        if entry == "forward":
            g.displacement_forward([w.data_ptr()], [p.data_ptr() for p in psi])
        else:
            g.masked_displacement(w.data_ptr(), mask.data_ptr())

    # room for the noise and half a field more; the scratch takes three fields at least
    free = torch.cuda.mem_get_info()[0]
    assert free > 6 * FIELD
    filler = torch.empty(int(free - 2.2 * FIELD), dtype=torch.uint8, device="cuda")
    with pytest.raises(gic.GICError, match="memory"):
        call()
    with pytest.raises(gic.GICError, match="seeded"):
        g.field(gic.FIELD_OVERDENSITY, 0)
    with pytest.raises(gic.GICError):
        g.particles(0, count=10)
    del filler
    torch.cuda.empty_cache()
    call()
    got = g.field(gic.FIELD_OVERDENSITY, 0)
    g.close()
    g = _gen()
    call()
    assert np.array_equal(g.field(gic.FIELD_OVERDENSITY, 0), got)
    g.close()
