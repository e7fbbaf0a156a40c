"""Copies to the host in slots emptied by several threads: the same bytes as
the direct copies of small ranges, for sizes that fill the slots unevenly, on
one CPU, and into pinned memory."""
import os

import numpy as np
import pytest
import torch

from genetic_amd import gic

pytestmark = pytest.mark.gpu

HERE = os.path.dirname(os.path.abspath(__file__))
EH_TABLE = os.path.join(HERE, "..", "genetic_amd", "data", "eh_nowiggle_512.dat")


@pytest.fixture(scope="module")
def done():
    g = gic.ICGenerator(precision=gic.FLOAT32)
    g.set_cosmology(Om=0.31, Ol=0.69, hubble=0.677, s8=0.81, ns=0.967, z=99)
    g.set_camb(EH_TABLE)
    g.init_base_grid(50.0, 128)
    g.set_seed(5)
    g.zeldovich()
    # pieces of 2 x 1 MB, below the size that goes through the slots
    parts = [g.particles(0, start=s, count=min(90000, 128 ** 3 - s)) for s in range(0, 128 ** 3, 90000)]
    return g, np.concatenate([p[0] for p in parts]), np.concatenate([p[1] for p in parts])


# just past two slots in all, the last that is copied straight and the next (24 bytes
# a particle, 7 MB), an odd remainder, the level
@pytest.mark.parametrize("start,count", [(0, 174763), (3, 305834), (3, 305835), (12345, 700001), (1, 128 ** 3 - 1), (0, 128 ** 3)])
def test_particles_in_slots_equal_direct_copies(done, start, count):
    print("host copy of", count, "particles", flush=True)
    g, pos, vel = done
    p, v = g.particles(0, start=start, count=count)
    assert np.array_equal(p, pos[start:start + count]) and np.array_equal(v, vel[start:start + count])


def test_one_cpu_and_pinned_memory(done):
    print("host copy on one CPU, into pinned memory", flush=True)
    g, pos, vel = done
    cpus = os.sched_getaffinity(0)
    os.sched_setaffinity(0, {min(cpus)})
    try:
        p, v = g.particles(0)
    finally:
        os.sched_setaffinity(0, cpus)
    assert np.array_equal(p, pos) and np.array_equal(v, vel)
    pinned = [torch.empty((128 ** 3, 3), dtype=torch.float32, pin_memory=True) for _ in range(2)]
    g._check(gic.lib().gic_particles(g._h, 0, None, 0, 128 ** 3, pinned[0].data_ptr(), pinned[1].data_ptr()))
    assert np.array_equal(pinned[0].numpy(), pos) and np.array_equal(pinned[1].numpy(), vel)


@pytest.mark.parametrize("offset", [1, 3, 4, 8, 17])
def test_arrays_of_any_alignment(done, offset):
    """A level's field into an array that starts anywhere in memory."""
    print("host copy to offset", offset, flush=True)
    g = done[0]
    n3 = 128 ** 3
    want = g.field(gic.FIELD_PSI_X, 0, dtype=np.float32).ravel()
    raw = np.full(4 * n3 + 4096, 0x5A, dtype=np.uint8)
    at = -raw.ctypes.data % 2048 + offset
    g._check(gic.lib().gic_copy_field(g._h, gic.FIELD_PSI_X, 0, gic.REAL_SPACE, raw.ctypes.data + at, gic.DTYPE_F32))
    assert raw[at:at + 4 * n3].tobytes() == want.tobytes()
    assert (raw[:at] == 0x5A).all() and (raw[at + 4 * n3:] == 0x5A).all()
