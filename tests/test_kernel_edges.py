"""GPU kernels at the sizes where their work splits change: digit groups and
block lengths of the sort, chunk and tile remainders."""
import ctypes
import sys

import numpy as np
import pytest

from vpic_amd import _lib
from vpic_amd import types as T

import helpers as H

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture(scope="module")
def dev():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    _lib.call("vpic_hip_init", 0)
    from vpic_amd import device
    return device


def _box(nx, ny, nz, cell=1.0):
    dt = 0.95 * T.courant_length(nx * cell, ny * cell, nz * cell, nx, ny, nz)
    return T.grid_periodic(0, 0, 0, nx * cell, ny * cell, nz * cell, nx, ny,
                           nz, dt)


# one digit of three axes, two of them (xy; yz), none; at the digit limit of
# 2048 values (one axis; 14*12*12 = 2016 and 16*16*8 = 2048 together); lengths
# around a block, and past 512 * 4096 where the blocks grow
@pytest.mark.parametrize("n,np_", [
    ((12, 10, 9), 1), ((12, 10, 9), 511), ((12, 10, 10), 513),
    ((14, 14, 6), 5000), ((32, 31, 30), 20001), ((70, 30, 3), 4097),
    ((512, 1, 7), 30000), ((2046, 1, 1), 9000), ((1, 2046, 2), 9001),
    ((65, 60, 3), 2097152 + 777), ((97, 61, 83), 100003)],
    ids=lambda v: str(v).replace(" ", ""))
def test_sort_digit_groups(dev, n, np_):
    """Stable by voxel with the partition, whatever the axes share a digit;
    from the particles and from a copy of their keys."""
    g = _box(*n)
    rng = np.random.default_rng(np_)
    p = np.zeros(np_, dtype=T.PARTICLE)
    x, y, z = (rng.integers(1, k + 1, np_) for k in n)
    p["i"] = g.voxel(x, y, z)
    p["w"] = np.arange(np_, dtype=np.float32)
    p["ux"] = rng.standard_normal(np_).astype(np.float32)
    want = p[np.argsort(p["i"], kind="stable")]
    part = np.searchsorted(want["i"], np.arange(g.nv + 1)).astype(np.int32)
    for keys in (None, dev.DeviceArray.from_host(p["i"].copy())):
        dp, aux = dev.DeviceArray.from_host(p), dev.particles(np_)
        dpart = dev.DeviceArray((g.nv + 1,), np.int32)
        say("sort_p", n, np_, "keys" if keys else "particles")
        if keys is None:
            _lib.call("vpic_hip_sort_p", dp.ptr, aux.ptr, np_, dpart.ptr,
                      ctypes.byref(g), 0, None)
        else:
            _lib.call("vpic_hip_sort_p_keys", dp.ptr, aux.ptr, np_, dpart.ptr,
                      keys.ptr, ctypes.byref(g), 0, None)
        assert H.same_bits(aux.download(), want)
        assert np.array_equal(dpart.download(), part)
