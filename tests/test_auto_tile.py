"""The partition-driven push with the tile it chooses itself: grids of fewer
tiles than CUs, of several tiles per CU in density order, between walls, one
cell thick, and particles past the partition."""
import ctypes
import sys

import numpy as np
import pytest

from oracle.oracle import host_grid
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


@pytest.fixture(autouse=True)
def chosen_tile():
    was = (ctypes.c_int32 * 4)()
    _lib.call("vpic_hip_push_get_tile", was)
    _lib.call("vpic_hip_push_tile", 0, 0, 0)
    yield
    _lib.call("vpic_hip_push_tile_window", *was)


def _particles(g, np_, seed, dense):
    """Random cells, four fifths of them in a slab of the share `dense` of the
    longest axis (0: none)."""
    rng = np.random.default_rng(seed)
    p = np.zeros(np_, dtype=T.PARTICLE)
    n = (g.nx, g.ny, g.nz)
    c = [rng.integers(1, k + 1, np_) for k in n]
    if dense:
        a = int(np.argmax(n))
        c[a] = np.where(rng.random(np_) < 0.8,
                        1 + n[a] // 2 + c[a] % max(int(n[a] * dense), 1),
                        c[a])
    p["i"] = g.voxel(*c)
    for k in ("dx", "dy", "dz"):
        p[k] = rng.uniform(-1, 1, np_).astype(np.float32)
    for k in ("ux", "uy", "uz"):
        p[k] = (0.3 * rng.standard_normal(np_)).astype(np.float32)
    p["w"] = rng.uniform(0.5, 1.5, np_).astype(np.float32)
    return p


# a single cell; fewer tiles than CUs; more, with a dense slab; a thin
# grid; particle walls; particles appended after the sort, also more than it
# sorted
@pytest.mark.parametrize("n,np_,dense,walls,extra", [
    ((1, 1, 1), 40, False, False, 0), ((12, 10, 9), 3000, False, False, 70),
    ((64, 48, 40), 60000, True, False, 0), ((200, 1, 90), 30000, True, True, 5),
    ((3, 90, 80), 20000, True, False, 1),
    ((20, 18, 16), 4000, False, False, 9001)],
    ids=lambda v: str(v).replace(" ", ""))
def test_push_auto_tile(dev, orc, n, np_, dense, walls, extra):
    """Two species in one call against the oracle: particles bit for bit, the
    currents within 1e-5 of the largest (the order of the sums differs)."""
    dt = 0.95 * T.courant_length(*n, *n) if max(n) > 1 else 0.5
    g = T.grid_periodic(0, 0, 0, *n, *n, dt)
    if walls:
        for k in (0, 3):
            g.fbc[k] = T.BC_PEC_FIELDS
            g.pbc[k] = T.BC_REFLECT_PARTICLES
    _push_against_oracle(dev, orc, g, np_, 0.1 if dense else 0, extra, 2)


def _push_against_oracle(dev, orc, g, np_, dense, extra, nsp):
    f = H.random_fields(g, 6, 0.05, 0.1)
    fi = H.interp_array(g)
    orc.load_interpolator(fi, f, g)
    hg = host_grid(g)
    ao = H.acc_array(g)
    keep, want = [], []
    for k, (q, m) in enumerate(((-1.0, 1.0), (1.0, 25.0))[:nsp]):
        p = _particles(g, np_, 7 + k, dense)
        part = orc.sort_p(p, g)
        if extra:
            p = np.concatenate([p, _particles(g, extra, 17 + k, False)])
        po = p.copy()
        nm, ign, pmo = orc.advance_p(po, q, m, ao, fi, hg)
        want.append((po, nm, ign))
        keep.append([dev.DeviceArray.from_host(p), dev.movers(len(p)),
                     dev.DeviceArray((4,), np.int32),
                     dev.DeviceArray.from_host(part.astype(np.int32)),
                     len(p), q, m])
    da, dfi = dev.DeviceArray.from_host(H.acc_array(g)), \
        dev.DeviceArray.from_host(fi)
    arr = (T.PushSpecies * nsp)(*[
        T.PushSpecies(a.ptr, ln, q, m, pm.ptr, ln, nm.ptr, part.ptr, None)
        for a, pm, nm, part, ln, q, m in keep])
    say("advance_p_species, chosen tile", g.nx, g.ny, g.nz, np_, dense)
    _lib.call("vpic_hip_advance_p_species", nsp, arr, da.ptr, dfi.ptr,
              ctypes.byref(g), None)
    for (a, pm, nm, *_), (po, nmo, igo) in zip(keep, want):
        assert H.same_bits(a.download(), po)
        assert tuple(nm.download()[:3]) == (nmo, igo, 0)
    assert H.acc_rel_err(da.download(), ao) <= 1e-5


# a plane of every orientation; the densest cells at the mean, at several times
# it and at far more, where the push has tiles of three sizes to take; fewer
# tiles of the largest size than CUs, and more; particles past the partition
@pytest.mark.parametrize("dense", [0, 0.25, 0.05, 0.004])
@pytest.mark.parametrize("n,ppc,nsp,extra", [
    ((203, 1, 150), 14, 2, 3), ((1, 190, 161), 30, 1, 0),
    ((260, 243, 1), 8, 2, 0)], ids=lambda v: str(v).replace(" ", ""))
def test_push_tile_by_density(dev, orc, n, ppc, nsp, extra, dense):
    g = T.grid_periodic(0, 0, 0, *n, *n, 0.95 * T.courant_length(*n, *n))
    np_ = ppc * n[0] * n[1] * n[2]
    out, k = (ctypes.c_int32 * 12)(), ctypes.c_int32()
    _lib.call("vpic_hip_push_tile_choices", ctypes.byref(g), nsp * np_, out,
              ctypes.byref(k))
    assert k.value >= 2
    _push_against_oracle(dev, orc, g, np_, dense, extra, nsp)
