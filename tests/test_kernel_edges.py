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


def _adjoint_inputs(g, np_, seed, fp64):
    """Particles in random cells (so that no tile has the average), fields
    with ghosts, as tensors of the run's precision."""
    import torch
    from vpic_amd import adjoint as A
    rng = np.random.default_rng(seed)
    p = np.zeros(np_, dtype=T.PARTICLE)
    x, y, z = (rng.integers(1, k + 1, np_) for k in (g.nx, g.ny, g.nz))
    p["i"] = g.voxel(x, y, z)
    for c in ("dx", "dy", "dz"):
        p[c] = rng.uniform(-1, 1, np_).astype(np.float32)
    for c in ("ux", "uy", "uz"):
        p[c] = (0.6 * rng.standard_normal(np_)).astype(np.float32)
    p["w"] = np.float32(g.dV / max(np_ / (g.nx * g.ny * g.nz), 1))
    f = H.random_fields(g, seed + 1, 0.02, 0.02)
    if fp64:
        P, F = A.host_particles64(p), A.fields64(f)
    else:
        P, F = p.view(np.float32).reshape(-1, 8), \
            f.view(np.float32).reshape(-1, 20)
    return torch.from_numpy(P).cuda(), torch.from_numpy(F).cuda()


# tiles of 8x4x4 cells: one tile with a window that wraps onto itself, two
# tiles an axis, a last tile of one cell, axes of one cell, an axis too long
# to sort or few particles (chunks of particles, no windows), the chunks at their
# shortest and longer; particle counts around a
# wavefront and a workgroup; steps past a sort, checkpoints that do and
# do not fall on one
@pytest.mark.parametrize("n,np_,steps,ckpt", [
    ((3, 2, 4), 1, 3, 2), ((8, 4, 4), 65, 10, 4), ((9, 5, 5), 257, 17, 3),
    ((17, 8, 9), 3000, 9, 20), ((16, 1, 13), 1500, 12, 5),
    ((1, 9, 1), 300, 9, 8), ((2100, 1, 1), 9000, 10, 4),
    ((2100, 1, 1), 530000, 3, 2), ((20, 15, 14), 1399, 9, 4),
    ((20, 15, 14), 1400, 9, 4)],
    ids=lambda v: str(v).replace(" ", ""))
def test_adjoint_tiles(dev, n, np_, steps, ckpt):
    """The gradients do not depend on how particles share tiles: the same
    particles in another order, each with its own gradient.  In FP64 the two
    runs differ by the rounding of sums of at most np terms in another order
    over the steps: 1e-10 of the largest is 1e5 times the rounding of one
    value, for growth of a factor below that over these steps."""
    import torch
    from vpic_amd import adjoint as A
    g = _box(*n, cell=0.1)
    P, F = _adjoint_inputs(g, np_, 5, True)
    order = torch.randperm(np_, generator=torch.Generator().manual_seed(3)
                           ).cuda()
    say("adjoint", n, np_, steps, ckpt)
    w1, u1, d1, f1 = A.run(P, F, g, -1.0, 1.0, steps, ckpt, True, True, True)
    w2, u2, d2, f2 = A.run(P[order].contiguous(), F, g, -1.0, 1.0, steps,
                           ckpt, True, True, True)
    w3 = A.run(P, F, g, -1.0, 1.0, steps, grads=False)[0]
    assert abs(w1 - w2) <= 1e-12 * abs(w1) and abs(w1 - w3) <= 1e-12 * abs(w1)
    for a, b in ((u1[order], u2), (d1[order], d2), (f1, f2)):
        assert float((a - b).abs().max()) <= 1e-10 * float(a.abs().max())
    # FP32 against FP64: few particles and steps, so crossings fall on the
    # same steps; 1e-2 in norm (the unstable 64^3 run over 200 steps, with
    # moved crossings, parts by 1.6e-2)
    P4, F4 = _adjoint_inputs(g, np_, 5, False)
    w4, u4, d4, f4 = A.run(P4, F4, g, -1.0, 1.0, steps, ckpt, True, True,
                           True)
    assert abs(w4 - w1) <= 1e-5 * abs(w1)
    assert float((u4.double() - u1).norm()) <= 1e-2 * float(u1.norm())
    assert float((f4.double() - f1).norm()) <= 1e-2 * float(f1.norm())


def test_adjoint_workspace(dev):
    """The caller's workspace gives the call's own allocation's result; one
    too small or misaligned is refused."""
    import torch
    from vpic_amd import adjoint as A
    g = _box(9, 5, 5, cell=0.1)
    P, F = _adjoint_inputs(g, 700, 8, True)
    need = ctypes.c_int64()
    _lib.call("vpic_hip_adjoint_workspace", 700, ctypes.byref(g), 9, 4, 8, 1,
              ctypes.byref(need))
    ws = torch.empty(need.value + 512, dtype=torch.uint8, device="cuda")
    en = ctypes.c_double()
    ub = torch.empty((700, 3), dtype=torch.float64, device="cuda")

    def call(ptr, n):
        _lib.call("vpic_hip_adjoint_bfield_energy_ws", P.data_ptr(), 700,
                  -1.0, 1.0, F.data_ptr(), ctypes.byref(g), 9, 4, 8,
                  ctypes.byref(en), ub.data_ptr(), None, None, ptr, n, None)
    call(None, 0)
    w, u = en.value, ub.clone()
    call(ws.data_ptr(), need.value)
    assert abs(en.value - w) <= 1e-12 * abs(w)
    # sums of at most 700 terms in another order over nine steps
    assert float((ub - u).abs().max()) <= 1e-10 * float(u.abs().max())
    for ptr, n in ((ws.data_ptr(), need.value - 1),
                   (ws.data_ptr() + 16, need.value)):
        with pytest.raises(_lib.VpicError):
            call(ptr, n)
    assert A.run(P, F, g, -1.0, 1.0, 9, 4)[0] == pytest.approx(w, rel=1e-12)


# one particle, around a workgroup's round, past one chunk per workgroup of
# the least and of the most particles; in cell order (with drift), in no order
# on a grid of more nodes than a chunk's table holds, axes of one cell
@pytest.mark.parametrize("n,np_,order", [
    ((4, 3, 5), 1, "sorted"), ((4, 3, 5), 511, "sorted"),
    ((16, 9, 7), 513, "drifted"), ((64, 20, 10), 600001, "drifted"),
    ((90, 60, 50), 40000, "random"), ((40, 1, 30), 70000, "drifted"),
    ((1, 1, 6), 5000, "random")],
    ids=lambda v: str(v).replace(" ", ""))
def test_accumulate_rho_chunks(dev, n, np_, order):
    """rhof against the same weights summed in FP64.  A node's sum of k terms
    is off by at most k roundings of 2^-24 of the terms' magnitudes.  A term
    w (1 +- dx)(1 +- dy)(1 +- dz) is formed as w -+ dx w and so on: six
    roundings of values up to 8 w, whatever cancels."""
    g = _box(*n)
    rng = np.random.default_rng(np_ + 1)
    c = [rng.integers(1, k + 1, np_) for k in n]
    i = g.voxel(*c)
    if order != "random":
        i = np.sort(i)
    p = np.zeros(np_, dtype=T.PARTICLE)
    if order == "drifted":
        moved = rng.random(np_) < 0.4
        x = i % (g.nx + 2)
        i = np.where(moved, i - x + 1 + (x + np_ % 2) % g.nx, i)
    p["i"] = i
    for k in ("dx", "dy", "dz"):
        p[k] = rng.uniform(-1, 1, np_).astype(np.float32)
    p["w"] = rng.uniform(0.5, 2, np_).astype(np.float32)
    f = H.random_full_fields(g, 3)
    want = f["rhof"].astype(np.float64)
    mag, terms, full = np.abs(want), np.zeros(g.nv), np.zeros(g.nv)
    d = [p[k].astype(np.float64) for k in ("dx", "dy", "dz")]
    for k in range(8):
        s = [(k >> a & 1) for a in range(3)]
        w = p["w"] * (-0.7 * np.float64(g.r8V))
        for a in range(3):
            w = w * (1 + (2 * s[a] - 1) * d[a])
        at = p["i"] + s[0] + s[1] * g.sy + s[2] * g.sz
        np.add.at(want, at, w)
        np.add.at(mag, at, np.abs(w))
        np.add.at(terms, at, 1)
        np.add.at(full, at, 8 * p["w"] * 0.7 * np.float64(g.r8V))
    df, dp = dev.DeviceArray.from_host(f), dev.DeviceArray.from_host(p)
    say("accumulate_rho_p", n, np_, order)
    _lib.call("vpic_hip_accumulate_rho_p", df.ptr, dp.ptr, np_, -0.7,
              ctypes.byref(g), None)
    out = df.download()
    err = np.abs(out["rhof"] - want)
    assert np.all(err <= 2.0 ** -24 * ((terms + 2) * mag + 6 * full))
    for k in T.FIELD_FLOATS:
        if k != "rhof":
            assert np.array_equal(out[k], f[k])


# one particle; 16 lanes of one voxel and one more; few particles over a grid
# of two slabs of voxels; planes just below and above half a slab, and far above;
# axes of one cell; an axis too long to sort by; just below and above a particle
# in twelve cells
@pytest.mark.parametrize("n,np_", [
    ((4, 3, 5), 1), ((2, 1, 2), 16 * 4 + 1), ((9, 8, 7), 12000),
    ((70, 70, 63), 30000), ((385, 384, 3), 60000), ((386, 384, 3), 60000),
    ((900, 700, 1), 60000), ((33, 1, 20), 5000), ((2100, 1, 1), 4000),
    ((20, 20, 20), 666), ((20, 20, 20), 667)],
    ids=lambda v: str(v).replace(" ", ""))
def test_hydro_voxel_sums(dev, orc, n, np_):
    """The moments of particles in no order against the oracle's, within the
    1e-5 of each moment's largest value that its other order of summing
    allows; added to what the array holds."""
    g = _box(*n)
    rng = np.random.default_rng(np_)
    f = H.random_fields(g, 4, 0.1, 0.2)
    fi = H.interp_array(g)
    orc.load_interpolator(fi, f, g)
    p = np.zeros(np_, dtype=T.PARTICLE)
    p["i"] = g.voxel(*(rng.integers(1, k + 1, np_) for k in n))
    for k in ("dx", "dy", "dz"):
        p[k] = rng.uniform(-1, 1, np_).astype(np.float32)
    for k in ("ux", "uy", "uz"):
        p[k] = (0.3 * rng.standard_normal(np_)).astype(np.float32)
    p["w"] = rng.uniform(0.5, 2, np_).astype(np.float32)
    want = np.zeros(g.nv, dtype=T.HYDRO)
    want["rho"] = 0.25
    dh = dev.DeviceArray.from_host(want)
    orc.accumulate_hydro_p(want, p, -1.0, 1.0, fi, g)
    dp, dfi = dev.DeviceArray.from_host(p), dev.DeviceArray.from_host(fi)
    say("accumulate_hydro_p", n, np_)
    import torch
    free = torch.cuda.mem_get_info()[0]
    _lib.call("vpic_hip_accumulate_hydro_p", dh.ptr, dp.ptr, np_, -1.0, 1.0,
              dfi.ptr, ctypes.byref(g), None, None)
    # (scratch: 128 MiB of sums, an eighth more, and what a particle and a
    # voxel take)
    assert free - torch.cuda.mem_get_info()[0] < 200 << 20
    got = dh.download()
    for k in T.HYDRO_FIELDS:
        assert np.max(np.abs(got[k] - want[k])) <= \
            1e-5 * np.max(np.abs(want[k])), k
    # a particle whose nodes leave the grid is skipped and reported
    p["i"][np_ // 2] = g.nv - 3
    dp = dev.DeviceArray.from_host(p)
    with pytest.raises(_lib.VpicError, match="1 particles"):
        _lib.call("vpic_hip_accumulate_hydro_p", dh.ptr, dp.ptr, np_, -1.0,
                  1.0, dfi.ptr, ctypes.byref(g), None, None)


# the one-launch jf fold and tangential-B ghosts where an axis has one or two
# cells (its two faces are neighbours), periodic or with walls on one axis
@pytest.mark.parametrize("wall", [None, 0, 1, 2])
@pytest.mark.parametrize("n", [(1, 1, 1), (1, 5, 3), (2, 2, 2), (4, 1, 1),
                               (3, 2, 70)],
                         ids=lambda v: "x".join(map(str, v)))
def test_faces_in_one_launch(dev, orc, n, wall):
    """Bit for bit the oracle's axis after axis."""
    g = T.grid_periodic(0, 0, 0, *n, *n, 0.4)
    if wall is not None:
        g.fbc[wall] = g.fbc[wall + 3] = T.BC_PEC_FIELDS
    f = H.random_full_fields(g, 9)
    mp = T.vacuum_params()
    df = dev.DeviceArray.from_host(f)
    say("faces", n, wall)
    G = ctypes.byref(g)
    _lib.call("vpic_hip_synchronize_jf", df.ptr, G, None)
    _lib.call("vpic_hip_vacuum_advance_e", df.ptr, G, ctypes.byref(mp), 1.0,
              None)
    _lib.call("vpic_hip_compute_div_e_err", df.ptr, G, ctypes.byref(mp), None)
    _lib.call("vpic_hip_clean_div_b", df.ptr, G, None)
    orc.synchronize_jf(f, g)
    orc.vacuum_advance_e(f, g, mp)
    orc.compute_div_e_err(f, g, mp)
    orc.clean_div_b(f, g)
    got = df.download()
    for c in T.FIELD_FLOATS:
        assert H.same_bits(got[c], f[c]), c


# batches of voxels in the collision operator: 64 voxels at most (sparse, most
# voxels with 0 or 1 particle), batches that end inside a neighbourhood, and
# voxels that just fill a batch of 1792 particles or exceed it; partners many,
# few and none; few particles in so many voxels that each has a lane
@pytest.mark.parametrize("n,lo,hi,crowd", [
    ((70, 2, 2), 0, 2, ()), ((13, 5, 4), 20, 90, ()),
    ((4, 3, 3), 0, 9, (1791, 1792, 1793, 4100)), ((2, 1, 1), 1792, 1792, ()),
    ((3, 2, 1), 700, 1500, ()), ((64, 64, 33), 0, 2, (3000, 1))],
    ids=["sparse", "ordinary", "crowded", "full", "large", "many"])
def test_collision_batches(dev, orc, n, lo, hi, crowd):
    """Bit for bit the oracle's voxel after voxel, within a species and
    between two in both orders of their sizes."""
    g = T.grid_periodic(0, 0, 0, *n, *n, 0.2)
    rng = np.random.default_rng(17)
    v = np.arange(g.nv)
    x, y, z = v % (g.nx + 2), v // (g.nx + 2) % (g.ny + 2), v // (
        (g.nx + 2) * (g.ny + 2))
    inner = np.nonzero((x >= 1) & (x <= g.nx) & (y >= 1) & (y <= g.ny) &
                       (z >= 1) & (z <= g.nz))[0]

    def species(lo, hi, crowd, w):
        c = np.zeros(g.nv, np.int64)
        c[inner] = rng.integers(lo, hi + 1, len(inner))
        c[inner[1:1 + len(crowd)]] = crowd
        p = np.zeros(int(c.sum()), T.PARTICLE)
        p["i"] = np.repeat(np.arange(g.nv, dtype=np.int32), c)
        for k in ("dx", "dy", "dz"):
            p[k] = rng.uniform(-1, 1, len(p)).astype(np.float32)
        for k in ("ux", "uy", "uz"):
            p[k] = (0.1 * rng.standard_normal(len(p))).astype(np.float32)
        p["w"] = rng.choice(np.array(w, np.float32), len(p))
        part = np.zeros(g.nv + 1, np.int32)
        part[1:] = np.cumsum(c)
        return p, part

    pe, parte = species(lo, hi, crowd, [1.0])
    pi, parti = species(0, 7 if len(inner) < 1 << 17 else 2, crowd[:2],
                        [1.0, 2.5])
    de, dpe = dev.DeviceArray.from_host(pe), dev.DeviceArray.from_host(parte)
    di, dpi = dev.DeviceArray.from_host(pi), dev.DeviceArray.from_host(parti)
    E = (pe, parte, de, dpe, -1.0, 1.0)
    I = (pi, parti, di, dpi, 1.0, 25.0)
    # a draw that the shuffle rejects, so that the words behind it move up:
    # the 693rd of voxel 18 (1792 particles where each voxel has as many)
    word = int(orc.philox4x32((693 // 4, 18, 5469, 0), (1234, 0))[693 % 4])
    assert word // ((2**32 - 1) // (1792 - 693)) >= 1792 - 693
    for call, a, b in [(0, E, E), (1, E, I), (2, I, E), (5469, E, E)]:
        say("collide", n, call)
        orc.takizuka_abe(a[0], a[1], a[4], a[5], b[0], b[1], b[4], b[5], 0.5,
                         2, 1234, call, g)
        _lib.call("vpic_hip_takizuka_abe", a[2].ptr, a[3].ptr, len(a[0]),
                  a[4], a[5], b[2].ptr, b[3].ptr, len(b[0]), b[4], b[5], 0.5,
                  2, 1234, call, ctypes.byref(g), None)
        assert H.same_bits(de.download(), pe), call
        assert H.same_bits(di.download(), pi), call


# the field part of a step in four launches, where axes have one or two cells
# (ghosts and faces are neighbours), rows past a workgroup, and with walls
# (the separate calls) or without a work array
@pytest.mark.parametrize("wall,work", [(None, True), (None, False),
                                       (1, True)])
@pytest.mark.parametrize("n", [(1, 1, 1), (1, 5, 3), (2, 2, 2), (4, 1, 1),
                               (3, 2, 70), (300, 2, 3), (17, 16, 15)],
                         ids=lambda v: "x".join(map(str, v)))
def test_field_step(dev, n, wall, work):
    """Bit for bit the separate calls, ghosts and interpolators included, from
    any content of the work array, twice in a row."""
    g = T.grid_periodic(0, 0, 0, *n, *n, 0.4)
    if wall is not None:
        g.fbc[wall] = g.fbc[wall + 3] = T.BC_PEC_FIELDS
    f = H.random_full_fields(g, 9)
    rng = np.random.default_rng(2)
    acc = rng.standard_normal((g.nv, 12)).astype(np.float32)
    mp = T.vacuum_params(damp=0.02)
    G, M = ctypes.byref(g), ctypes.byref(mp)
    da = dev.DeviceArray.from_host(acc)
    a, b = (dev.DeviceArray.from_host(f) for _ in range(2))
    ia, ib = dev.interpolators(g), dev.interpolators(g)
    ia.zero()
    ib.zero()
    w = dev.DeviceArray.from_host(
        np.full((g.nv, 4), np.nan, np.float32)) if work else None
    say("field step", n, wall, work)
    for _ in range(2):
        _lib.call("vpic_hip_clear_jf_unload_accumulator_array", a.ptr, da.ptr,
                  G, None)
        _lib.call("vpic_hip_synchronize_jf", a.ptr, G, None)
        _lib.call("vpic_hip_advance_b", a.ptr, G, 0.5, None)
        _lib.call("vpic_hip_vacuum_advance_e", a.ptr, G, M, 1.0, None)
        _lib.call("vpic_hip_advance_b", a.ptr, G, 0.5, None)
        _lib.call("vpic_hip_load_interpolator_array", ia.ptr, a.ptr, G, None)
        _lib.call("vpic_hip_field_step", b.ptr, da.ptr, ib.ptr,
                  w.ptr if work else None, G, M, None)
        assert H.same_bits(b.download(), a.download())
        assert H.same_bits(ib.download(), ia.download())


# the jf fold of all axes and the B ghosts in one launch, and their transposes,
# where an axis has one or two cells (the copies of an element are neighbours)
@pytest.mark.parametrize("n", [(3, 2, 4), (1, 5, 3), (2, 1, 6), (7, 1, 1)],
                         ids=lambda v: "x".join(map(str, v)))
def test_adjoint_faces(dev, orc, n):
    """FP64: the run's energy is the FP64 oracle's, and its gradient in the
    fields gives the central difference along a random direction (step 1e-6
    of fields of 0.02: truncation and rounding both below 1e-8 of it, where no
    particle crosses a face in between; 1e-5 leaves room for their sum over
    the steps)."""
    import torch
    from oracle.trace import OracleRun
    from vpic_amd import adjoint as A
    g = _box(*n, cell=0.1)
    P, F = _adjoint_inputs(g, 40, 8, True)
    f = H.random_fields(g, 9, 0.02, 0.02)  # the inputs' fields
    P32, _ = _adjoint_inputs(g, 40, 8, False)
    p = P32.cpu().numpy().reshape(-1).view(T.PARTICLE)
    steps = 6
    say("adjoint faces", n)
    w, _, _, fb = A.run(P, F, g, -1.0, 1.0, steps, 4, True, True, True)
    r = OracleRun(g, [("electron", -1.0, 1.0, p)], fp64=True, fields=f)
    r.load_interpolator()
    for _ in range(steps):
        r.advance()
    wo = r.energies()[0][3:6].sum()
    r.close()
    assert abs(w - wo) <= 1e-12 * abs(wo)
    d = torch.from_numpy(np.random.default_rng(3).standard_normal(
        (g.nv, 6))).cuda()
    dF = torch.zeros_like(F)
    dF[:, 0:3], dF[:, 4:7] = d[:, 0:3], d[:, 3:6]
    eps = 2e-8
    hi, lo = (A.run(P, (F + s * eps * dF).contiguous(), g, -1.0, 1.0, steps,
                    grads=False)[0] for s in (1, -1))
    want = (hi - lo) / (2 * eps)
    got = float((fb * d).sum())
    say("adjoint", got, "difference", want)
    assert abs(got - want) <= 1e-5 * abs(want)


def test_sort_scratch_across_streams(dev):
    """A sort left queued on one stream and the next use of its thread's
    scratch on another (the hydro moments, the adjoint run, another sort): the
    results of one call after the other, bit for bit (the gradient's sums have
    no fixed order: within 1e-10 of its largest, as above)."""
    import torch
    from vpic_amd import adjoint as A
    g = _box(48, 40, 36)
    n_a, n_b = 3000000, 2900000
    rng = np.random.default_rng(8)

    def cloud(n):
        p = np.zeros(n, dtype=T.PARTICLE)
        p["i"] = g.voxel(*(rng.integers(1, k + 1, n)
                           for k in (g.nx, g.ny, g.nz)))
        p["w"] = np.arange(n, dtype=np.float32)
        p["ux"] = rng.standard_normal(n).astype(np.float32)
        return p
    a, b = cloud(n_a), cloud(n_b)
    da, db = dev.DeviceArray.from_host(a), dev.DeviceArray.from_host(b)
    dfi = dev.DeviceArray.from_host(H.interp_array(g))
    hydro = dev.DeviceArray((g.nv,), T.HYDRO)
    P, F = _adjoint_inputs(_box(9, 5, 5, 0.1), 257, 5, True)

    def moments(stream):
        _lib.call("vpic_hip_accumulate_hydro_p", hydro.ptr, db.ptr, n_b, -1.0,
                  1.0, dfi.ptr, ctypes.byref(g), None, stream)
        return hydro.download()

    def gradient(stream):  # (always on the default stream)
        return A.run(P, F, _box(9, 5, 5, 0.1), -1.0, 1.0, 9,
                     4)[1].cpu().numpy()

    aux_b = dev.particles(n_b)
    part_b = dev.DeviceArray((g.nv + 1,), np.int32)

    def other_sort(stream):
        _lib.call("vpic_hip_sort_p", db.ptr, aux_b.ptr, n_b, part_b.ptr,
                  ctypes.byref(g), 0, stream)
        return aux_b.download()

    order = np.argsort(a["i"], kind="stable")
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    for name, second in (("hydro", moments), ("adjoint", gradient),
                         ("sort_p", other_sort)):
        hydro.zero()
        torch.cuda.synchronize()
        want = second(None)
        aux = dev.particles(n_a)
        part = dev.DeviceArray((g.nv + 1,), np.int32)
        hydro.zero()
        torch.cuda.synchronize()
        say("sort_p, then", name, "on another stream")
        _lib.call("vpic_hip_sort_p", da.ptr, aux.ptr, n_a, part.ptr,
                  ctypes.byref(g), 0, s1.cuda_stream)
        got = second(s2.cuda_stream)
        torch.cuda.synchronize()
        assert H.same_bits(aux.download(), a[order])
        if name == "adjoint":
            assert np.max(np.abs(got - want)) <= 1e-10 * np.max(np.abs(want))
        else:
            assert H.same_bits(got, want)


@pytest.mark.parametrize("limit", [16000, 40000])
def test_hydro_without_scratch(dev, orc, limit):
    """Where the scratch of the sorted sums is not there (the particles' keys;
    the voxels' sums) the particles go one by one, with the oracle's moments
    and each bad voxel counted once."""
    g = _box(3, 2, 3)
    np_ = 7000
    rng = np.random.default_rng(4)
    fi = H.interp_array(g)
    orc.load_interpolator(fi, H.random_fields(g, 4, 0.1, 0.2), g)
    p = np.zeros(np_, dtype=T.PARTICLE)
    p["i"] = g.voxel(*(rng.integers(1, k + 1, np_)
                       for k in (g.nx, g.ny, g.nz)))
    p["dx"] = rng.uniform(-1, 1, np_).astype(np.float32)
    p["ux"] = (0.3 * rng.standard_normal(np_)).astype(np.float32)
    p["w"] = 1.0
    want = np.zeros(g.nv, dtype=T.HYDRO)
    orc.accumulate_hydro_p(want, p, -1.0, 1.0, fi, g)
    bad = p.copy()
    bad["i"][5] = g.nv - 2
    dfi = dev.DeviceArray.from_host(fi)

    def moments(q):
        dh = dev.DeviceArray((g.nv,), T.HYDRO)
        dh.zero()
        dp = dev.DeviceArray.from_host(q)
        _lib.call("vpic_hip_accumulate_hydro_p", dh.ptr, dp.ptr, np_, -1.0,
                  1.0, dfi.ptr, ctypes.byref(g), None, None)
        return dh.download()
    say("accumulate_hydro_p, scratch limit", limit)
    try:
        _lib.call("vpic_hip_scratch_limit", limit)
        got = moments(p)
        with pytest.raises(_lib.VpicError, match="1 particles"):
            moments(bad)
    finally:
        _lib.call("vpic_hip_scratch_limit", 0)
    for k in T.HYDRO_FIELDS:
        assert np.max(np.abs(got[k] - want[k])) <= \
            1e-5 * max(np.max(np.abs(want[k])), 1e-30), k


@pytest.mark.parametrize("n", [(9, 5, 5), (2100, 1, 1)],
                         ids=lambda v: str(v).replace(" ", ""))
@pytest.mark.parametrize("fp64", [False, True])
def test_adjoint_refuses_particles_in_no_cell(dev, n, fp64):
    """A particle in a ghost voxel belongs to no tile: refused, not left out
    with a gradient of zero; the same where the voxel is off the grid."""
    import torch
    from vpic_amd import adjoint as A
    g = _box(*n, cell=0.1)
    P, F = _adjoint_inputs(g, 300, 8, fp64)
    cells = P.view(-1).view(torch.int32)
    at = (7 * 16 + 6) if fp64 else (7 * 8 + 3)  # particle 7's voxel
    good = int(cells[at])
    A.run(P, F, g, -1.0, 1.0, 3, 2)
    for v in (g.voxel(0, 1, 1), g.voxel(1, 1, n[2] + 1), g.nv, -1):
        cells[at] = v
        say("adjoint, particle in voxel", v, n, fp64)
        for grads in (True, False):
            with pytest.raises(_lib.VpicError, match="1 particles"):
                A.run(P, F, g, -1.0, 1.0, 3, 2, grads)
    cells[at] = good
    A.run(P, F, g, -1.0, 1.0, 3, 2)


def test_adjoint_large_workspace_is_given_back(dev, monkeypatch):
    """A call that needs more than its share of the GPU's memory leaves nothing
    in torch's cache, where the library could not use it."""
    import torch
    from vpic_amd import adjoint as A
    g = _box(33, 25, 25, cell=0.1)
    P, F = _adjoint_inputs(g, 257, 5, True)
    w, u = A.run(P, F, g, -1.0, 1.0, 9, 4)[:2]
    need = ctypes.c_int64()
    _lib.call("vpic_hip_adjoint_workspace", 257, ctypes.byref(g), 9, 4, 8, 1,
              ctypes.byref(need))
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.empty_cache()
    before = torch.cuda.memory_reserved()
    say("adjoint, workspace beyond its share")
    monkeypatch.setattr(A, "KEEP_SHARE", (need.value - 1) / total)
    w2, u2 = A.run(P, F, g, -1.0, 1.0, 9, 4)[:2]
    # (u2 itself is a small block of torch's, from its 2-MiB pools)
    assert need.value > 20 << 20
    assert torch.cuda.memory_reserved() - before <= 4 << 20
    assert abs(w - w2) <= 1e-12 * abs(w)
    assert float((u - u2).abs().max()) <= 1e-10 * float(u.abs().max())
    monkeypatch.setattr(A, "KEEP_SHARE", need.value / total)
    A.run(P, F, g, -1.0, 1.0, 9, 4)
    assert torch.cuda.memory_reserved() - before >= need.value
