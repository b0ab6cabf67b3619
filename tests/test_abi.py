"""CPU checks of the C-ABI library: it loads, exports every entry point the
headers declare, and rejects bad arguments before touching a device (the
reference's "Bad args" paths, e.g. advance_p_pipeline.cc:263-270)."""
import ctypes
import os
import re
import subprocess
import sys

import pytest

from vpic_amd import _lib
from vpic_amd import types as T

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _header(fn):
    src = open(os.path.join(ROOT, "include", fn)).read()
    return re.sub(r"/\*.*?\*/", "", src, flags=re.S)


def _declared(fn="vpic_hip.h"):
    return sorted(set(re.findall(r"\b(vpic_hip_\w+)\s*\(", _header(fn))))


# The reference-named functions of vpic_dropin.h (function declarations:
# a return type, the name, an argument list ending in ");").
DROPIN_NAMES = sorted(set(re.findall(
    r"^(?:void|int|double)\s+(\w+)\s*\([^;]*\);", _header("vpic_dropin.h"),
    flags=re.M)))


def test_library_loads():
    lib = _lib.load()
    assert b"gfx950" in lib.vpic_hip_version()


@pytest.mark.parametrize("name", _declared() + DROPIN_NAMES)
def test_symbol_exported(name):
    lib = _lib.load()
    assert hasattr(lib, name), name


def test_dropin_declares_reference_kernels():
    for name in ("advance_p", "sort_p", "move_p", "energy_p",
                 "accumulate_rho_p", "center_p", "uncenter_p",
                 "load_interpolator_array", "clear_accumulator_array",
                 "reduce_accumulator_array", "unload_accumulator_array",
                 "vpic_hip_install_field_kernels"):
        assert name in DROPIN_NAMES, name


def test_binding_covers_header():
    assert set(_declared()) <= set(_lib.EXPORTS) | {"vpic_hip_version"}


def test_dropin_header_in_c(tmp_path):
    """vpic_dropin.h compiles as C99, and the library's layout table agrees
    with the header's own types (no device needed)."""
    src = tmp_path / "t.c"
    src.write_text(
        '#include "vpic_dropin.h"\n#include "vpic_dropin_layout.h"\n'
        "#include <stdio.h>\n"
        "int main(void) {\n"
        "  const int64_t mine[] = {VPIC_DROPIN_LAYOUT(VPIC_DROPIN_SIZE,"
        " VPIC_DROPIN_OFFSET)};\n"
        "  int64_t lib[512];\n"
        "  int n = (int)(sizeof mine / sizeof mine[0]);\n"
        "  int c = vpic_hip_dropin_layout(lib, 512);\n"
        "  if (c != n) return 2;\n"
        "  for (int k = 0; k < n; k++) if (lib[k] != mine[k]) return 3;\n"
        "  printf(\"%d\\n\", n);\n  return 0;\n}\n")
    exe = tmp_path / "t"
    libdir = os.path.dirname(_lib.LIB_PATH)
    subprocess.run(["gcc", "-std=c99", "-Wall", "-Werror", "-I",
                    os.path.join(ROOT, "include"), str(src), "-o", str(exe),
                    "-L" + libdir, "-l:libvpichip.so",
                    "-Wl,-rpath," + libdir, "-Wl,-rpath,/opt/rocm/lib"],
                   check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out
    assert int(out.stdout) > 150


REF_CHECK = os.path.join(ROOT, "oracle", "_ref", "dropin_check")


@pytest.mark.ref
@pytest.mark.skipif(not os.path.exists(REF_CHECK),
                    reason="oracle/_ref (reference build) not present")
def test_dropin_layout_matches_reference_headers():
    """A program compiled against lanl/vpic's own headers sees the same
    sizes and offsets as the library."""
    out = subprocess.run([REF_CHECK, "--layout"], capture_output=True,
                         text=True)
    assert out.returncode == 0, out.stdout + out.stderr
    assert "ok layout" in out.stdout


def test_grid_helper_matches_reference_math():
    g1 = T.Grid()
    _lib.call("vpic_hip_grid_periodic", ctypes.byref(g1), 0.0, 0.0, 0.0,
              32.0, 16.0, 8.0, 32, 16, 8, 0.5, 1.0, 1.0)
    g2 = T.grid_periodic(0, 0, 0, 32, 16, 8, 32, 16, 8, 0.5)
    assert bytes(g1) == bytes(g2)


def test_bad_args_rejected():
    lib = _lib.load()
    g = T.grid_periodic(0, 0, 0, 4, 4, 4, 4, 4, 4, 0.5)
    nm = ctypes.c_int32()
    # NULL accumulator / interpolator
    rc = lib.vpic_hip_advance_p(None, 0, -1.0, 1.0, None, 0,
                                ctypes.byref(nm), None, None, None,
                                ctypes.byref(g), None, None)
    assert rc < 0 and b"NULL" in lib.vpic_hip_last_error()
    # inconsistent strides
    bad = g.copy()
    bad.sy += 1
    rc = lib.vpic_hip_advance_b(ctypes.c_void_p(16), ctypes.byref(bad), 0.5,
                                None)
    assert rc < 0 and b"strides" in lib.vpic_hip_last_error()
    # advance_e frac != 1 (vacuum_advance_e_pipeline.cc:58-61)
    mp = T.vacuum_params()
    rc = lib.vpic_hip_vacuum_advance_e(ctypes.c_void_p(16), ctypes.byref(g),
                                       ctypes.byref(mp), 0.5, None)
    assert rc < 0 and b"frac" in lib.vpic_hip_last_error()
    # absorbing field faces are not supported
    ab = g.copy()
    ab.fbc[0] = ab.fbc[3] = T.BC_ABSORB_FIELDS
    rc = lib.vpic_hip_advance_b(ctypes.c_void_p(16), ctypes.byref(ab), 0.5,
                                None)
    assert rc < 0 and b"absorbing" in lib.vpic_hip_last_error()
    # one-sided periodic axis
    one = g.copy()
    one.pbc[0] = T.BC_REFLECT_PARTICLES
    rc = lib.vpic_hip_sort_p(ctypes.c_void_p(16), ctypes.c_void_p(32), 1,
                             ctypes.c_void_p(64), ctypes.byref(one), 1, None)
    assert rc < 0 and b"partner" in lib.vpic_hip_last_error()


def test_species_push_args_rejected():
    """vpic_hip_advance_p_species checks its species before any device
    work: a count outside 1..2, and two species sharing a per-species
    output (dev_nm counters, movers, keys)."""
    lib = _lib.load()
    g = T.grid_periodic(0, 0, 0, 4, 4, 4, 4, 4, 4, 0.5)
    v = ctypes.c_void_p
    arr = (T.PushSpecies * 2)(
        T.PushSpecies(16, 8, -1.0, 1.0, 4096, 8, 8192, None, None),
        T.PushSpecies(32, 8, 1.0, 25.0, 4096 * 3, 8, 8192, None, None))
    rc = lib.vpic_hip_advance_p_species(3, arr, v(64), v(128),
                                        ctypes.byref(g), None)
    assert rc < 0 and b"species in one advance_p" in lib.vpic_hip_last_error()
    rc = lib.vpic_hip_advance_p_species(2, arr, v(64), v(128),
                                        ctypes.byref(g), None)
    assert rc < 0 and b"dev_nm" in lib.vpic_hip_last_error()
    arr[1].dev_nm = 8192 + 64
    arr[1].pm = 4096
    rc = lib.vpic_hip_advance_p_species(2, arr, v(64), v(128),
                                        ctypes.byref(g), None)
    assert rc < 0 and b"mover array" in lib.vpic_hip_last_error()
    arr[1].pm = 4096 * 3
    arr[0].keys = arr[1].keys = 1 << 20
    rc = lib.vpic_hip_advance_p_species(2, arr, v(64), v(128),
                                        ctypes.byref(g), None)
    assert rc < 0 and b"key array" in lib.vpic_hip_last_error()


def test_neighbor_table_matches_oracle(orc):
    import numpy as np
    from oracle.oracle import neighbor_table
    g = T.grid_periodic(0, 0, 0, 4, 5, 6, 4, 5, 6, 0.5)
    g.pbc[0] = g.pbc[3] = T.BC_REFLECT_PARTICLES
    g.pbc[2] = g.pbc[5] = T.BC_ABSORB_PARTICLES
    nb = np.zeros(6 * g.nv, dtype=np.int64)
    _lib.call("vpic_hip_grid_neighbor_table", ctypes.byref(g),
              nb.ctypes.data_as(ctypes.c_void_p))
    assert np.array_equal(nb, neighbor_table(g))


def test_field_step_rejects_what_the_separate_calls_do():
    """NULL or misaligned arrays, inconsistent strides, absorbing faces."""
    lib = _lib.load()
    g = T.grid_periodic(0, 0, 0, 4, 4, 4, 4, 4, 4, 0.5)
    mp = T.vacuum_params()

    def step(f, a, fi, work, grid=g):
        vp = ctypes.c_void_p
        return lib.vpic_hip_field_step(vp(f), vp(a), vp(fi), vp(work),
                                       ctypes.byref(grid), ctypes.byref(mp),
                                       None)

    for bad in [(None, 16, 16, 16), (16, None, 16, 16), (16, 16, None, 16),
                (20, 16, 16, 16), (16, 16, 20, 16), (16, 16, 16, 20)]:
        assert step(*bad) < 0
        assert b"argument" in lib.vpic_hip_last_error(), bad
    g2 = g.copy()
    g2.sy += 1
    assert step(16, 16, 16, 16, g2) < 0
    assert b"strides" in lib.vpic_hip_last_error()
    g3 = g.copy()
    g3.fbc[0] = g3.fbc[3] = T.BC_ABSORB_FIELDS
    assert step(16, 16, 16, 16, g3) < 0
    assert b"absorbing" in lib.vpic_hip_last_error()


def _push_tile(n, np_, walls=False):
    g = T.grid_periodic(0, 0, 0, *n, *n, 0.5)
    if walls:
        g.fbc[0] = g.fbc[3] = T.BC_PEC_FIELDS
        g.pbc[0] = g.pbc[3] = T.BC_REFLECT_PARTICLES
    out, k = (ctypes.c_int32 * 12)(), ctypes.c_int32()
    _lib.call("vpic_hip_push_tile_choices", ctypes.byref(g), int(np_), out,
              ctypes.byref(k))
    return [tuple(out[4 * j:4 * j + 4]) for j in range(k.value)]


def test_push_tile_saved_and_restored():
    """What the getter gives restores the push's own choice as well as a tile
    that was set; a tile that is refused changes nothing."""
    was, now = (ctypes.c_int32 * 4)(), (ctypes.c_int32 * 4)()
    _lib.call("vpic_hip_push_tile", 0, 0, 0)
    small, large = _push_tile((12, 10, 9), 20000), \
        _push_tile((256, 128, 128), 8 * 10 ** 8)
    assert small != [(7, 8, 7, 1)] and large == [(7, 8, 7, 1)]
    _lib.call("vpic_hip_push_get_tile", was)
    assert tuple(was) == (0, 0, 0, 1)
    _lib.call("vpic_hip_push_tile_window", *was)
    assert _push_tile((12, 10, 9), 20000) == small
    _lib.call("vpic_hip_push_tile_window", 7, 8, 7, 1)
    assert _push_tile((12, 10, 9), 20000) == [(7, 8, 7, 1)]
    _lib.call("vpic_hip_push_get_tile", now)
    assert tuple(now) == (7, 8, 7, 1)
    with pytest.raises(_lib.VpicError):
        _lib.call("vpic_hip_push_tile", 0, 8, 7)
    assert _push_tile((5, 3, 2), 100) == [(5, 3, 2, 1)]
    _lib.call("vpic_hip_push_tile_window", *was)
    assert _push_tile((12, 10, 9), 20000) == small


def test_push_tile_choice_costs_little():
    """A run asks for its tile at every push: with particle numbers that drift
    and species that go in pairs of several totals it neither searches anew
    (20 to 55 us) nor changes the shape from step to step."""
    import time
    _lib.call("vpic_hip_push_tile", 0, 0, 0)
    g = T.grid_periodic(0, 0, 0, 32, 32, 32, 32, 32, 32, 0.5)
    out, k = (ctypes.c_int32 * 12)(), ctypes.c_int32()
    fn = _lib.load().vpic_hip_push_tile_choices
    ref = ctypes.byref(g), ctypes.byref(k)
    seen = set()
    fn(ref[0], 1000000, out, ref[1]), fn(ref[0], 2000000, out, ref[1])
    t0 = time.process_time()
    for step in range(2000):
        for np_ in (1000000 + step, 2000000 - 3 * step):
            fn(ref[0], np_, out, ref[1])
            seen.add(tuple(out[:3]))
    # (4000 searches: 0.08 to 0.2 s; 4000 calls that find an answer: 0.006 s)
    assert time.process_time() - t0 < 0.04
    assert len(seen) <= 2


def test_push_tiles_for_dense_regions():
    """Where the tile for a uniform plasma is larger than 7x8x7 cut to the
    grid, so that a dense region would fall on fewer CUs, the push has smaller
    ones to take; walls make no difference."""
    _lib.call("vpic_hip_push_tile", 0, 0, 0)
    for n, ppc in (((512, 1, 257), 96), ((256, 1, 256), 128),
                   ((300, 200, 1), 80), ((1, 300, 200), 80),
                   ((128, 1, 128), 128)):
        t = _push_tile(n, ppc * n[0] * n[1] * n[2])
        cells = [a * b * c for a, b, c, _ in t]
        assert cells[0] > 49 and cells == sorted(cells, reverse=True)
        assert cells[-1] <= 64 and len(t) >= 2
        assert _push_tile(n, ppc * n[0] * n[1] * n[2], True) == t
    # 7x8x7 where few or no tiles are saved: cut tiles in a second round of
    # CUs, whole tiles in one more round
    for n, ppc in (((63, 25, 53), 64), ((256, 32, 32), 64),
                   ((13, 183, 35), 224), ((29, 117, 153), 46)):
        assert _push_tile(n, ppc * n[0] * n[1] * n[2]) == [(7, 8, 7, 1)]
    # a cut tile that would wait for a whole one on its die
    assert _push_tile((178, 20, 20), 184 * 178 * 400) != [(7, 10, 4, 1)]
    n = (100, 3, 100)
    t = _push_tile(n, 134 * n[0] * n[1] * n[2])[0]
    assert -(-100 // t[0]) * -(-100 // t[2]) <= 256
    for n, ppc in (((12, 10, 9), 16), ((32, 32, 32), 128), ((64, 1, 64), 128),
                   ((97, 61, 83), 40), ((256, 128, 128), 200)):
        assert len(_push_tile(n, ppc * n[0] * n[1] * n[2])) == 1


def test_adjoint_workspace_of_any_checkpoint_interval():
    """An interval past the run's end, up to the largest int, is the run's
    length: as much memory as one segment takes."""
    g = T.grid_periodic(0, 0, 0, 4, 4, 4, 4, 4, 4, 0.5)
    need = ctypes.c_int64()

    def bytes_for(steps, ckpt):
        _lib.call("vpic_hip_adjoint_workspace", 100, ctypes.byref(g), steps,
                  ckpt, 4, 1, ctypes.byref(need))
        return need.value
    for ckpt in (11, 20, 2 ** 31 - 9, 2 ** 31 - 1, 0, -1):
        assert bytes_for(10, ckpt) == bytes_for(10, 10)
    assert bytes_for(10, 4) < bytes_for(10, 10)


def test_adjoint_lists_beyond_the_hosts_memory():
    """A run whose lists of checkpoints do not fit the host's memory is an
    error, not an exception through the C entry (which ends the process)."""
    code = """
import ctypes, resource, sys
sys.path.insert(0, %r)
from vpic_amd import _lib, types as T
g = T.grid_periodic(0, 0, 0, 4, 4, 4, 4, 4, 4, 0.5)
n = ctypes.c_int64()
_lib.load()
size = int(open("/proc/self/statm").read().split()[0]) * 4096
resource.setrlimit(resource.RLIMIT_AS, (size + (1 << 30),) * 2)
try:
    _lib.call("vpic_hip_adjoint_workspace", 100, ctypes.byref(g), 2 ** 31 - 1,
              1, 4, 1, ctypes.byref(n))
except _lib.VpicError as e:
    print("refused:", e)
""" % ROOT
    out = subprocess.run([sys.executable, "-c", code], capture_output=True,
                         text=True, timeout=120)
    assert out.returncode == 0 and "refused" in out.stdout, out.stderr
