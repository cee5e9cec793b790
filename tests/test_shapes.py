"""Index and shape arithmetic of csrc/sifv_shapes.hpp, compiled here with the host
compiler: the LDS rings of the marching kernels, the rule that picks
stage tiles, the bound of the IGR strips' waits and
their period and record slots, the planes a thread of the fine restriction walks."""
import ctypes as C
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "semiimplicitfv_amd", "csrc")
SHIM = """
#include "sifv_shapes.hpp"
extern "C" {
int ring_slot(int row, int n) { return sifv::ring_slot(row, n); }
int first_ring_row(int R) { return sifv::first_ring_row(R); }
int tile_waves(int nx, int ny, int nph, int fp32) { return sifv::tile_waves_of(nx, ny, nph, fp32 != 0); }
int tile_blocks(int nx, int ny, int tw) { return sifv::tile_shape_of(nx, ny, tw).blocks(1); }
int scratch_partials() { return sifv::kScratchPartials; }
long long strip_wait_ticks(int khz) { return sifv::strip_wait_ticks(khz); }
void strip_period(int ny, int W, int perX, int* p) {
    const sifv::StripPeriod s = sifv::strip_period(ny, W, perX != 0);
    p[0] = s.period;
    p[1] = s.slots;
}
int restrict_planes(int nx, int ny, int nz) { return sifv::restrict_planes(nx, ny, nz); }
int stress_partials() { return sifv::kStressPartials; }
}
"""


@pytest.fixture(scope="module")
def shapes(tmp_path_factory):
    d = tmp_path_factory.mktemp("shapes")
    src, out = d / "shim.cpp", d / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", CSRC, "-o", str(out), str(src)], check=True)
    lib = C.CDLL(str(out))
    lib.strip_wait_ticks.restype = C.c_longlong
    return lib


@pytest.mark.parametrize("R", [1, 2, 3])
def test_ring_slots_in_range_and_distinct(shapes, R):
    """Rows -2 + R (warm-up rows of the first segment enter two rows early) and up; the
    z march enters its first plane one row earlier.  Any R + 1 rows in a row, the ones
    between entering the ring and their update, have slots of their own."""
    n = R + 1
    assert shapes.first_ring_row(R) == R - 2
    slots = [shapes.ring_slot(r, n) for r in range(R - 3, 40)]
    assert all(0 <= s < n for s in slots)
    assert all(len(set(slots[i:i + n])) == n for i in range(len(slots) - n + 1))


@pytest.mark.parametrize("nph,fp32", [(0, 0), (2, 0), (0, 1), (2, 1)])
def test_tiles_fit_the_allocation_free_partials(shapes, nph, fp32):
    """A mesh on tiles leaves dt partials enough for the allocation-free loop, as its
    march does (16384 waves and 2048 blocks of stress limits against 65536)."""
    cap, stress = shapes.scratch_partials(), shapes.stress_partials()
    tiled = 0
    for nx in list(range(1, 70)) + [500, 4000, 80000, 640000]:
        for ny in (1, 2, 9, 800, 5000, 300000, 360000, 507904, 524289, 600000, 640000):
            tw = shapes.tile_waves(nx, ny, nph, fp32)
            assert tw in (0, 4, 10)
            if tw:
                tiled += 1
                assert shapes.tile_blocks(nx, ny, tw) + stress <= cap, (nx, ny)
    assert (tiled == 0) == bool(nph and fp32)
    # the line is in tiles of 62 columns x 8 rows: full strips and strips of 8 columns alike
    line = 0 if nph and fp32 else 1280 if nph or fp32 else 768
    for nx, strips in ((8, 1), (62, 1), (63, 2), (496, 8)):
        ny = 8 * (line // strips)
        assert shapes.tile_waves(nx, max(ny, 1), nph, fp32) == (10 if line else 0)
        assert shapes.tile_waves(nx, ny + 8, nph, fp32) == 0


def test_strip_waits_are_bounded_by_time(shapes):
    """At least 20 s, so that a sweep whose strips wait for another stream's kernels is
    not given up, at the wall clock's 100 MHz and ten times that (more than 32 bits); a
    rate that the device does not tell counts as 100 MHz."""
    for khz in (100000, 1000000):
        assert 20.0 <= shapes.strip_wait_ticks(khz) / (khz * 1e3) <= 60.0
    assert shapes.strip_wait_ticks(0) == shapes.strip_wait_ticks(100000)


def test_strip_period_and_slots(shapes):
    """Slots for every row and for less than twice the rows, a period of whole multiples
    of them with room for the skew of all strips, at most 1/16 and a few steps more."""
    out = (C.c_int * 2)()
    for ny in list(range(152, 420)) + [1000, 1024, 2048, 4097, 8192, 20000]:
        for W in (1, 2, 3, 4, 11, 16, 64, 105, 128, 256):
            shapes.strip_period(ny, W, 0, out)
            assert tuple(out) == (ny, ny)
            shapes.strip_period(ny, W, 1, out)
            period, slots = out
            need = max(ny, 64 * W + 96)
            assert ny <= slots < 2 * ny and period % slots == 0
            assert need <= period <= need + max(period // slots, ny // 16)
    for (ny, W), want in {(1024, 16): (1120, 1120), (152, 64): (4212, 156), (200, 11): (800, 200)}.items():
        shapes.strip_period(ny, W, 1, out)
        assert tuple(out) == want


def test_restriction_walk(shapes):
    """Whole coarse cells, and no long walks while the mesh has few columns."""
    for n, want in {(24, 24, 24): 2, (48, 64, 40): 2, (90, 80, 70): 2, (128, 100, 96): 4, (160, 144, 176): 8,
                    (224, 224, 224): 16, (256, 256, 256): 16, (5, 3, 2): 2, (2000, 2000, 1): 16}.items():
        assert shapes.restrict_planes(*n) == want, n
