"""Index and shape arithmetic of csrc/sifv_shapes.hpp, compiled here with the host
compiler: the LDS rings of the marching kernels."""
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
}
"""


@pytest.fixture(scope="module")
def shapes(tmp_path_factory):
    d = tmp_path_factory.mktemp("shapes")
    src, out = d / "shim.cpp", d / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", CSRC, "-o", str(out), str(src)], check=True)
    return C.CDLL(str(out))


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
