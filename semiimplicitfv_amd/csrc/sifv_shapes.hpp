// sifv_shapes.hpp - index and shape arithmetic shared by kernels and host code.
// Standard C++ only, so that tests compile it with the host compiler.
#pragma once

namespace sifv {

// Slot of a row (or plane) in a ring of n; the warm-up rows of a march start at
// -2, so a row may be as low as -n.
constexpr int ring_slot(int row, int n) { return (row + n) % n; }

// First row (plane) a march puts into its ring of R + 1: row + R of the first
// warm-up row of the first segment.
constexpr int first_ring_row(int R) { return -2 + R; }

}  // namespace sifv
