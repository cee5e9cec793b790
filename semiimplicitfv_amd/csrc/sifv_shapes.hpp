// sifv_shapes.hpp - index and shape arithmetic shared by kernels and host code.
// Standard C++ only, so that tests compile it with the host compiler.
#pragma once

#include <algorithm>

namespace sifv {

// Slot of a row (or plane) in a ring of n; the warm-up rows of a march start at
// -2, so a row may be as low as -n.
constexpr int ring_slot(int row, int n) { return (row + n) % n; }

// First row (plane) a march puts into its ring of R + 1: row + R of the first
// warm-up row of the first segment.
constexpr int first_ring_row(int R) { return -2 + R; }

constexpr int kOwn = 62;  // owned columns per wave in the x-marching and tile kernels
constexpr int kTileSmall = 4, kTileWaves = 10;  // waves per workgroup of the 2D tile kernel

// dt block minima: room of the allocation-free time loop (512 KiB of FP64), and
// the most that the stress limits' reduction adds to a stage's own.
constexpr int kScratchPartials = 65536;
constexpr int kStressPartials = 2048;

// Decomposition of a stage: strips of kOwn columns x segments of `rows` rows, a
// wave each (a workgroup of tileWaves waves where that is not 0).
struct StageShape {
    int nstrip, nseg, rows, tileWaves;
    int blocks(int planes) const { return nstrip * nseg * planes; }
};

inline StageShape march_shape_of(int dim, int nx, int ny, int nz, int rowsOverride) {
    const int nstrip = (nx + kOwn - 1) / kOwn;
    if (dim == 1) return StageShape{nstrip, 1, 1, 0};
    const long planes = dim == 3 ? nz : 1;
    int rows = rowsOverride;
    if (rowsOverride <= 0) {
        // aim for >= ~8k waves so every CU holds several waves (2D: ~16k,
        // 16 rows per wave at 4096^2, the fastest of 8..128 rows measured for
        // both the FP64 and the FP32-bulk kernels); meshes too small for 8 rows
        // per wave at that count get about one wave per SIMD slot (3072 at three
        // waves per SIMD) with 4..8 rows, trading the 2-row warm-up against
        // filling the chip (1024^2: 6 rows, measured fastest of 4..16)
        const long target = dim == 2 ? 16384 : 8192;
        const long cols = (long)ny * nstrip * planes;
        const long r = cols / target;
        if (r >= 8) {
            rows = 8;
            while (rows < 64 && rows * 2 <= r) rows *= 2;
        } else {
            rows = (int)std::max<long>(4, std::min<long>(8, (cols + 3071) / 3072));
        }
    }
    rows = std::min(rows, ny);
    return StageShape{nstrip, (ny + rows - 1) / rows, rows, 0};
}

inline StageShape tile_shape_of(int nx, int ny, int waves) {
    const int rows = waves - 2;
    return StageShape{(nx + kOwn - 1) / kOwn, (ny + rows - 1) / rows, rows, waves};
}

// Waves per workgroup of the 2D tile kernel (sifv_tile.hpp) for an explicit
// stage, or 0 for the marching kernel.  Meshes whose marching waves cannot fill
// the chip take tiles: a wave's serial chain of 6 rows costs 22 us there, a
// tile 11 us (128^2 FP64; 128^2 water/air 44 -> 16 us, FP32 21 -> 10 us).  The
// line is where the 256 CUs take one more round of tiles than that is worth, and
// lies in tiles, not in cells: a strip of 8 columns costs what one of 62 does.
// us a step of 3 stages, tiles against march, with the number of 8-row tiles:
//   FP64       752: 83 / 97 (190x1500),  720: 83 / 97 (576^2),  810: 98 / 97
//              (5000x80),  880: 104 / 98 (640^2),  2500: 249 / 178 (8x20000)
//   FP32       1222: 76 / 89 (750^2),  1300: 89 / 90 (800^2),  2500: 160 / 124
//   water/air  1222: 232 / 267 (750^2),  1250: 234 / 264 (63x5000),  1300: 274 / 271
//              and with LF 284 / 273 (800^2),  2125: 406 / 375 (1000^2),  2500: 453 /
//              400; below it 880: 187 / 182 (640^2) and 1000: 190 / 182 (80x4000) lose
// Small tiles (2 rows) while those of 8 rows would leave half the 256 CUs idle:
// 128^2 10.8 against 12.8 us a stage, 320^2 16.0 against 13.7.
inline int tile_waves_of(int nx, int ny, int nph, bool fp32) {
    if (fp32 && nph) return 0;
    const int blocks = tile_shape_of(nx, ny, kTileWaves).blocks(1);
    if (blocks > (fp32 || nph ? 1280 : 768)) return 0;
    return blocks < 128 ? kTileSmall : kTileWaves;
}

// Planes a thread of the multigrid's fine restriction walks (3D, FP64; a brick is 64
// columns x 8 rows): up to 16, to carry densities and vector up the column, as long as
// there are 600 bricks for the 256 CUs, and never less than the 2 of a coarse cell.
// us a launch with 2 / 4 / 8 / 16 planes, and of the form before the walk:
//   24^3            4.8 /   6.4 /   9.5 /  15.1,   5.3
//   48x64x40        5.4 /   7.3 /  10.5 /  16.9,   5.6
//   90x80x70        7.4 /   8.1 /   9.8 /  15.6,   5.7
//   128x100x96     12.4 /  11.9 /  13.7 /  18.3,  14.1
//   160x144x176    43.5 /  37.5 /  33.6 /  36.8,  53.8
//   224^3         158   / 135   / 125   / 127,    162
constexpr int restrict_planes(int nx, int ny, int nz) {
    const long columns = (long)((nx + 63) / 64) * ((ny + 7) / 8);
    int p = 16;
    while (p > 2 && columns * ((nz + p - 1) / p) < 600) p /= 2;
    return p;
}

// Longest wait of a strip of the IGR sweep for another one, 30 s, in ticks of a clock
// of `khz` (the device's wall clock: 100 MHz, also where the rate is not told).
constexpr long long strip_wait_ticks(int khz) { return 30LL * 1000 * (khz > 0 ? khz : 100000); }

// Period of the IGR strips' sweeps (steps from one sweep to the next) and record
// slots per strip, of which the period is a multiple.  On a wrapping x axis a sweep
// trails its wrap neighbour by the skew of all W strips (and 32 steps of margin), so
// a period of a mesh with fewer rows has idle rows.  They need no slots of their own:
// the period is split into as many runs of slots as it holds ny (a remainder up to
// ny / 16 short of one more counts as that one), so the slots stay below 2 ny and the
// period grows by less than a run's remainder, or by ny / 16.  4096 x 152: 156 slots
// and 4212 steps instead of 4192 of both, 31 MB of records instead of 824; slots of
// ny rows alone would cost 1024^2 a period of 2048 steps instead of 1120.
struct StripPeriod {
    int period, slots;
};
inline StripPeriod strip_period(int ny, int W, bool perX) {
    constexpr int lanes = 64, margin = 32;
    const int need = perX ? std::max(ny, W * lanes + lanes + margin) : ny;
    const int runs = (need + ny / 16) / ny;
    const int slots = std::max(ny, (need + runs - 1) / runs);
    return StripPeriod{runs * slots, slots};
}

}  // namespace sifv
