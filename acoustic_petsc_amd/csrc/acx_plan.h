// acx_plan.h -- index and launch rules in plain C++: what the kernels and their
// launchers compute from sizes alone, usable without a device.
#pragma once
#include <stdint.h>

namespace acx {

constexpr int kNumXcd = 8;   // XCDs of the device, each with an L2 of its own

// Stages of a compensated FP32 step by what they read: no increment yet, the
// increment, the increment and the state the step ends in.
enum { F32_FIRST = 0, F32_MID = 1, F32_LAST = 2 };

// Index i of a periodic axis of n cells, from anywhere outside it.
constexpr int wrap(int i, int n)
{
    const int r = i % n;
    return r < 0 ? r + n : r;
}

// Cell of a plane (nx x ny, periodic) at row r, column c of the staged region
// of the tile at (x0, y0), which starts `halo` cells before it.  The region of
// a tile at the grid's edge reaches more than one grid length past it where an
// axis is shorter than a tile; every cell it names exists.
constexpr uint32_t region_cell(int x0, int y0, int halo, int r, int c, int nx, int ny)
{
    return (uint32_t)wrap(y0 - halo + r, ny) * (uint32_t)nx + (uint32_t)wrap(x0 - halo + c, nx);
}

// Whether a plane's byte offsets (cells of cell_bytes) need more than the 32
// bits the all-periodic marches keep them in.
constexpr bool plane_beyond_32_bits(int nx, int ny, int cell_bytes)
{
    return (uint64_t)nx * (uint64_t)ny * (uint64_t)cell_bytes > 0xffffffffu;
}

} // namespace acx
