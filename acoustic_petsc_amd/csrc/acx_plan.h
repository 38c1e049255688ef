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

// Automatic z-chunk of a 2.5D march.  A launch runs in ceil(workgroups /
// slots) rounds (slots = CUs, or places for workgroups), each about as long
// as one workgroup's march of zc planes plus a fixed start of `start` planes'
// worth (z-halo planes, prologue); of the even divisions of the planes the one
// that minimises rounds x (zc + start) is taken, the longer march on a tie.
// Against a fixed list of 8 .. 128 planes: a walled FP64 step at 150 x 131 x
// 90 225 -> 151 us (32 planes left 135 workgroups on 256 CUs, 18 planes 225),
// a 32^3 WAVE2 step 34 -> 21 us (8 planes: 8 workgroups; 1 plane: 64), the
// FP32 step at 384^3 2.57 -> 2.50 ms (77 planes instead of 128); the same
// chunk as before at 256^3.
// pair > 0: a slot holds two workgroups, which then take `pair` times as long
// as one alone.  cost (may be null): of the chunk taken, in planes.
// Every launch comes through here, so only the about 2 sqrt(nz) different
// chunks are looked at, each at its smallest number of pieces.
inline int auto_zc(int ntx, int nty, int nz, int slots, int start, double *cost = nullptr, double pair = 0.0)
{
    int best = nz, z = nz;
    double best_cost = -1.0;
    for (;;) {
        const long long wg = (long long)ntx * nty * (((long long)nz + z - 1) / z);
        double rounds = (double)((wg + slots - 1) / slots);
        if (pair > 0.0) {
            const long long full = wg / (2LL * slots), rest = wg - full * 2 * slots;
            rounds = (double)full * pair + (rest == 0 ? 0.0 : rest <= slots ? 1.0 : pair);
        }
        const double c = rounds * ((double)z + start);
        if (best_cost < 0 || c < best_cost) {
            best_cost = c;
            best = z;
        }
        if (z <= 1) break;
        const long long pieces = ((long long)nz + z - 2) / (z - 1);   // the fewest with a shorter chunk
        z = (int)((nz + pieces - 1) / pieces);
    }
    if (cost) *cost = best_cost;
    return best;
}

// Kernel of one leapfrog update.  2D and 1D programs (an axis of one cell): a
// thread per cell.  3D: the LDS-DMA march where x is even and the arrays it
// copies (POLD, P, C: `in`, their addresses or'ed) are 16-byte aligned, else the
// register march.  Up to CTCS_PAIR_CELLS and with PNEW (`out`) aligned too, a
// thread per pair of cells with its 16-byte store (four arrays of 80 MB together,
// which stay in the caches between steps).  us per update, DMA march and pairs:
// 48^3 6.8 / 3.3, 64^3 7.1 / 3.9, 100^3 11.7 / 7.8, 128^3 15.6 / 14.4, 160^3 24.2 /
// 26.2, 256^3 108 / 132.
enum { CTCS_CELLS, CTCS_MARCH, CTCS_DMA, CTCS_PAIRS };
constexpr uint64_t CTCS_PAIR_CELLS = 2500000;

constexpr int ctcs_route(int nx, int ny, int nz, uintptr_t in, uintptr_t out)
{
    if (nx < 5 || ny < 5 || nz < 5) return CTCS_CELLS;
    if (nx % 2 != 0 || in % 16 != 0 || (uint64_t)nx * (uint64_t)ny >= 0xffffffffu) return CTCS_MARCH;
    return (uint64_t)nx * (uint64_t)ny * (uint64_t)nz <= CTCS_PAIR_CELLS && out % 16 == 0 ? CTCS_PAIRS : CTCS_DMA;
}

} // namespace acx
