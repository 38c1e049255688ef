"""The index and launch rules of csrc/acx_plan.h, compiled for the host: what a
kernel reads and what a launcher chooses, from sizes alone.  Each case is a
small program that says nothing when the rule holds.
"""
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "acoustic_petsc_amd", "csrc")

PROLOGUE = """
#include <cstdio>
#include <cstdlib>
#include <initializer_list>
#include "acx_plan.h"
using namespace acx;
#define CHECK(c, ...) do { if (!(c)) { std::printf(__VA_ARGS__); std::printf("\\n"); std::exit(1); } } while (0)
"""


@pytest.fixture
def run_host(tmp_path):
    def run(body, timeout=60):
        src, exe = tmp_path / "t.cpp", tmp_path / "t"
        src.write_text(PROLOGUE + body)
        subprocess.run(["g++", "-std=c++17", "-O2", "-Wall", "-Werror", f"-I{CSRC}", str(src), "-o", str(exe)], check=True)
        r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=timeout)
        assert r.returncode == 0 and r.stdout == "", r.stdout
    return run


# tile and halo of the FP64 LDS-DMA march and of the judge of the selective step
@pytest.mark.parametrize("bx, by, halo", [(32, 16, 3), (32, 8, 2)])
def test_staged_regions_name_cells_of_the_plane(bx, by, halo, run_host):
    """Every cell of every tile's region exists, and the cells a stencil needs
    (up to `halo` around a column of the grid) are the periodic ones."""
    run_host(f"""
int main()
{{
    const int bx = {bx}, by = {by}, h = {halo};
    for (int nx = 1; nx <= 70; ++nx)
        for (int ny = 1; ny <= 70; ++ny)
            for (int y0 = 0; y0 < ny; y0 += by)
                for (int x0 = 0; x0 < nx; x0 += bx)
                    for (int r = 0; r < by + 2 * h; ++r)
                        for (int c = 0; c < bx + 2 * h; ++c) {{
                            const uint32_t q = region_cell(x0, y0, h, r, c, nx, ny);
                            CHECK(q < (uint32_t)(nx * ny), "%d x %d, tile %d %d, row %d column %d: cell %u", nx, ny, x0, y0, r, c, q);
                            const int x = x0 - h + c, y = y0 - h + r;
                            CHECK(((int)(q % nx) - x) % nx == 0 && ((int)(q / nx) - y) % ny == 0, "%d x %d: %d %d -> %u", nx, ny, x, y, q);
                        }}
}}
""")


@pytest.mark.parametrize("fit", [(512, 256), (256, 512), (3, 7), (1, 8), (77, 304)])
def test_ensemble_lists_hold_every_item_once(fit, run_host):
    """Launched with the workgroups its schedule is made for, each stage runs
    every (problem, tile, z-chunk) exactly once, and the items cover the grids."""
    run_host(f"""
#include <set>
#include "acx_ensemble_plan.h"
int main()
{{
    const std::vector<int> dims = {{64, 96, 128, 4, 4, 4, 65, 9, 31, 160, 64, 5, 7, 130, 257}};
    const std::vector<size_t> off = {{0, 1, 2, 3, 4}};
    const int fit[2] = {{{fit[0]}, {fit[1]}}};
    for (int by : {{8, 12}})
        for (int zc : {{16, 32, 64, 128}}) {{
            const EnsPlan plan = ens_plan(ens_problems(dims, off, {{by, zc}}), fit);
            long cells = 0;
            for (const EnsProblem &q : plan.probs) {{
                CHECK(q.ntx * ENS_BX >= q.n[0] && q.nty * by >= q.n[1] && q.ntz * q.zc >= q.n[2], "tiles short of the grid");
                CHECK((q.ntz - 1) * q.zc < q.n[2] && q.zc <= zc, "an empty or overlong chunk");
                cells += (long)q.ntx * q.nty * q.ntz;
            }}
            for (int stage : {{F32_FIRST, F32_MID, F32_LAST}}) {{
                const EnsSchedule &s = plan.schedule[ens_schedule_of(stage)];
                CHECK(s.blocks() == fit[ens_schedule_of(stage)], "stage %d: lists for %d workgroups", stage, s.blocks());
                std::set<std::pair<int, int>> seen;
                for (int b = 0; b < s.blocks(); ++b)
                    for (int k = s.first[b]; k < s.first[b + 1]; ++k) {{
                        const EnsItem i = s.items[k];
                        const EnsProblem &q = plan.probs[i.prob];
                        CHECK(i.tile >= 0 && i.tile < q.ntx * q.nty * q.ntz, "tile %d of problem %d", i.tile, i.prob);
                        CHECK(seen.insert({{i.prob, i.tile}}).second, "item twice");
                    }}
                CHECK((long)seen.size() == cells && s.items.size() == seen.size(), "stage %d: %zu of %ld items", stage, seen.size(), cells);
            }}
        }}
}}
""")


def test_plane_offsets_of_32_bits(run_host):
    """The largest byte offset inside a plane fits 32 bits where the rule says so."""
    run_host("""
#include "acx_ensemble_plan.h"
int main()
{
    CHECK(!plane_beyond_32_bits(16384, 16383, 16), "a plane below 2^32 bytes");
    CHECK(plane_beyond_32_bits(16384, 16384, 16) && plane_beyond_32_bits(16400, 16400, 16), "2^32 bytes and more");
    CHECK(plane_beyond_32_bits(2147483647, 4, 8) && !plane_beyond_32_bits(1 << 27, 3, 8), "long rows");
    CHECK(ens_wide({64, 64, 64, 16384, 16384, 4}) && !ens_wide({64, 64, 64, 16384, 16383, 4}), "any problem of a batch");
}
""")


def test_leapfrog_routes(run_host):
    """What each kernel form asks of sizes and alignment, and no more: the march
    that copies POLD, P and C stores 8 bytes at a time."""
    run_host("""
int main()
{
    CHECK(ctcs_route(100, 100, 100, 0x1000, 0x2000) == CTCS_PAIRS, "small and aligned");
    CHECK(ctcs_route(256, 256, 256, 0x1000, 0x2000) == CTCS_DMA, "large and aligned");
    CHECK(ctcs_route(256, 256, 256, 0x1000, 0x2008) == CTCS_DMA, "PNEW off alignment, large");
    CHECK(ctcs_route(100, 100, 100, 0x1000, 0x2008) == CTCS_DMA, "PNEW off alignment, small");
    CHECK(ctcs_route(256, 256, 256, 0x1008, 0x2000) == CTCS_MARCH, "POLD, P or C off alignment");
    CHECK(ctcs_route(255, 256, 256, 0, 0) == CTCS_MARCH && ctcs_route(101, 100, 100, 0, 0) == CTCS_MARCH, "odd rows");
    CHECK(ctcs_route(256, 256, 1, 0, 0) == CTCS_CELLS && ctcs_route(256, 1, 1, 0, 0) == CTCS_CELLS, "2D, 1D");
}
""")


def test_z_chunk_is_the_best_even_division(run_host):
    """The chunk of the round model against all even divisions of the planes, and
    its cost on an axis of two thousand million planes (a launch's host time)."""
    run_host("""
static int all_divisions(int ntx, int nty, int nz, int slots, int start, double *cost, double pair)
{
    int best = nz, prev = 0;
    double best_cost = -1.0;
    for (int k = 1; k <= nz; ++k) {
        const int z = (nz + k - 1) / k;
        if (z == prev) continue;
        prev = z;
        const long long wg = (long long)ntx * nty * ((nz + z - 1) / z);
        double rounds = (double)((wg + slots - 1) / slots);
        if (pair > 0.0) {
            const long long full = wg / (2LL * slots), rest = wg - full * 2 * slots;
            rounds = (double)full * pair + (rest == 0 ? 0.0 : rest <= slots ? 1.0 : pair);
        }
        const double c = rounds * (z + start);
        if (best_cost < 0 || c < best_cost) best_cost = c, best = z;
    }
    *cost = best_cost;
    return best;
}

int main()
{
    for (int nz = 1; nz <= 520; nz += nz < 130 ? 1 : 13)
        for (int ntx : {1, 2, 5, 9, 12, 65})
            for (int nty : {1, 3, 16, 26})
                for (int slots : {256, 512, 1024})
                    for (int start : {4, 10})
                        for (double pair : {0.0, 1.5}) {
                            double a, b;
                            const int z = auto_zc(ntx, nty, nz, slots, start, &a, pair);
                            const int w = all_divisions(ntx, nty, nz, slots, start, &b, pair);
                            CHECK(z == w && a == b, "%d planes, %d x %d tiles, %d slots: %d (%g), best %d (%g)", nz, ntx, nty, slots, z, a, w, b);
                        }
    CHECK(auto_zc(1, 1, 2000000000, 256, 10) == 7812500, "a long axis");
}
""", timeout=10)
