// acx_linear_core.h -- one tile of the fused linear-scheme stage (see
// acx_linear.hip for the method); shared by the per-grid kernel and the
// persistent ensemble kernel.
#pragma once
#include <type_traits>
#include "acx_device.h"
#include "acx_internal.h"
#include "acx_plan.h"

namespace acx {

// Epilogue kinds
enum { EPI_RHS = 0, EPI_AXPY = 1, EPI_COMB = 2, EPI_F32C = 3 };

// FP32 compensated stages.  One tile: columns [x0, x0+64) x [y0, y0+BY),
// planes [zb, ze) of the grid described by p (shared by the per-grid kernel and
// the ensemble kernel).  WALLS = false: every axis periodic (no ghost signs,
// wrap-only index maps).  STAGE: F32_FIRST no increment D yet; F32_MID reads
// HI and D, writes the next increment; F32_LAST also reads LO and writes the
// new (HI, LO).
//
// Lead-plane march: at iteration j the plane j is staged in LDS (own column
// and halo loaded for the same plane index as the neighbouring blocks load
// those rows as their interior, so shared rows meet in L2), its in-plane
// (x, y) part of the RHS is formed and kept, and plane j-3, whose
// z-neighbourhood j-6 .. j is now complete in registers, is finished and
// stored.
//
// The stage moves 32 to 80 bytes per cell and was bound by issue and by waits
// before it was bound by those bytes: per cell 175 FP32 and 67 move
// instructions.  Now about 135 and none:
// - the loop is unrolled by the 8 planes of the register ring, so no plane
//   ever moves between registers, and a load lands in the register that
//   keeps its plane;
// - the sums s_k = q(+k) + q(-k) over the axes are taken before the weights
//   (the differences of A7 likewise), in units of s/(48 h);
// - a cell is one 16-byte LDS entry (12 16-byte reads);
// - results are stored (STREAM: nontemporal, for fields beyond the last-level
//   cache) through a buffer descriptor per wavefront row, whose
//   bound drops the columns past the grid: without a branch around the store
//   the compiler can count it, and waits for a plane's loads alone instead of
//   for every load and store before them;
// - D of the last four planes waits in LDS for the epilogue, which leaves room
//   for 3 wavefronts per SIMD without spills.
// Measured at 384^3, us per stage (first, second and third, last) against the
// register-queue march it replaces: 475 -> 345, 590 -> 520, 857 -> 840 of
// 279, 418, 697 at the copy's rate; the step 2.51 -> 2.23 ms, at 256^3 0.72 ->
// 0.66 ms.  Its error against 64-bit steps is lower too (one step of
// ACOUSTIC4 7.7e-9 -> 7.4e-9, of WAVE2 7.9e-7 -> 7.3e-7).

template <int SYS, int BY>
struct Tile32 {
    static constexpr int BX = 64;
    static constexpr int NV = SYS == ACX_ACOUSTIC4 ? 4 : 2;   // components in memory
    static constexpr int NS = SYS == ACX_ACOUSTIC4 ? 4 : 1;   // components in the stencil
    static constexpr int LX = BX + 6, LY = BY + 6;
    static constexpr int NHALO = 6 * BX + 6 * BY;              // star stencil: no plane corners
    struct alignas(4 * NS) Entry { float v[NS]; };
    // the two planes being read and staged, and D of the last four planes of
    // every column (its own thread's only)
    struct Lds { Entry q[2][LY][LX]; };
    struct LdsD : Lds { Cell<float, NV> d[4][BY][BX]; };
    template <int STAGE> using Shared = typename std::conditional<STAGE == F32_FIRST, Lds, LdsD>::type;
};

typedef unsigned acx_u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned acx_u32x2 __attribute__((ext_vector_type(2)));

// Store of this lane's cell of a wavefront row (STREAM: nontemporal): row points
// at the row's first cell (wave-uniform), bytes bounds the cells that exist.
template <int NV, bool STREAM>
__device__ __forceinline__ void store_row(float *row, unsigned bytes, const Cell<float, NV> &c)
{
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(row, 0, (int)bytes, 0x00020000);
    const int off = (int)__lane_id() * NV * 4;
    if constexpr (NV == 4)
        __builtin_amdgcn_raw_buffer_store_b128(
            acx_u32x4{__float_as_uint(c.v[0]), __float_as_uint(c.v[1]), __float_as_uint(c.v[2]), __float_as_uint(c.v[3])},
            r, off, 0, STREAM ? 2 : 0);
    else
        __builtin_amdgcn_raw_buffer_store_b64(acx_u32x2{__float_as_uint(c.v[0]), __float_as_uint(c.v[1])}, r, off, 0, STREAM ? 2 : 0);
}

template <int SYS, int BY, int STAGE, bool WALLS, bool STREAM>
__device__ __forceinline__ void linear_tile32(const LinArgs &p, int x0, int y0, int zb,
                                              typename Tile32<SYS, BY>::template Shared<STAGE> &lds)
{
    using Tile = Tile32<SYS, BY>;
    constexpr int NV = Tile::NV, NS = Tile::NS, BX = Tile::BX;
    constexpr bool AC = SYS == ACX_ACOUSTIC4, HAS_D = STAGE != F32_FIRST, LAST = STAGE == F32_LAST;
    using C = Cell<float, NV>;
    static_assert(BX * BY >= Tile::NHALO, "every halo cell of a plane needs a thread of its own");

    const float *__restrict__ Q = static_cast<const float *>(p.q);
    const float *__restrict__ D = static_cast<const float *>(p.d);
    const float *__restrict__ LO = static_cast<const float *>(p.lo);
    const int nx = p.nx, ny = p.ny, nz = p.nz;
    const int tx = threadIdx.x, ty = __builtin_amdgcn_readfirstlane((int)threadIdx.y), tid = ty * BX + tx;
    const int ze = min(zb + p.zc, nz);
    const size_t plane = (size_t)nx * ny;
    const int bcx = WALLS ? p.bc[0] : 0, bcy = WALLS ? p.bc[1] : 0, bcz = WALLS ? p.bc[2] : 0;

    // own column
    float sgx = 1.f, sgy = 1.f;
    const int mx = map_axis(x0 + tx, nx, bcx, sgx);
    const int my = map_axis(y0 + ty, ny, bcy, sgy);
    const size_t col = (size_t)my * nx + mx;

    // halo cell of this thread (x halo for rows 0..BY-1, y halo for cols
    // 0..BX-1); threads without one load one cell per wavefront and write it
    // to the plane's unused corner, so that no branch holds back the loads
    int hx = 0, hy = 0;
    size_t hcol = (size_t)__builtin_amdgcn_readfirstlane(my) * nx + __builtin_amdgcn_readfirstlane(mx);
    float hsx = 1.f, hsy = 1.f;
    if (tid < Tile::NHALO) {
        int t = tid;
        if (t < 6 * BY) {            // x halo: 3 left, 3 right per row
            const int row = t / 6, k = t % 6;
            hy = row + 3;
            hx = k < 3 ? k : BX + k;  // 0,1,2 | BX+3..BX+5
        } else {
            t -= 6 * BY;
            const int colx = t % BX, k = t / BX;
            hx = colx + 3;
            hy = k < 3 ? k : BY + k;
        }
        const int gx = map_axis(x0 + hx - 3, nx, bcx, hsx);
        const int gy = map_axis(y0 + hy - 3, ny, bcy, hsy);
        hcol = (size_t)gy * nx + gx;
    }

    // Byte offsets inside a plane: 32 bits in the all-periodic instantiation
    // (taken when a plane is below 4 GB), so a load's address is a scalar
    // base and one register.
    using Off = typename std::conditional<WALLS, size_t, uint32_t>::type;
    const Off colb = (Off)(col * NV * 4), hcolb = (Off)(hcol * NV * 4);
    auto load = [](const float *plane_base, Off o) {
        return load_cell<float, NV>(reinterpret_cast<const float *>(reinterpret_cast<const char *>(plane_base) + o), 0);
    };
    // (load_cell_nt: nontemporal for the 16-byte cells of ACOUSTIC4 alone)
    auto load_lo = [&](size_t cell) { return STREAM ? load_cell_nt<float, NV>(LO, cell) : load_cell<float, NV>(LO, cell); };
    // the plane loaded next, its offset and its ghost sign
    int zi = 0;
    size_t zoff = 0;
    float zs = 1.f;
    auto seek = [&](int z) {
        zs = 1.f;
        zi = map_axis(z, nz, bcz, zs);
        zoff = (size_t)zi * plane * NV;
    };
    auto step = [&](int z) {   // from plane z - 1 to z
        if constexpr (WALLS) {
            seek(z);
        } else {
            ++zi;
            zoff = zi == nz ? 0 : zoff + plane * NV;
            zi = zi == nz ? 0 : zi;
        }
    };
    // this wavefront's row of the results
    const unsigned row_bytes = y0 + ty < ny ? (unsigned)min(BX, nx - x0) * NV * 4u : 0u;
    const size_t row0 = (size_t)(y0 + ty) * nx + x0;

    // Rings in registers, slot (plane - zb - 3) & 7; what is live at a time is
    // less than a ring.
    C q[8];                 // the column's planes j-6 .. j (HI + D, signed)
    C hi[8];                // HI of plane j+1 as loaded (F32_LAST: of planes j-3 .. j+1)
    C d;                    // D of plane j+1 (those of planes j-3 .. j wait in LDS, slot & 3)
    float xy[8][NS];        // in-plane parts of the RHS of planes j-3 .. j
    C hq, hd;               // halo cell of plane j+1
    C lo;                   // F32_LAST: LO of the plane to be finished next

    auto load_column = [&](C &qq, C &dd) {
        qq = load(Q + zoff, colb);
        if constexpr (HAS_D) dd = load(D + zoff, colb);
    };
    auto load_halo = [&](C &qq, C &dd) {
        qq = load(Q + zoff, hcolb);
        if constexpr (HAS_D) dd = load(D + zoff, hcolb);
    };
    auto value = [&](const C &a, const C &b, float sx, float sy, float sz) -> C {
        C c = a;
        if constexpr (HAS_D) {
#pragma unroll
            for (int v = 0; v < NV; ++v) c.v[v] += b.v[v];
        }
        if constexpr (WALLS) apply_bc_sign<float, NV>(c, sx, sy, sz);
        return c;
    };
    auto stage = [&](int buf, const C &own, const C &hq, const C &hd, float zs) {
        typename Tile::Entry e;
#pragma unroll
        for (int v = 0; v < NS; ++v) e.v[v] = own.v[v];
        lds.q[buf][ty + 3][tx + 3] = e;
        const C h = value(hq, hd, hsx, hsy, zs);
#pragma unroll
        for (int v = 0; v < NS; ++v) e.v[v] = h.v[v];
        lds.q[buf][hy][hx] = e;
    };
    // In-plane part without the centre's share.  The nearest neighbours, which
    // carry the largest weight, enter as differences from the centre q0 (exact
    // for smooth data): B7 = s3 - 6 s2 + 15 (s1 - 2 q0) + 10 q0 per axis, L7 =
    // -s3 + 2 s2 + 49 (s1 - 2 q0) - 2 q0.
    const float ks = float(p.K_s), rs = float(p.invrho_s);
    auto in_plane = [&](int buf, const C &q0, float (&o)[NS]) {
        float a[3];   // A7 sums: u along x plus v along y, p along x, p along y
        auto ring = [&](int k, float wB, float wA, bool first) {
            const typename Tile::Entry xp = lds.q[buf][ty + 3][tx + 3 + k], xm = lds.q[buf][ty + 3][tx + 3 - k];
            const typename Tile::Entry yp = lds.q[buf][ty + 3 + k][tx + 3], ym = lds.q[buf][ty + 3 - k][tx + 3];
            float s[NS];
#pragma unroll
            for (int v = 0; v < NS; ++v)
                s[v] = k == 1 ? ((xp.v[v] - q0.v[v]) + (xm.v[v] - q0.v[v])) + ((yp.v[v] - q0.v[v]) + (ym.v[v] - q0.v[v]))
                              : (xp.v[v] + xm.v[v]) + (yp.v[v] + ym.v[v]);
#pragma unroll
            for (int v = 0; v < NS; ++v) o[v] = first ? (AC ? s[v] : -s[v]) : fmaf(wB, s[v], o[v]);
            if constexpr (AC) {
                const float t[3] = {(xp.v[1] - xm.v[1]) + (yp.v[2] - ym.v[2]), xp.v[0] - xm.v[0], yp.v[0] - ym.v[0]};
#pragma unroll
                for (int c = 0; c < 3; ++c) a[c] = first ? t[c] : fmaf(wA, t[c], a[c]);
            }
        };
        // one ring of neighbours in registers at a time
        ring(3, 1.f, 1.f, true);
        asm volatile("" ::: "memory");
        ring(1, AC ? 15.f : 49.f, 37.f, false);
        asm volatile("" ::: "memory");
        ring(2, AC ? -6.f : 2.f, -8.f, false);
        if constexpr (AC) {
            o[0] = fmaf(-ks, a[0], o[0]);
            o[1] = fmaf(-rs, a[1], o[1]);
            o[2] = fmaf(-rs, a[2], o[2]);
        }
    };

    // prologue: planes zb-3 .. zb+2 and the halos of the last three all in
    // flight at once, then plane zb+3, then the in-plane parts
    {
        C dd[6], ph[3], pd[3];
        float sz[6];
        seek(zb - 3);
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            load_column(q[2 + k], dd[k]);
            if (k >= 3) load_halo(ph[k - 3], pd[k - 3]);
            sz[k] = zs;
            step(zb - 2 + k);
        }
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            if (k >= 3) {
                if constexpr (HAS_D) lds.d[(2 + k) & 3][ty][tx] = dd[k];
                hi[2 + k] = q[2 + k];
            }
            q[2 + k] = value(q[2 + k], dd[k], sgx, sgy, sz[k]);
        }
        load_column(hi[0], d);
        load_halo(hq, hd);
        if constexpr (LAST) lo = load_lo((size_t)zb * plane + col);
#pragma unroll
        for (int k = 3; k < 6; ++k) {
            stage(k & 1, q[2 + k], ph[k - 3], pd[k - 3], sz[k]);
            __syncthreads();
            in_plane(k & 1, q[2 + k], xy[2 + k]);
            // formed here, not when it is needed: the neighbours of three
            // planes at once would set the kernel's registers
#pragma unroll
            for (int v = 0; v < NS; ++v) asm volatile("" : "+v"(xy[2 + k][v]));
        }
    }

    // epilogue factors: the RHS in units of s/(48 h) (WAVE2: c^2/(48 h^2))
    // in two floats: rounded to one, a factor shifts every step the same way
    const double ccd = AC ? p.c * p.inv48h * p.s : p.c * p.lapc;
    const float cc = float(ccd), ccl = float(ccd - cc), cb = float(p.b), c1 = float(p.c), c1l = float(p.c - c1);
    const bool active = tx < nx - x0 && y0 + ty < ny;
    bool nfbad = false;   // non-finite watch of this thread's outputs

    // iteration of plane j = zb + 3 + u (mod 8): finishes plane c = j - 3
    auto body = [&](auto uu, int j) {
        constexpr int u = decltype(uu)::value, uc = (u + 5) & 7;
        q[u] = value(hi[u], d, sgx, sgy, zs);
        if constexpr (HAS_D) lds.d[u & 3][ty][tx] = d;
        const bool more = j < ze;   // planes ze .. ze+2 serve the z-stencils only
        if (more) stage(u & 1, q[u], hq, hd, zs);
        step(j + 1);
        load_column(hi[(u + 1) & 7], d);
        load_halo(hq, hd);
        if (more) {
            __syncthreads();
            in_plane(u & 1, q[u], xy[u]);
        } else {
#pragma unroll
            for (int v = 0; v < NS; ++v) xy[u][v] = 0.f;   // unused; ends the life of plane j-8's
        }
        const int c = j - 3;
        const C &zm3 = q[(u + 2) & 7], &zm2 = q[(u + 3) & 7], &zm1 = q[(u + 4) & 7], &q0 = q[uc];
        const C &zp1 = q[(u + 6) & 7], &zp2 = q[(u + 7) & 7], &zp3 = q[u];
        C o, dc;
        if constexpr (HAS_D) dc = lds.d[uc & 3][ty][tx];
        if constexpr (AC) {
            float r[4];
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const float s1 = (zp1.v[v] - q0.v[v]) + (zm1.v[v] - q0.v[v]);
                const float s2 = zp2.v[v] + zm2.v[v], s3 = zp3.v[v] + zm3.v[v];
                r[v] = xy[uc][v] + fmaf(15.f, s1, fmaf(30.f, q0.v[v], fmaf(-6.f, s2, s3)));
            }
            auto A = [&](int v) {
                const float t1 = zp1.v[v] - zm1.v[v], t2 = zp2.v[v] - zm2.v[v], t3 = zp3.v[v] - zm3.v[v];
                return fmaf(-8.f, t2, fmaf(37.f, t1, t3));
            };
            r[0] = fmaf(-ks, A(3), r[0]);
            r[3] = fmaf(-rs, A(0), r[3]);
#pragma unroll
            for (int v = 0; v < 4; ++v) o.v[v] = fmaf(cc, r[v], HAS_D ? fmaf(ccl, r[v], cb * dc.v[v]) : ccl * r[v]);
        } else {
            const float s1 = (zp1.v[0] - q0.v[0]) + (zm1.v[0] - q0.v[0]);
            const float s2 = zp2.v[0] + zm2.v[0], s3 = zp3.v[0] + zm3.v[0];
            const float r = xy[uc][0] + fmaf(49.f, s1, fmaf(-6.f, q0.v[0], fmaf(2.f, s2, -s3)));
            const float v = q0.v[1];   // du/dt = v (rhs_function.c:330)
            o.v[0] = fmaf(c1, v, HAS_D ? fmaf(c1l, v, cb * dc.v[0]) : c1l * v);
            o.v[1] = fmaf(cc, r, HAS_D ? fmaf(ccl, r, cb * dc.v[1]) : ccl * r);
        }
        const size_t out = ((size_t)c * plane + row0) * NV;
        if constexpr (LAST) {
            // HI' + LO' = HI + (LO + increment), exact
            C nh, nl;
#pragma unroll
            for (int v = 0; v < NV; ++v) two_sum(hi[uc].v[v], lo.v[v] + o.v[v], nh.v[v], nl.v[v]);
            store_row<NV, STREAM>(static_cast<float *>(p.out2) + out, row_bytes, nl);
            o = nh;
            lo = load_lo((size_t)min(c + 1, ze - 1) * plane + col);
        }
        store_row<NV, STREAM>(static_cast<float *>(p.out) + out, row_bytes, o);
        if constexpr (LAST) {
            C w = o;
#pragma unroll
            for (int v = 0; v < NV; ++v) w.v[v] = active ? o.v[v] : 0.f;
            finite_acc<float, NV>(nfbad, w);
        }
    };
    const int jend = ze + 2;
    for (int j = zb + 3;; j += 8) {
        body(std::integral_constant<int, 0>{}, j);
        if (j + 1 > jend) break;
        body(std::integral_constant<int, 1>{}, j + 1);
        if (j + 2 > jend) break;
        body(std::integral_constant<int, 2>{}, j + 2);
        if (j + 3 > jend) break;
        body(std::integral_constant<int, 3>{}, j + 3);
        if (j + 4 > jend) break;
        body(std::integral_constant<int, 4>{}, j + 4);
        if (j + 5 > jend) break;
        body(std::integral_constant<int, 5>{}, j + 5);
        if (j + 6 > jend) break;
        body(std::integral_constant<int, 6>{}, j + 6);
        if (j + 7 > jend) break;
        body(std::integral_constant<int, 7>{}, j + 7);
        if (j + 8 > jend) break;
    }
    watch_flush(p.nf, nfbad);
}

// Centre-plane march for FP64 ACOUSTIC4 fields beyond the last-level cache: the
// own column's z-queue holds planes z-3 .. z+3 before plane z is computed, and
// plane z (with its x/y halo) is staged in LDS and finished in the same
// iteration.  The halo of plane z+4 is loaded together with the column's plane
// z+4, i.e. at the iteration in which the neighbouring tiles load those cells
// as their interior, so the shared rows are still in L2; it waits in its slot
// of a 5-plane LDS ring until plane z+4 is computed.  Epilogue operands and
// results stream past L2 (nontemporal), leaving L2 to the stage input that
// neighbouring tiles re-read as halo.
struct LinTile {
    static constexpr int BX = 32, BY = 16, NV = 4;
    static constexpr int NHALO = 6 * BX + 6 * BY;              // star stencil: no plane corners
};

template <int EPI, bool WALLS>
__device__ __forceinline__ void linear_tile_centre(const LinArgs &p, int x0, int y0, int zb,
                                                   double (&lds)[5][LinTile::NV][LinTile::BY + 6][LinTile::BX + 6])
{
    using Tile = LinTile;
    constexpr int NV = Tile::NV, BX = Tile::BX, BY = Tile::BY;
    using C = Cell<double, NV>;
    static_assert(BX * BY >= Tile::NHALO, "every halo cell of a plane needs a thread of its own");

    const double *__restrict__ Q = static_cast<const double *>(p.q);
    const double *__restrict__ U0 = static_cast<const double *>(p.u0);
    double *__restrict__ OUT = static_cast<double *>(p.out);

    const int nx = p.nx, ny = p.ny, nz = p.nz;
    const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * BX + tx;
    const int ze = min(zb + p.zc, nz);
    const bool active = (x0 + tx < nx) && (y0 + ty < ny);
    const size_t plane = (size_t)nx * ny;
    const int bcx = WALLS ? p.bc[0] : 0, bcy = WALLS ? p.bc[1] : 0, bcz = WALLS ? p.bc[2] : 0;

    float sgx = 1.f, sgy = 1.f;
    const int mx = map_axis(x0 + tx, nx, bcx, sgx);
    const int my = map_axis(y0 + ty, ny, bcy, sgy);
    const size_t col = (size_t)my * nx + mx;

    int hx = -1, hy = -1;
    size_t hcol = 0;
    float hsx = 1.f, hsy = 1.f;
    if (tid < Tile::NHALO) {
        int t = tid;
        if (t < 6 * BY) {
            int row = t / 6, k = t % 6;
            hy = row + 3;
            hx = k < 3 ? k : BX + k;
        } else {
            t -= 6 * BY;
            int colx = t % BX, k = t / BX;
            hx = colx + 3;
            hy = k < 3 ? k : BY + k;
        }
        int gx = map_axis(x0 + hx - 3, nx, bcx, hsx);
        int gy = map_axis(y0 + hy - 3, ny, bcy, hsy);
        hcol = (size_t)gy * nx + gx;
    }
    struct Raw {
        C q;
        float s;
    };
    auto issue = [&](Raw &r, size_t c, int z) {
        r.s = 1.f;
        r.q = load_cell<double, NV>(Q, (size_t)map_axis(z, nz, bcz, r.s) * plane + c);
    };
    auto apply = [&](const Raw &r, float sx, float sy) -> C {
        C c = r.q;
        if constexpr (WALLS) apply_bc_sign<double, NV>(c, sx, sy, r.s);
        return c;
    };

    C qz[7];
#pragma unroll
    for (int d = -3; d <= 3; ++d) {
        Raw r;
        issue(r, col, zb + d);
        qz[d + 3] = apply(r, sgx, sgy);
    }
    // halos of planes zb .. zb+3 into ring slots 0..3 (visible after the
    // first barrier of the march)
    if (hx >= 0) {
#pragma unroll
        for (int d = 0; d < 4; ++d) {
            if (zb + d < ze) {
                Raw r;
                issue(r, hcol, zb + d);
                const C c = apply(r, hsx, hsy);
#pragma unroll
                for (int v = 0; v < NV; ++v) lds[d][v][hy][hx] = c.v[v];
            }
        }
    }
    // Drain the prologue loads before the march.  Otherwise the queue and
    // halo registers enter the loop as pending load targets, and the
    // compiler's conservative merge at the loop header makes every iteration
    // wait for its own 4-planes-ahead prefetch before the barrier.
    __builtin_amdgcn_s_waitcnt(0);

    const double inv48h = p.inv48h, Kc = p.K, irho = p.invrho, sLLF = p.s;

    bool nfbad = false;   // non-finite watch of this thread's outputs
    int buf = 0;          // slot of plane z
    int hslot = 4;        // slot of plane z + 4
    for (int z = zb; z < ze; ++z) {
        // column and halo of plane z+4
        Raw cq, ch;
        issue(cq, col, z + 4);
        if (hx >= 0 && z + 4 < ze) issue(ch, hcol, z + 4);
        const size_t idx = (size_t)z * plane + col;
        C e0;
        if constexpr (EPI == EPI_COMB) { if (active) e0 = load_cell_nt<double, NV>(U0, idx); }
#pragma unroll
        for (int v = 0; v < NV; ++v) lds[buf][v][ty + 3][tx + 3] = qz[3].v[v];
        __syncthreads();
        C r;
        double accB[4], dAp[3], dAvel = 0.0;
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const double *row = &lds[buf][v][ty + 3][tx + 3];
            const double xm3 = row[-3], xm2 = row[-2], xm1 = row[-1], xp1 = row[1], xp2 = row[2], xp3 = row[3];
            const double ym3 = lds[buf][v][ty][tx + 3], ym2 = lds[buf][v][ty + 1][tx + 3];
            const double ym1 = lds[buf][v][ty + 2][tx + 3];
            const double yp1 = lds[buf][v][ty + 4][tx + 3], yp2 = lds[buf][v][ty + 5][tx + 3];
            const double yp3 = lds[buf][v][ty + 6][tx + 3];
            const double q0 = qz[3].v[v];
            accB[v] = stencil_B7(xm3, xm2, xm1, q0, xp1, xp2, xp3) + stencil_B7(ym3, ym2, ym1, q0, yp1, yp2, yp3) +
                      stencil_B7(qz[0].v[v], qz[1].v[v], qz[2].v[v], q0, qz[4].v[v], qz[5].v[v], qz[6].v[v]);
            if (v == 0) {
                dAp[0] = stencil_A7(xm3, xm2, xm1, xp1, xp2, xp3);
                dAp[1] = stencil_A7(ym3, ym2, ym1, yp1, yp2, yp3);
                dAp[2] = stencil_A7(qz[0].v[0], qz[1].v[0], qz[2].v[0], qz[4].v[0], qz[5].v[0], qz[6].v[0]);
            } else if (v == 1) {
                dAvel += stencil_A7(xm3, xm2, xm1, xp1, xp2, xp3);
            } else if (v == 2) {
                dAvel += stencil_A7(ym3, ym2, ym1, yp1, yp2, yp3);
            } else {
                dAvel += stencil_A7(qz[0].v[3], qz[1].v[3], qz[2].v[3], qz[4].v[3], qz[5].v[3], qz[6].v[3]);
            }
        }
        r.v[0] = inv48h * (sLLF * accB[0] - Kc * dAvel);
        r.v[1] = inv48h * (sLLF * accB[1] - irho * dAp[0]);
        r.v[2] = inv48h * (sLLF * accB[2] - irho * dAp[1]);
        r.v[3] = inv48h * (sLLF * accB[3] - irho * dAp[2]);

        if (active) {
            C o;
            if constexpr (EPI == EPI_RHS) {
                o = r;
            } else if constexpr (EPI == EPI_AXPY) {
                const double cc = p.c;
#pragma unroll
                for (int v = 0; v < NV; ++v) o.v[v] = qz[3].v[v] + cc * r.v[v];
            } else {
                const double aa = p.a, bb = p.b, cc = p.c;
#pragma unroll
                for (int v = 0; v < NV; ++v) o.v[v] = aa * e0.v[v] + bb * qz[3].v[v] + cc * r.v[v];
            }
            if (p.nf) finite_acc<double, NV>(nfbad, o);
            store_cell_nt<double, NV>(OUT, idx, o);
        }

#pragma unroll
        for (int k = 0; k < 6; ++k) qz[k] = qz[k + 1];
        qz[6] = apply(cq, sgx, sgy);
        // slot of plane z+4 = slot of plane z-1, whose readers all passed
        // this iteration's barrier
        if (hx >= 0 && z + 4 < ze) {
            const C h = apply(ch, hsx, hsy);
#pragma unroll
            for (int v = 0; v < NV; ++v) lds[hslot][v][hy][hx] = h.v[v];
        }
        buf = buf == 4 ? 0 : buf + 1;
        hslot = hslot == 4 ? 0 : hslot + 1;
    }
    watch_flush(p.nf, nfbad);
}

// FP64 march (every WAVE2 stage, and the ACOUSTIC4 stages of fields that fit the
// last-level cache).  The own column's ring holds planes c-3 .. c+3 when plane
// c is finished; plane c is staged in LDS over the halo that already waits there.
// Column and halo of plane c+4 are loaded together, at the iteration in which
// the neighbouring tiles load those cells as their interior, so the shared
// rows are still in L2; the halo is put into its slot of a 4-plane LDS ring an
// iteration later.  Every load and store is unconditional (clamped planes,
// out-of-range buffer stores): the compiler then counts what is in flight and
// a load has a whole iteration to arrive.  (In the centre-plane march above
// a plane's loads are waited for in the iteration that issues them.)
//   Bound, ACOUSTIC4: 24 16-byte LDS reads a thread and plane, 0.75 us for
//   the 512 threads of a CU, and about 160 FP64 instructions, 0.53 us.  A walled
//   step at 150 x 131 x 90 took 150 us with the centre-plane march, 155 with
//   this one and streaming results, 114 with cached ones.  Finishing plane c
//   from in-plane parts kept for three planes, as in FP32, took three more
//   iterations a chunk (combining stage 41 -> 47 us); loading the base states
//   together with the columns, 45.
//   LDS: an ACOUSTIC4 cell as two 16-byte halves, (p, u) and (v, w), in
//   arrays of their own, so that neighbouring lanes read neighbouring words.
//   Tile: 32 x 16 columns (a wavefront is two rows of 32), or 32 x 8.
template <int SYS, int ROWS>
struct Tile64 {
    static constexpr int BX = 32, BY = ROWS;
    static constexpr int NV = SYS == ACX_ACOUSTIC4 ? 4 : 2;   // components in memory
    static constexpr int NS = SYS == ACX_ACOUSTIC4 ? 4 : 1;   // components in the stencil
    static constexpr int LX = BX + 6, LY = BY + 6;
    static constexpr int NHALO = 6 * BX + 6 * BY;              // star stencil: no plane corners
    static constexpr int NP = SYS == ACX_ACOUSTIC4 ? 2 : 1;
    using Word = typename std::conditional<SYS == ACX_ACOUSTIC4, double2, double>::type;
    struct Lds { Word q[4][NP][LY][LX]; };
};

// Store of this lane's cell of a wavefront's two rows (STREAM: nontemporal):
// row points at the first row's first cell (wave-uniform), off at the lane's
// cell behind it (beyond bytes: no store).
constexpr unsigned kNoStore = 0x80000000u;   // above every bound
template <int NV, bool STREAM>
__device__ __forceinline__ void store_cell_buf(double *row, unsigned bytes, unsigned off, const Cell<double, NV> &c)
{
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(row, 0, (int)bytes, 0x00020000);
#pragma unroll
    for (int k = 0; k < NV; k += 2) {
        union { double d[2]; acx_u32x4 u; } w;
        w.d[0] = c.v[k];
        w.d[1] = c.v[k + 1];
        __builtin_amdgcn_raw_buffer_store_b128(w.u, r, (int)off + 8 * k, 0, STREAM ? 2 : 0);
    }
}

// MEM_CACHED: results may stay in the caches, for fields small enough that the
// next stage finds them there; MEM_STREAM: nontemporal results; MEM_WIDE: the
// same for rows of 2 GB or longer (a store descriptor for each of the two rows).
// Base states are read through the caches in every mode (streaming is for
// WAVE2 only here, whose 16-byte cells load_cell_nt reads the same way).
enum { MEM_CACHED = 0, MEM_STREAM = 1, MEM_WIDE = 2 };

template <int SYS, int EPI, bool WALLS, int MEM, int ROWS>
__device__ __forceinline__ void linear_tile64(const LinArgs &p, int x0, int y0, int zb, typename Tile64<SYS, ROWS>::Lds &lds)
{
    using Tile = Tile64<SYS, ROWS>;
    constexpr int NV = Tile::NV, NS = Tile::NS, BX = Tile::BX, BY = Tile::BY;
    constexpr bool AC = SYS == ACX_ACOUSTIC4, COMB = EPI == EPI_COMB, STREAM = MEM != MEM_CACHED, WIDE = MEM == MEM_WIDE;
    using C = Cell<double, NV>;
    static_assert(BX * BY >= Tile::NHALO, "every halo cell of a plane needs a thread of its own");

    const double *__restrict__ Q = static_cast<const double *>(p.q);
    const double *__restrict__ U0 = static_cast<const double *>(p.u0);
    const int nx = p.nx, ny = p.ny, nz = p.nz;
    const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * BX + tx;
    const int ze = min(zb + p.zc, nz);
    const size_t plane = (size_t)nx * ny;
    const int bcx = WALLS ? p.bc[0] : 0, bcy = WALLS ? p.bc[1] : 0, bcz = WALLS ? p.bc[2] : 0;

    // own column
    float sgx = 1.f, sgy = 1.f;
    const int mx = map_axis(x0 + tx, nx, bcx, sgx);
    const int my = map_axis(y0 + ty, ny, bcy, sgy);
    const size_t col = (size_t)my * nx + mx;

    // halo cell of this thread; threads without one load one cell per
    // wavefront and write it to the plane's unused corner
    int hx = 0, hy = 0;
    size_t hcol = (size_t)__builtin_amdgcn_readfirstlane(my) * nx + __builtin_amdgcn_readfirstlane(mx);
    float hsx = 1.f, hsy = 1.f;
    if (tid < Tile::NHALO) {
        int t = tid;
        if (t < 6 * BY) {            // x halo: 3 left, 3 right per row
            const int row = t / 6, k = t % 6;
            hy = row + 3;
            hx = k < 3 ? k : BX + k;  // 0,1,2 | BX+3..BX+5
        } else {
            t -= 6 * BY;
            const int colx = t % BX, k = t / BX;
            hx = colx + 3;
            hy = k < 3 ? k : BY + k;
        }
        const int gx = map_axis(x0 + hx - 3, nx, bcx, hsx);
        const int gy = map_axis(y0 + hy - 3, ny, bcy, hsy);
        hcol = (size_t)gy * nx + gx;
    }

    // byte offsets inside a plane: 32 bits in the all-periodic instantiation
    using Off = typename std::conditional<WALLS, size_t, uint32_t>::type;
    const Off colb = (Off)(col * NV * 8), hcolb = (Off)(hcol * NV * 8);
    auto load = [](const double *plane_base, Off o) {
        return load_cell<double, NV>(reinterpret_cast<const double *>(reinterpret_cast<const char *>(plane_base) + o), 0);
    };
    auto load_u0 = [&](int z) {
        return load(U0 + (size_t)z * plane * NV, colb);
    };
    // the plane loaded next, its offset and its ghost sign
    int zi = 0;
    size_t zoff = 0;
    float zs = 1.f;
    auto seek = [&](int z) {
        zs = 1.f;
        zi = map_axis(z, nz, bcz, zs);
        zoff = (size_t)zi * plane * NV;
    };
    auto step = [&](int z) {   // from plane z - 1 to z
        if constexpr (WALLS) {
            seek(z);
        } else {
            ++zi;
            zoff = zi == nz ? 0 : zoff + plane * NV;
            zi = zi == nz ? 0 : zi;
        }
    };
    // this wavefront's rows of the results
    const int ty0 = __builtin_amdgcn_readfirstlane(ty);
    const bool active = tx < nx - x0 && y0 + ty < ny;
    const unsigned pair_bytes = (unsigned)(nx + BX) * NV * 8u;
    const unsigned off = active ? (unsigned)tx * NV * 8u + (WIDE ? 0u : (unsigned)(ty - ty0) * (unsigned)nx * NV * 8u) : kNoStore;
    const size_t row0 = (size_t)(y0 + ty0) * nx + x0;
    auto store = [&](int c, const C &o) {
        double *row = static_cast<double *>(p.out) + ((size_t)c * plane + row0) * NV;
        if constexpr (!WIDE) {
            store_cell_buf<NV, STREAM>(row, pair_bytes, off, o);
        } else {
            store_cell_buf<NV, STREAM>(row, BX * NV * 8u, ty == ty0 ? off : kNoStore, o);
            store_cell_buf<NV, STREAM>(row + (size_t)nx * NV, BX * NV * 8u, ty != ty0 ? off : kNoStore, o);
        }
    };

    C q[8];    // ring, slot (plane - zb + 3) & 7: the column's planes c-3 .. c+3 (signed), c+4 as loaded
    C h[2];    // halo cells of planes c+3, c+4, slot (plane - zb) & 1
    C e0;      // COMB: base state of plane c

    auto value = [&](C c, float sx, float sy, float sz) -> C {
        if constexpr (WALLS) apply_bc_sign<double, NV>(c, sx, sy, sz);
        return c;
    };
    auto put = [&](int buf, int y, int x, const C &c) {
        if constexpr (AC) {
            lds.q[buf][0][y][x] = make_double2(c.v[0], c.v[1]);
            lds.q[buf][1][y][x] = make_double2(c.v[2], c.v[3]);
        } else {
            lds.q[buf][0][y][x] = c.v[0];
        }
    };
    // In-plane part without the centre's share.  The nearest neighbours, which
    // carry the largest weight, enter as differences from the centre q0 (exact
    // for smooth data): B7 = s3 - 6 s2 + 15 (s1 - 2 q0) + 10 q0 per axis, L7 =
    // -s3 + 2 s2 + 49 (s1 - 2 q0) - 2 q0.
    // a: the A7 sums, u along x plus v along y, p along x, p along y.
    const double sLLF = p.s, Kc = p.K, irho = p.invrho;
    auto in_plane = [&](int buf, const C &q0, double (&o)[NS], double (&a)[3]) {
#pragma unroll
        for (int part = 0; part < Tile::NP; ++part) {
            const auto &P = lds.q[buf][part];
            auto ring = [&](int k, double wB, double wA, bool first) {
                const auto xp = P[ty + 3][tx + 3 + k], xm = P[ty + 3][tx + 3 - k];
                const auto yp = P[ty + 3 + k][tx + 3], ym = P[ty + 3 - k][tx + 3];
                auto sum = [&](double xpv, double xmv, double ypv, double ymv, double c) {
                    return k == 1 ? ((xpv - c) + (xmv - c)) + ((ypv - c) + (ymv - c)) : (xpv + xmv) + (ypv + ymv);
                };
                auto acc = [&](double &r, double w, double t) { r = first ? t : fma(w, t, r); };
                if constexpr (AC) {
                    const double s0 = sum(xp.x, xm.x, yp.x, ym.x, q0.v[2 * part]);
                    const double s1 = sum(xp.y, xm.y, yp.y, ym.y, q0.v[2 * part + 1]);
                    acc(o[2 * part], wB, s0);
                    acc(o[2 * part + 1], wB, s1);
                    if (part == 0) {
                        acc(a[1], wA, xp.x - xm.x);
                        acc(a[2], wA, yp.x - ym.x);
                        acc(a[0], wA, xp.y - xm.y);
                    } else {
                        a[0] = fma(wA, yp.x - ym.x, a[0]);
                    }
                } else {
                    const double s0 = sum(xp, xm, yp, ym, q0.v[0]);
                    acc(o[0], wB, first ? -s0 : s0);
                }
            };
            ring(3, 1.0, 1.0, true);
            ring(1, AC ? 15.0 : 49.0, 37.0, false);
            ring(2, AC ? -6.0 : 2.0, -8.0, false);
        }
    };

    // prologue: planes zb-3 .. zb+3 and the halos of the last four all in
    // flight at once
    size_t hoff = 0;   // plane of the halo loaded next (those past the chunk are not needed)
    {
        C ph[3];
        float sz[6];
        seek(zb - 3);
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            q[k] = load(Q + zoff, colb);
            if (k >= 3) {
                if (zb + k - 3 < ze) hoff = zoff;
                ph[k - 3] = load(Q + hoff, hcolb);
            }
            sz[k] = zs;
            step(zb - 2 + k);
        }
        q[6] = load(Q + zoff, colb);
        if (zb + 3 < ze) hoff = zoff;
        h[1] = load(Q + hoff, hcolb);
        if constexpr (COMB) e0 = load_u0(zb);
#pragma unroll
        for (int k = 0; k < 6; ++k) {
            q[k] = value(q[k], sgx, sgy, sz[k]);
            if (k >= 3) put(k - 3, hy, hx, value(ph[k - 3], hsx, hsy, sz[k]));
        }
    }

    const double cc = EPI == EPI_RHS ? 1.0 : p.c, cF = AC ? cc * p.inv48h : cc * p.lapc;
    bool nfbad = false;   // non-finite watch of this thread's outputs

    // iteration of plane c = zb + u (mod 8)
    auto body = [&](auto uu, int c) {
        constexpr int u = decltype(uu)::value;
        const float z3 = zs;   // sign of plane c+3
        step(c + 4);
        q[(u + 7) & 7] = load(Q + zoff, colb);
        if (c + 4 < ze) hoff = zoff;
        h[u & 1] = load(Q + hoff, hcolb);
        const C &zm3 = q[u], &zm2 = q[(u + 1) & 7], &zm1 = q[(u + 2) & 7], &q0 = q[(u + 3) & 7];
        const C &zp1 = q[(u + 4) & 7], &zp2 = q[(u + 5) & 7];
        C &zp3 = q[(u + 6) & 7];
        put(u & 3, ty + 3, tx + 3, q0);
        zp3 = value(zp3, sgx, sgy, z3);
        __syncthreads();
        double xy[NS], a[3];
        in_plane(u & 3, q0, xy, a);
        // halo of plane c+3 over plane c-1, which everyone has read
        put((u + 3) & 3, hy, hx, value(h[(u + 1) & 1], hsx, hsy, z3));
        C r, o;
        if constexpr (AC) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const double s1 = (zp1.v[v] - q0.v[v]) + (zm1.v[v] - q0.v[v]);
                const double s2 = zp2.v[v] + zm2.v[v], s3 = zp3.v[v] + zm3.v[v];
                r.v[v] = sLLF * (xy[v] + fma(15.0, s1, fma(30.0, q0.v[v], fma(-6.0, s2, s3))));
            }
            auto A = [&](int v) {
                const double t1 = zp1.v[v] - zm1.v[v], t2 = zp2.v[v] - zm2.v[v], t3 = zp3.v[v] - zm3.v[v];
                return fma(-8.0, t2, fma(37.0, t1, t3));
            };
            r.v[0] = fma(-Kc, a[0] + A(3), r.v[0]);
            r.v[1] = fma(-irho, a[1], r.v[1]);
            r.v[2] = fma(-irho, a[2], r.v[2]);
            r.v[3] = fma(-irho, A(0), r.v[3]);
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                if constexpr (EPI == EPI_RHS) o.v[v] = cF * r.v[v];
                else if constexpr (EPI == EPI_AXPY) o.v[v] = fma(cF, r.v[v], q0.v[v]);
                else o.v[v] = fma(cF, r.v[v], fma(p.b, q0.v[v], p.a * e0.v[v]));
            }
        } else {
            const double s1 = (zp1.v[0] - q0.v[0]) + (zm1.v[0] - q0.v[0]);
            const double s2 = zp2.v[0] + zm2.v[0], s3 = zp3.v[0] + zm3.v[0];
            const double l = xy[0] + fma(49.0, s1, fma(-6.0, q0.v[0], fma(2.0, s2, -s3)));
            const double v = q0.v[1];   // du/dt = v (rhs_function.c:330)
            if constexpr (EPI == EPI_RHS) {
                o.v[0] = v;
                o.v[1] = cF * l;
            } else if constexpr (EPI == EPI_AXPY) {
                o.v[0] = fma(cc, v, q0.v[0]);
                o.v[1] = fma(cF, l, v);
            } else {
                o.v[0] = fma(cc, v, fma(p.b, q0.v[0], p.a * e0.v[0]));
                o.v[1] = fma(cF, l, fma(p.b, v, p.a * e0.v[1]));
            }
        }
        if constexpr (COMB) e0 = load_u0(min(c + 1, ze - 1));
        store(c, o);
        C w = o;
#pragma unroll
        for (int v = 0; v < NV; ++v) w.v[v] = active ? o.v[v] : 0.0;
        finite_acc<double, NV>(nfbad, w);
    };
    for (int c = zb;; c += 8) {
        body(std::integral_constant<int, 0>{}, c);
        if (c + 1 >= ze) break;
        body(std::integral_constant<int, 1>{}, c + 1);
        if (c + 2 >= ze) break;
        body(std::integral_constant<int, 2>{}, c + 2);
        if (c + 3 >= ze) break;
        body(std::integral_constant<int, 3>{}, c + 3);
        if (c + 4 >= ze) break;
        body(std::integral_constant<int, 4>{}, c + 4);
        if (c + 5 >= ze) break;
        body(std::integral_constant<int, 5>{}, c + 5);
        if (c + 6 >= ze) break;
        body(std::integral_constant<int, 6>{}, c + 6);
        if (c + 7 >= ze) break;
        body(std::integral_constant<int, 7>{}, c + 7);
        if (c + 8 >= ze) break;
    }
    watch_flush(p.nf, nfbad);
}

// ---------------------------------------------------------------------------
// LDS-DMA march (FP64 ACOUSTIC4, all-periodic grids, RHS and AXPY stages).
//
// The same tile (32 x 16 columns) and arithmetic as the centre-plane march,
// with the plane traffic moved out of registers: every plane of the tile
// with its 3-cell x/y halo (22 x 38 cells, corners included) is copied from
// HBM straight into an LDS ring slot by direct-to-LDS loads (16 bytes per
// lane, global_load_lds_dwordx4), six slots deep (160.5 KB).  At iteration z
// the slots hold planes z .. z+5: plane z is the in-plane stencil's, planes
// z+1 .. z+3 have landed, z+4 and z+5 are in flight.  The z-stencil keeps
// the own column's planes z-3 .. z+3 in registers, the newest read from the
// slot of plane z+3 once it has landed.  So each plane's loads are issued
// five iterations before its stencil and two before its column value is
// needed, and two planes per CU are in flight while a plane is computed,
// without holding them in registers.  (Measured on MI355X at 256^3: loading
// each slot again right after a second barrier in the middle of the
// iteration, one plane deeper, and issuing the stores before the loads were
// both slower.)
//
// The loads are issued from inline assembly so that the compiler does not
// guard every LDS read with a wait for all of them; the waits are explicit:
// loads complete in issue order, and at iteration z the only loads issued
// after plane z+3's are those of plane z+4 (nj per wavefront), so vmcnt <= nj
// means plane z+3 has landed in this wavefront's part (stores count too,
// which can only lengthen the wait); the barrier that follows makes every
// wavefront's part visible and ends all reads of the slot the next loads
// overwrite.  Plane layout in a slot: two
// arrays of 22 x 38 16-byte entries, the (p, u) halves then the (v, w)
// halves of the cells, row-major; one wavefront load fills 64 consecutive
// entries.
struct DmaPlan {
    static constexpr int BX = 32, BY = 16, RW = BX + 6, RH = BY + 6;
    static constexpr int NE = RW * RH;              // 836 cells per plane
    static constexpr int NENT = 2 * NE;             // 1672 sixteen-byte entries
    static constexpr int SLOT = NENT * 16;          // 26752 bytes
    static constexpr int NSLOT = 6;
    static constexpr int NCHUNK = (NENT + 63) / 64; // 27 wavefront loads per plane
    static constexpr int NWAVE = BX * BY / 64;      // 8
    static constexpr int MAXJ = (NCHUNK + NWAVE - 1) / NWAVE;   // 4 loads per wavefront at most
};

template <int EPI, bool RS>
__device__ __forceinline__ void linear_tile_dma(const LinArgs &p, int x0, int y0, int zb, unsigned char *ring)
{
    using D = DmaPlan;
    static_assert(EPI == EPI_RHS || EPI == EPI_AXPY, "LDS-DMA march: RHS and AXPY stages");
    const double *__restrict__ Q = static_cast<const double *>(p.q);
    double *__restrict__ OUT = static_cast<double *>(p.out);
    const int nx = p.nx, ny = p.ny, nz = p.nz;
    const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * D::BX + tx;
    const int wave = tid >> 6, lane = tid & 63;
    const int ze = min(zb + p.zc, nz);
    const bool active = (x0 + tx < nx) && (y0 + ty < ny);
    const size_t plane = (size_t)nx * ny;

    // this lane's entries of a plane: chunk q = wave + 8 j covers entries 64 q .. 64 q + 63
    const int nj = wave + D::NWAVE * (D::MAXJ - 1) < D::NCHUNK ? D::MAXJ : D::MAXJ - 1;
    uint32_t eoff[D::MAXJ];
    bool eok[D::MAXJ];
#pragma unroll
    for (int j = 0; j < D::MAXJ; ++j) {
        const int e = (wave + D::NWAVE * j) * 64 + lane;
        eok[j] = j < nj && e < D::NENT;
        const int h = e / D::NE, idx = e - h * D::NE, r = idx / D::RW, c = idx - r * D::RW;
        // in 32 bits: the launcher takes planes below 2^31 doubles
        eoff[j] = eok[j] ? region_cell(x0, y0, 3, r, c, nx, ny) * 4u + 2u * h : 0u;
    }
    auto slot_of = [&](int z) { return (z - zb + 3) % D::NSLOT; };
    auto issue = [&](int z, int slot) {
        int zz = z % nz;
        zz = zz < 0 ? zz + nz : zz;
        const double *src = Q + (size_t)zz * plane * 4;
        unsigned char *dst = ring + slot * D::SLOT;
#pragma unroll
        for (int j = 0; j < D::MAXJ; ++j) {
            if (j < nj) {
                // LDS byte offset of the chunk (wave-uniform) into M0; the
                // lane's 16 bytes land at M0 + 16 * lane
                const unsigned lds = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(
                    (__attribute__((address_space(3))) unsigned char *)(dst + (wave + D::NWAVE * j) * 1024)));
                const double *g = src + eoff[j];
                if (eok[j])
                    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                                 :: "s"(lds), "v"(g) : "memory", "m0");
            }
        }
    };
    // s_waitcnt with only vmcnt constrained (gfx9 encoding: expcnt 7,
    // lgkmcnt 15): all but the loads of the `later` most recent planes
    auto wait_planes = [&](int later) {
        if (later == 0) {
            __builtin_amdgcn_s_waitcnt(0x0F70);
        } else if (later == 1) {
            if (nj == 4) __builtin_amdgcn_s_waitcnt(0x0F74);
            else __builtin_amdgcn_s_waitcnt(0x0F73);
        } else {
            if (nj == 4) __builtin_amdgcn_s_waitcnt(0x0F78);
            else __builtin_amdgcn_s_waitcnt(0x0F76);
        }
    };
    auto cell_at = [&](int slot, int r, int c) -> Cell<double, 4> {
        const unsigned char *b = ring + slot * D::SLOT;
        const double2 a = *reinterpret_cast<const double2 *>(b + (r * D::RW + c) * 16);
        const double2 v = *reinterpret_cast<const double2 *>(b + (D::NE + r * D::RW + c) * 16);
        Cell<double, 4> o;
        o.v[0] = a.x; o.v[1] = a.y; o.v[2] = v.x; o.v[3] = v.y;
        return o;
    };
    auto half_at = [&](int slot, int h, int r, int c) -> double2 {
        return *reinterpret_cast<const double2 *>(ring + slot * D::SLOT + (h * D::NE + r * D::RW + c) * 16);
    };

    // prologue: planes zb-3 .. zb+2 into slots 0 .. 5, their own-column values
    // into the z-queue, then planes zb+3 and zb+4 into the slots of zb-3, zb-2
    for (int d = 0; d < D::NSLOT; ++d) issue(zb - 3 + d, d);
    wait_planes(0);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    Cell<double, 4> qz[7];
#pragma unroll
    for (int d = 0; d < 6; ++d) qz[d + 1] = cell_at(d, ty + 3, tx + 3);
    qz[0] = qz[1];
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    issue(zb + 3, slot_of(zb + 3));
    if (zb + 4 <= ze + 2) issue(zb + 4, slot_of(zb + 4));

    const double inv48h = p.inv48h, Kc = p.K, irho = p.invrho, sLLF = p.s;
    // Results: RS false, each lane stores its own cell (two 16-byte stores,
    // (p, u) then (v, w)).  RS true, row-complete stores: lanes 0-31 of a
    // wavefront hold row y0 + 2 wave of the tile, lanes 32-63 the next row;
    // after one lane-half exchange (permlane32_swap) the first store writes
    // the first row whole (lane l: cell l & 31, half l >> 5) and the second
    // store the second row, so each 64-byte line of the output is written by
    // one instruction.  Measured on MI355X: the output bytes equal the
    // compulsory ones (7 % more with RS false, some lines reach memory
    // twice); 3.4 % faster at 384^3 (several rounds of workgroups per CU),
    // 0.8 % slower at 256^3 (one round).
    const size_t col = (size_t)(y0 + ty) * nx + (x0 + tx);
    bool nfbad = false;
    for (int z = zb; z < ze; ++z) {
        // plane z+3 landed: the loads issued after its loads are plane z+4's
        // (when issued: planes beyond ze+2 are not needed)
        wait_planes(z + 4 <= ze + 2);
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        // every wavefront is past iteration z-1: its slot takes plane z+5
        if (z + 5 <= ze + 2) issue(z + 5, slot_of(z + 5));
        const int s0 = slot_of(z);
#pragma unroll
        for (int k = 0; k < 6; ++k) qz[k] = qz[k + 1];
        qz[6] = cell_at(slot_of(z + 3), ty + 3, tx + 3);

        // in-plane stencils from the slot of plane z, one 16-byte half (two
        // components) at a time; z-stencils from the queue
        double accB[4], dAp[3], dAvel = 0.0;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            double2 xr[7], yc[7];
#pragma unroll
            for (int k = 0; k < 7; ++k) {
                xr[k] = half_at(s0, h, ty + 3, tx + k);
                yc[k] = half_at(s0, h, ty + k, tx + 3);
            }
#pragma unroll
            for (int w = 0; w < 2; ++w) {
                const int v = 2 * h + w;
                auto X = [&](int k) { return w ? xr[k].y : xr[k].x; };
                auto Y = [&](int k) { return w ? yc[k].y : yc[k].x; };
                const double q0 = qz[3].v[v];
                accB[v] = stencil_B7(X(0), X(1), X(2), q0, X(4), X(5), X(6)) +
                          stencil_B7(Y(0), Y(1), Y(2), q0, Y(4), Y(5), Y(6)) +
                          stencil_B7(qz[0].v[v], qz[1].v[v], qz[2].v[v], q0, qz[4].v[v], qz[5].v[v], qz[6].v[v]);
                if (v == 0) {
                    dAp[0] = stencil_A7(X(0), X(1), X(2), X(4), X(5), X(6));
                    dAp[1] = stencil_A7(Y(0), Y(1), Y(2), Y(4), Y(5), Y(6));
                    dAp[2] = stencil_A7(qz[0].v[0], qz[1].v[0], qz[2].v[0], qz[4].v[0], qz[5].v[0], qz[6].v[0]);
                } else if (v == 1) {
                    dAvel += stencil_A7(X(0), X(1), X(2), X(4), X(5), X(6));
                } else if (v == 2) {
                    dAvel += stencil_A7(Y(0), Y(1), Y(2), Y(4), Y(5), Y(6));
                } else {
                    dAvel += stencil_A7(qz[0].v[3], qz[1].v[3], qz[2].v[3], qz[4].v[3], qz[5].v[3], qz[6].v[3]);
                }
            }
        }
        Cell<double, 4> r;
        r.v[0] = inv48h * (sLLF * accB[0] - Kc * dAvel);
        r.v[1] = inv48h * (sLLF * accB[1] - irho * dAp[0]);
        r.v[2] = inv48h * (sLLF * accB[2] - irho * dAp[1]);
        r.v[3] = inv48h * (sLLF * accB[3] - irho * dAp[2]);
        if constexpr (RS) {
            Cell<double, 4> o;
            if constexpr (EPI == EPI_RHS) {
                o = r;
            } else {
                const double cc = p.c;
#pragma unroll
                for (int v = 0; v < 4; ++v) o.v[v] = qz[3].v[v] + cc * r.v[v];
            }
            if (active && p.nf) finite_acc<double, 4>(nfbad, o);
            // (p, u) of lanes 32-63 <-> (v, w) of lanes 0-31: all lanes take part
            swap_halves32(o.v[0], o.v[2]);
            swap_halves32(o.v[1], o.v[3]);
            const int xc = x0 + (lane & 31), rowA = y0 + 2 * wave;
            double *outA = OUT + ((size_t)z * plane + (size_t)rowA * nx + xc) * 4 + 2 * (lane >> 5);
            if (xc < nx && rowA < ny)
                __builtin_nontemporal_store(acx_dbl2{o.v[0], o.v[1]}, reinterpret_cast<acx_dbl2 *>(outA));
            if (xc < nx && rowA + 1 < ny)
                __builtin_nontemporal_store(acx_dbl2{o.v[2], o.v[3]}, reinterpret_cast<acx_dbl2 *>(outA + (size_t)nx * 4));
        } else if (active) {
            Cell<double, 4> o;
            if constexpr (EPI == EPI_RHS) {
                o = r;
            } else {
                const double cc = p.c;
#pragma unroll
                for (int v = 0; v < 4; ++v) o.v[v] = qz[3].v[v] + cc * r.v[v];
            }
            if (p.nf) finite_acc<double, 4>(nfbad, o);
            store_cell_nt<double, 4>(OUT, (size_t)z * plane + col, o);
        }
    }
    // every load issued has been waited for by the last iteration (vmcnt 0)
    watch_flush(p.nf, nfbad);
}

} // namespace acx
