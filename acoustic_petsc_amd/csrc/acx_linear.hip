// acx_linear.hip -- fused RHS + SSP-stage kernel for the linear (shipped)
// CWENO4 scheme, gamma_hi = 1, gamma_lo = 0.
//
// With those weights the reference's weno() returns the 4th-order central
// polynomial exactly (3d/weno4/plane_wave/reconstruction.c:42-59,236-257:
// gamma_R3 = 0 so w_R3 = 0 and wt_ratio = 1), and the 2x2 Gauss-point face
// averages of its value / normal gradient depend only on 1D five-point
// combinations along the face normal.  The RHS is then an axis-aligned
// 7-point star stencil per axis (see acx_device.h), fused here with the
// SSP stage combination  OUT = a*U0 + b*Q + c*F(Q).
//
// Layout: 2.5D blocking.  A block owns a BX x BY column tile and marches a
// chunk of z-planes.  Each plane is read once: staged in LDS with an x/y
// halo of 3 (one barrier per plane) for its in-plane stencils, and kept in
// per-thread registers for the z-stencils.  HBM traffic per stage is one read of Q
// (+ U0) and one write of OUT; halo rows are read by neighbouring tiles at
// the same plane index, so they meet in L2 (tiles are ordered per XCD).
#include "acx_linear_core.h"

namespace acx {

// FP64 march (acx_linear_core.h).  WALLS = false is the all-periodic
// instantiation (no ghost signs, offsets inside a plane in 32 bits).
template <int SYS, int EPI, bool WALLS, int MEM, int ROWS>
__global__ void __launch_bounds__(32 * ROWS) __attribute__((amdgpu_waves_per_eu(2)))
k_linear64(LinArgs p)
{
    using Tile = Tile64<SYS, ROWS>;
    __shared__ typename Tile::Lds lds;
    const int tile = xcd_logical_tile(blockIdx.x, gridDim.x);
    const int x0 = (tile % p.ntx) * Tile::BX, y0 = ((tile / p.ntx) % p.nty) * Tile::BY, zb = (tile / (p.ntx * p.nty)) * p.zc;
    linear_tile64<SYS, EPI, WALLS, MEM, ROWS>(p, x0, y0, zb, lds);
}

// Centre-plane march with the 5-plane halo ring (acx_linear_core.h), FP64
// ACOUSTIC4 on 32 x 16 tiles.  WALLS = false is the all-periodic instantiation
// (no ghost signs).
template <int EPI, bool WALLS>
__global__ void __launch_bounds__(32 * 16)
k_linear(LinArgs p)
{
    __shared__ double lds[5][LinTile::NV][LinTile::BY + 6][LinTile::BX + 6];
    const int tile = xcd_logical_tile(blockIdx.x, gridDim.x);
    const int x0 = (tile % p.ntx) * 32, y0 = ((tile / p.ntx) % p.nty) * 16, zb = (tile / (p.ntx * p.nty)) * p.zc;
    linear_tile_centre<EPI, WALLS>(p, x0, y0, zb, lds);
}

// LDS-DMA march (acx_linear_core.h): FP64 ACOUSTIC4 RHS / AXPY stages on
// all-periodic grids; one block of 512 threads per CU (the ring is 160.5 KB).
// RS: row-complete result stores, taken when the launch needs more than one
// round of workgroups.
template <int EPI, bool RS>
__global__ void __launch_bounds__(DmaPlan::BX *DmaPlan::BY) k_linear_dma(LinArgs p)
{
    __shared__ __attribute__((aligned(16))) unsigned char ring[DmaPlan::NSLOT * DmaPlan::SLOT];
    const int tile = xcd_logical_tile(blockIdx.x, gridDim.x);
    const int x0 = (tile % p.ntx) * DmaPlan::BX, y0 = ((tile / p.ntx) % p.nty) * DmaPlan::BY;
    const int zb = (tile / (p.ntx * p.nty)) * p.zc;
    linear_tile_dma<EPI, RS>(p, x0, y0, zb, ring);
}

template <int EPI>
static int launch_linear_dma(const LinArgs &a, hipStream_t s)
{
    LinArgs b = a;
    b.ntx = (a.nx + DmaPlan::BX - 1) / DmaPlan::BX;
    b.nty = (a.ny + DmaPlan::BY - 1) / DmaPlan::BY;
    static int per_cu = 0;
    if (!per_cu) {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void *>(&k_linear_dma<EPI, false>),
                                                         DmaPlan::BX * DmaPlan::BY, 0) != hipSuccess || n <= 0)
            n = 1;
        per_cu = n;
    }
    const int slots = device_cus() * per_cu;
    if (b.zc <= 0) b.zc = auto_zc(b.ntx, b.nty, a.nz, slots, 10);
    b.ntz = (a.nz + b.zc - 1) / b.zc;
    const long long wgs = (long long)b.ntx * b.nty * b.ntz;
    if (wgs > slots)
        hipLaunchKernelGGL((k_linear_dma<EPI, true>), dim3((unsigned)wgs), dim3(DmaPlan::BX, DmaPlan::BY), 0, s, b);
    else
        hipLaunchKernelGGL((k_linear_dma<EPI, false>), dim3((unsigned)wgs), dim3(DmaPlan::BX, DmaPlan::BY), 0, s, b);
    return hip_check(hipGetLastError(), "k_linear_dma launch");
}

// ---------------------------------------------------------------------------

// Slots of the round model: the CUs, or two blocks per CU with 8 rows.  (Two
// for the 16-row WAVE2 kernel, whose registers would allow it, halves its
// chunks: 256^3 159 us for the combining stage and 84.6 for the others, against
// 139 and 79.7.)
template <int SYS, int EPI, bool WALLS, int MEM, int ROWS = 16>
static int launch_linear64_w(const LinArgs &a, hipStream_t s)
{
    using Tile = Tile64<SYS, ROWS>;
    LinArgs b = a;
    b.ntx = (a.nx + Tile::BX - 1) / Tile::BX;
    b.nty = (a.ny + Tile::BY - 1) / Tile::BY;
    if (b.zc <= 0) b.zc = auto_zc(b.ntx, b.nty, a.nz, device_cus() * (16 / ROWS), 10);
    b.ntz = (a.nz + b.zc - 1) / b.zc;
    hipLaunchKernelGGL((k_linear64<SYS, EPI, WALLS, MEM, ROWS>), dim3(b.ntx * b.nty * b.ntz), dim3(Tile::BX, Tile::BY), 0, s, b);
    return hip_check(hipGetLastError(), "k_linear64 launch");
}

template <int EPI, bool WALLS>
static int launch_linear_v(const LinArgs &a, hipStream_t s)
{
    LinArgs b = a;
    b.ntx = (a.nx + LinTile::BX - 1) / LinTile::BX;
    b.nty = (a.ny + LinTile::BY - 1) / LinTile::BY;
    if (b.zc <= 0) b.zc = auto_zc(b.ntx, b.nty, a.nz, device_cus(), 10);
    b.ntz = (a.nz + b.zc - 1) / b.zc;
    hipLaunchKernelGGL((k_linear<EPI, WALLS>), dim3(b.ntx * b.nty * b.ntz), dim3(LinTile::BX, LinTile::BY), 0, s, b);
    return hip_check(hipGetLastError(), "k_linear launch");
}

// FP32 compensated stages (linear_tile32).
template <int SYS, int BY, int STAGE, bool WALLS, bool STREAM>
__global__ void __launch_bounds__(64 * BY) __attribute__((amdgpu_waves_per_eu(BY / 4)))
k_linear32(LinArgs p)
{
    __shared__ typename Tile32<SYS, BY>::template Shared<STAGE> lds;
    const int tile = xcd_logical_tile(blockIdx.x, gridDim.x);
    const int x0 = (tile % p.ntx) * 64, y0 = ((tile / p.ntx) % p.nty) * BY, zb = (tile / (p.ntx * p.nty)) * p.zc;
    linear_tile32<SYS, BY, STAGE, WALLS, STREAM>(p, x0, y0, zb, lds);
}

// Tiles of 64 x 12 columns (one block of 12 wavefronts per CU, at most 168
// VGPRs), or of 64 x 8 where their rounds come out shorter: a plane of the
// larger tile takes about 1.3 times as long for 1.5 times the cells.
// Measured, us per step: 384^3 2235 with 12 rows, 2490 with 8; 256^3 (22 tiles
// of 12 rows in y, two rounds; 32 of 8 rows, one round) 713 and 647.
//
// Results stay in the caches (STREAM = false) up to CACHED32_BYTES a field (a
// stage reads up to three fields and writes two): us per step, cached against
// streaming, ACOUSTIC4 128^3 92 against 103, 150 x 131 x 90 86 / 105, 160^3 183
// / 190, 192^3 299 / 274; WAVE2 128^3 55 / 64, 192^3 153 / 164, 256^3 433 / 407.
constexpr size_t CACHED32_BYTES = 80ull << 20;

template <int SYS, int STAGE, bool WALLS>
static int launch_linear32_w(const LinArgs &a, hipStream_t s)
{
    LinArgs b = a;
    const int slots = device_cus();
    b.ntx = (a.nx + 63) / 64;
    const int nty12 = (a.ny + 11) / 12, nty8 = (a.ny + 7) / 8;
    double c12, c8;
    const int z12 = auto_zc(b.ntx, nty12, a.nz, slots, 10, &c12), z8 = auto_zc(b.ntx, nty8, a.nz, slots, 10, &c8);
    const bool big = 1.3 * c12 <= c8;
    b.nty = big ? nty12 : nty8;
    if (b.zc <= 0) b.zc = big ? z12 : z8;
    b.ntz = (a.nz + b.zc - 1) / b.zc;
    const dim3 grd((unsigned)(b.ntx * b.nty * b.ntz));
    const bool cached = (size_t)a.nx * a.ny * a.nz * Tile32<SYS, 8>::NV * 4 <= CACHED32_BYTES;
    const void *k = big ? (cached ? reinterpret_cast<const void *>(&k_linear32<SYS, 12, STAGE, WALLS, false>)
                                  : reinterpret_cast<const void *>(&k_linear32<SYS, 12, STAGE, WALLS, true>))
                        : (cached ? reinterpret_cast<const void *>(&k_linear32<SYS, 8, STAGE, WALLS, false>)
                                  : reinterpret_cast<const void *>(&k_linear32<SYS, 8, STAGE, WALLS, true>));
    void *args[] = {&b};
    if (int rc = hip_check(hipLaunchKernel(k, grd, dim3(64, big ? 12 : 8), args, 0, s), "k_linear32 launch")) return rc;
    return hip_check(hipGetLastError(), "k_linear32 launch");
}

template <int SYS>
static int launch_linear32(const LinArgs &a, hipStream_t s)
{
    const bool general = a.bc[0] != ACX_PERIODIC || a.bc[1] != ACX_PERIODIC || a.bc[2] != ACX_PERIODIC ||
                         plane_beyond_32_bits(a.nx, a.ny, SYS == ACX_ACOUSTIC4 ? 16 : 8);
    if (a.final_stage)
        return general ? launch_linear32_w<SYS, F32_LAST, true>(a, s) : launch_linear32_w<SYS, F32_LAST, false>(a, s);
    if (a.d)
        return general ? launch_linear32_w<SYS, F32_MID, true>(a, s) : launch_linear32_w<SYS, F32_MID, false>(a, s);
    return general ? launch_linear32_w<SYS, F32_FIRST, true>(a, s) : launch_linear32_w<SYS, F32_FIRST, false>(a, s);
}

// FP64 stages.  Where a field is at most CACHED_BYTES, linear_tile64 with
// cached results (a stage's result is the next one's input, and the 256 MB
// last-level cache holds two fields).  Above, results stream, WAVE2 stays with
// linear_tile64, all-periodic ACOUSTIC4 RHS and AXPY stages take the LDS-DMA
// march and the other ACOUSTIC4 stages the centre-plane march.  Measured, us
// per step (all periodic, walled):
//                   others         linear_tile64   linear_tile64
//                                  streaming       cached
//   ACOUSTIC4 128^3   158, 155       157, 160        114, 116
//   ACOUSTIC4 192^3   436, 459       462, 464        466, 465
//   WAVE2 128^3       73.7, 68.2     73.1, 73.3      59.2, 58.7
//   WAVE2 192^3       217, 208       195, 195        195, 192
//   WAVE2 224^3       318, 346       317, 317        333, 333
//   WAVE2 384^3       1679, 1758     1683, 1674      1778, 1768
//
// Up to HALF_TILE_BYTES tiles of 8 rows, whose two blocks per CU have a barrier
// of their own each; above, their larger halo costs more.  8 against 16 rows, us
// per step: ACOUSTIC4 64^3 32.3, 33.5; 150 x 131 x 90 (54 MB) 108, 114; 200 x 150
// x 100 (96 MB) 202, 195.  WAVE2 96^3 33.2, 35.4; 200 x 150 x 100 (48 MB) 83.1,
// 86.7.
constexpr size_t CACHED_BYTES = 128ull << 20, HALF_TILE_BYTES = 64ull << 20;

template <int SYS, int EPI>
static int launch_linear64(const LinArgs &a, hipStream_t s)
{
    const bool walls = a.bc[0] != ACX_PERIODIC || a.bc[1] != ACX_PERIODIC || a.bc[2] != ACX_PERIODIC;
    const size_t plane_bytes = (size_t)a.nx * a.ny * Tile64<SYS, 16>::NV * 8;
    if (plane_bytes * a.nz <= HALF_TILE_BYTES)
        return walls ? launch_linear64_w<SYS, EPI, true, MEM_CACHED, 8>(a, s)
                     : launch_linear64_w<SYS, EPI, false, MEM_CACHED, 8>(a, s);
    if (plane_bytes * a.nz <= CACHED_BYTES)
        return walls ? launch_linear64_w<SYS, EPI, true, MEM_CACHED>(a, s)
                     : launch_linear64_w<SYS, EPI, false, MEM_CACHED>(a, s);
    if constexpr (SYS == ACX_ACOUSTIC4) {
        if constexpr (EPI != EPI_COMB) {
            // plane offsets in 32 bits
            if (!walls && (size_t)a.nx * a.ny * 4 < 0x7fffffffu) return launch_linear_dma<EPI>(a, s);
        }
        return walls ? launch_linear_v<EPI, true>(a, s) : launch_linear_v<EPI, false>(a, s);
    } else {
        if ((size_t)a.nx * 16 >= 0x7fff0000u) return launch_linear64_w<SYS, EPI, true, MEM_WIDE>(a, s);
        return walls || plane_bytes > 0xffffffffu ? launch_linear64_w<SYS, EPI, true, MEM_STREAM>(a, s)
                                                  : launch_linear64_w<SYS, EPI, false, MEM_STREAM>(a, s);
    }
}

int launch_linear(const LinArgs &a, int sys, int epi, bool fp32, hipStream_t s)
{
    if (fp32) {
        if (epi != EPI_F32C) return set_error(ACX_EUNSUPPORTED, "fp32 linear kernel supports the compensated stage only");
        return sys == ACX_ACOUSTIC4 ? launch_linear32<ACX_ACOUSTIC4>(a, s) : launch_linear32<ACX_WAVE2>(a, s);
    }
    if (sys == ACX_ACOUSTIC4) {
        switch (epi) {
        case EPI_RHS: return launch_linear64<ACX_ACOUSTIC4, EPI_RHS>(a, s);
        case EPI_AXPY: return launch_linear64<ACX_ACOUSTIC4, EPI_AXPY>(a, s);
        case EPI_COMB: return launch_linear64<ACX_ACOUSTIC4, EPI_COMB>(a, s);
        }
    } else {
        switch (epi) {
        case EPI_RHS: return launch_linear64<ACX_WAVE2, EPI_RHS>(a, s);
        case EPI_AXPY: return launch_linear64<ACX_WAVE2, EPI_AXPY>(a, s);
        case EPI_COMB: return launch_linear64<ACX_WAVE2, EPI_COMB>(a, s);
        }
    }
    return set_error(ACX_EUNSUPPORTED, "linear kernel: unsupported epilogue");
}

} // namespace acx
