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
// halo of 3 (double-buffered, one barrier per plane) for its in-plane
// stencils, and pushed into a per-thread register queue that supplies the
// z-stencil three planes later.  HBM traffic per stage is one read of Q
// (+ U0) and one write of OUT; halo rows are read by neighbouring tiles at
// the same plane index, so they meet in L2 (tiles are ordered per XCD).
#include "acx_linear_core.h"

namespace acx {

// Centre-plane march with the 5-plane halo ring (acx_linear_core.h), FP64, on
// 32 x 16 tiles.  WALLS = false is the all-periodic instantiation (no ghost
// signs).
template <int SYS, int EPI, bool WALLS>
__global__ void __launch_bounds__(32 * 16)
k_linear(LinArgs p)
{
    __shared__ double lds[5][LinTile<SYS, 32, 16>::NS][16 + 6][32 + 6];
    const int tile = xcd_logical_tile(blockIdx.x, gridDim.x);
    const int x0 = (tile % p.ntx) * 32, y0 = ((tile / p.ntx) % p.nty) * 16, zb = (tile / (p.ntx * p.nty)) * p.zc;
    linear_tile_centre<SYS, 32, 16, EPI, WALLS>(p, x0, y0, zb, lds);
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

// WAVE2 RHS / AXPY stages on the same march: 80 KB of LDS, two blocks per CU
// (registers capped for 4 waves per SIMD).
template <int EPI>
__global__ void __launch_bounds__(DmaPlan::BX *DmaPlan::BY) __attribute__((amdgpu_waves_per_eu(4)))
k_linear_dma_w2(LinArgs p)
{
    __shared__ __attribute__((aligned(16))) unsigned char ring[DmaPlanW2::NSLOT * DmaPlanW2::SLOT];
    const int tile = xcd_logical_tile(blockIdx.x, gridDim.x);
    const int x0 = (tile % p.ntx) * DmaPlan::BX, y0 = ((tile / p.ntx) % p.nty) * DmaPlan::BY;
    const int zb = (tile / (p.ntx * p.nty)) * p.zc;
    linear_tile_dma_w2<EPI>(p, x0, y0, zb, ring);
}

template <int EPI>
static int launch_linear_dma_w2(const LinArgs &a, hipStream_t s)
{
    LinArgs b = a;
    b.ntx = (a.nx + DmaPlan::BX - 1) / DmaPlan::BX;
    b.nty = (a.ny + DmaPlan::BY - 1) / DmaPlan::BY;
    static int per_cu = 0;
    if (!per_cu) {
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, reinterpret_cast<const void *>(&k_linear_dma_w2<EPI>),
                                                         DmaPlan::BX * DmaPlan::BY, 0) != hipSuccess || n <= 0)
            n = 1;
        per_cu = n;
    }
    if (b.zc <= 0) b.zc = auto_zc(b.ntx, b.nty, a.nz, device_cus() * per_cu, 10);
    b.ntz = (a.nz + b.zc - 1) / b.zc;
    hipLaunchKernelGGL(k_linear_dma_w2<EPI>, dim3((unsigned)(b.ntx * b.nty * b.ntz)), dim3(DmaPlan::BX, DmaPlan::BY),
                       0, s, b);
    return hip_check(hipGetLastError(), "k_linear_dma_w2 launch");
}

// ---------------------------------------------------------------------------

template <int SYS, int EPI, bool WALLS>
static int launch_linear_v(const LinArgs &a, hipStream_t s)
{
    LinArgs b = a;
    b.ntx = (a.nx + 31) / 32;
    b.nty = (a.ny + 15) / 16;
    if (b.zc <= 0) {
        // workgroups of this instantiation that fit a CU at once (queried once)
        static int per_cu = 0;
        if (!per_cu) {
            int n = 0;
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                    &n, reinterpret_cast<const void *>(&k_linear<SYS, EPI, WALLS>), 32 * 16, 0) != hipSuccess || n <= 0)
                n = 1;
            per_cu = n;
        }
        // At most two blocks per CU count as slots: the round model takes the
        // smallest z-chunk that fills one round, and with four co-resident
        // blocks of the WAVE2 kernel that was 32 planes at 256^3, whose z-halo
        // re-reads cost more than the round saved (measured at 256^3: WAVE2
        // step 0.458 ms with the COMB stage at 32 planes, 0.450 at 64).
        b.zc = auto_zc(b.ntx, b.nty, a.nz, device_cus() * (per_cu < 2 ? per_cu : 2), 10);
    }
    b.ntz = (a.nz + b.zc - 1) / b.zc;
    hipLaunchKernelGGL((k_linear<SYS, EPI, WALLS>), dim3(b.ntx * b.nty * b.ntz), dim3(32, 16), 0, s, b);
    return hip_check(hipGetLastError(), "k_linear launch");
}

// FP32 compensated stages (linear_tile32).
template <int SYS, int BY, int STAGE, bool WALLS>
__global__ void __launch_bounds__(64 * BY) __attribute__((amdgpu_waves_per_eu(BY / 4)))
k_linear32(LinArgs p)
{
    __shared__ typename Tile32<SYS, BY>::template Shared<STAGE> lds;
    const int tile = xcd_logical_tile(blockIdx.x, gridDim.x);
    const int x0 = (tile % p.ntx) * 64, y0 = ((tile / p.ntx) % p.nty) * BY, zb = (tile / (p.ntx * p.nty)) * p.zc;
    linear_tile32<SYS, BY, STAGE, WALLS>(p, x0, y0, zb, lds);
}

// Tiles of 64 x 12 columns (one block of 12 wavefronts per CU, at most 168
// VGPRs), or of 64 x 8 where their rounds come out shorter: a plane of the
// larger tile takes about 1.3 times as long for 1.5 times the cells.
// Measured, us per step: 384^3 2235 with 12 rows, 2490 with 8; 256^3 (22 tiles
// of 12 rows in y, two rounds; 32 of 8 rows, one round) 713 and 647.
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
    if (big) hipLaunchKernelGGL((k_linear32<SYS, 12, STAGE, WALLS>), grd, dim3(64, 12), 0, s, b);
    else hipLaunchKernelGGL((k_linear32<SYS, 8, STAGE, WALLS>), grd, dim3(64, 8), 0, s, b);
    return hip_check(hipGetLastError(), "k_linear32 launch");
}

template <int SYS>
static int launch_linear32(const LinArgs &a, hipStream_t s)
{
    // the all-periodic instantiation keeps offsets inside a plane in 32 bits
    const bool general = a.bc[0] != ACX_PERIODIC || a.bc[1] != ACX_PERIODIC || a.bc[2] != ACX_PERIODIC ||
                         (size_t)a.nx * a.ny * (SYS == ACX_ACOUSTIC4 ? 16 : 8) > 0xffffffffu;
    if (a.final_stage)
        return general ? launch_linear32_w<SYS, F32_LAST, true>(a, s) : launch_linear32_w<SYS, F32_LAST, false>(a, s);
    if (a.d)
        return general ? launch_linear32_w<SYS, F32_MID, true>(a, s) : launch_linear32_w<SYS, F32_MID, false>(a, s);
    return general ? launch_linear32_w<SYS, F32_FIRST, true>(a, s) : launch_linear32_w<SYS, F32_FIRST, false>(a, s);
}

// FP64 stages: all-periodic RHS and AXPY stages take the LDS-DMA march, the
// others the centre-plane march.
template <int SYS, int EPI>
static int launch_linear64(const LinArgs &a, hipStream_t s)
{
    const bool walls = a.bc[0] != ACX_PERIODIC || a.bc[1] != ACX_PERIODIC || a.bc[2] != ACX_PERIODIC;
    if constexpr (SYS == ACX_ACOUSTIC4 && (EPI == EPI_RHS || EPI == EPI_AXPY)) {
        // the LDS-DMA march (measured at 256^3: AXPY stage 207 -> 196 us,
        // step 0.958 -> 0.905 ms): periodic grids whose plane offsets fit 32 bits
        if (!walls && (size_t)a.nx * a.ny * 4 < 0x7fffffffu)
            return launch_linear_dma<EPI>(a, s);
    }
    if constexpr (SYS == ACX_WAVE2 && (EPI == EPI_RHS || EPI == EPI_AXPY)) {
        // measured: the WAVE2 step 0.485 -> 0.459 ms at 256^3, 1.904 -> 1.760 ms
        // at 384^3, bit-identical to the halo-ring kernel
        if (!walls && (size_t)a.nx * a.ny * 2 < 0x7fffffffu)
            return launch_linear_dma_w2<EPI>(a, s);
    }
    return walls ? launch_linear_v<SYS, EPI, true>(a, s) : launch_linear_v<SYS, EPI, false>(a, s);
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
