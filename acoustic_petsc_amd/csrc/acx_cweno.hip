// acx_cweno.hip -- fused RHS + SSP-stage kernel for the general (nonlinear)
// CWENO4 scheme: smoothness indicators, nonlinear weights, face averages,
// Riemann flux and divergence in one pass.
//
// Reconstruction: 3d/weno4/plane_wave/reconstruction.c:38-259 with the linear
// weights of the caller (the nonlinear setting of the reference is
// gamma_hi = gamma_lo = 0.85, Viscous-Multiphase-Fourth-Order/reconstruction.c:42-43).
// Only what the face averages need is formed: the 2x2 Gauss rule on a face
// annihilates every tangential basis term, so the face average of the value
// is c0 +- c1/2 + c4/6 +- c10/20 along x (c2,c5,c11 along y; c3,c6,c12 along
// z) and of the normal gradient (c1 +- c4 + 3/5 c10)/h.  The smoothness
// indicators still use the full 33-point stencil.
//
// Fluxes: LLF of PDEConsFlux (3d/weno3/LinearisedEuler/pde.c:35-95) for
// ACOUSTIC4, the central flux of pde.c:12-34 for WAVE2; both are linear in
// the face states, so the flux of the face averages equals the reference's
// average of Gauss-point fluxes.
//
// Layout: a block covers BX x BY reconstruction columns, the outer ring being
// the face-neighbour halo of the (BX-2) x (BY-2) output tile, and marches a
// chunk of z-planes with the planes of its stencil region in an LDS ring (the
// next plane is loaded one iteration ahead into registers).  x-neighbour face states move by
// lane shuffles inside a 32-lane row, y-neighbours through LDS,
// z-neighbours stay in registers.  k_cweno: the compensated FP32 stage, whose
// selective mode (per-cell flags) replaces the full CWENO by the linear
// 4th-order polynomial wherever the flag bit of a component is 0.
// k_cweno64: the FP64 right-hand side and stages.
#include <algorithm>

#include "acx_device.h"
#include "acx_internal.h"
#include "acx_cweno_core.h"

namespace acx {

enum { EPI_RHS = 0, EPI_AXPY = 1, EPI_COMB = 2, EPI_F32C = 3 };

// Flux across a face normal to axis d from left (+face) and right (-face)
// states: 1/2 (F(Q_L) + F(Q_R) - s (Q_R - Q_L)), F_p = K u_n, F_un = p / rho0.
__device__ __forceinline__ void face_flux(int d, const float (&L)[4], const float (&R)[4], float K, float irho, float s,
                                          float (&F)[4])
{
#pragma unroll
    for (int v = 0; v < 4; ++v) F[v] = -s * (R[v] - L[v]);
    F[0] += K * (L[1 + d] + R[1 + d]);
    F[1 + d] += irho * (L[0] + R[0]);
#pragma unroll
    for (int v = 0; v < 4; ++v) F[v] *= 0.5f;
}

// FP32 compensated stage.  Shared-memory plan of one block (dynamic LDS):
//   ring  [6][NS][BY+4][BX+4]  planes m-2 .. m+3 of the stencil region
//   fy    [2][NS][2][BY][BX]   -y and +y face states of each reconstruction column
// Iteration m reads planes m-2 .. m+2 and takes plane m+3 over plane m-3; with
// two sets of face states and both y fluxes formed by each thread one barrier
// a plane is enough.
struct CwLds {
    static constexpr int BX = 32, BY = 16;   // reconstruction columns per block (output tile 30 x 14)
    static constexpr int NS = 4;
    static constexpr int LX = BX + 4, LY = BY + 4;
    static constexpr int NR = 6;
    static constexpr size_t ring = (size_t)NR * NS * LY * LX;
    static constexpr size_t bytes = (ring + 4ull * NS * BY * BX) * sizeof(float);
};

// Waves per SIMD the register allocation aims for.  The selective patch
// marches a few hundred marked tiles of zc + 2 planes each, and the time of one
// tile's march is what counts: one block per CU without spills (2 waves per
// SIMD) beat two blocks per CU with 60 spilled registers (1.076 against 1.146
// ms for a steep pulse's step at 256^3, 232 marked tiles, one round either
// way).  A 256^3 patch is 56 (first stage) to 61 us (last; 54 and 58 before the
// branch for the smooth side of a jump, when the vector instructions of ten
// planes issued for about 43); it was 84 us with cweno_weights + cweno_combine, a linear branch of its own and each epilogue
// load waited for at its place, and 57 to 61 with two barriers a plane.  The full-grid kernel keeps the registers too.
template <bool SEL>
struct CwWaves {
    static constexpr int min_per_simd = SEL ? 2 : 1;
};

// WALLS = false: every axis periodic (wrap-only index maps, no ghost signs).
// STAGE: F32_FIRST no increment D yet; F32_MID reads D; F32_LAST also adds the
// step's increment to the state HI + LO.
template <bool SEL, bool WALLS, int STAGE>
__global__ void __launch_bounds__(CwLds::BX *CwLds::BY) __attribute__((amdgpu_waves_per_eu(CwWaves<SEL>::min_per_simd)))
k_cweno(CwArgs p)
{
    using T = float;
    using L = CwLds;
    constexpr int NV = 4, NS = L::NS, BX = L::BX, BY = L::BY, NT = BX * BY;
    constexpr int LX = L::LX, LY = L::LY;
    constexpr bool HAS_D = STAGE != F32_FIRST, LAST = STAGE == F32_LAST;
    static_assert(BX == 32, "x exchange uses 32-lane row shuffles");
    extern __shared__ __align__(16) unsigned char smem[];
    T(*ring)[NS][LY][LX] = reinterpret_cast<T(*)[NS][LY][LX]>(smem);
    T(*s_fy)[NS][2][BY][BX] = reinterpret_cast<T(*)[NS][2][BY][BX]>(smem + L::ring * sizeof(T));

    const T *__restrict__ Q = static_cast<const T *>(p.q);
    const T *__restrict__ D = static_cast<const T *>(p.d);
    const T *__restrict__ LO = static_cast<const T *>(p.lo);
    T *__restrict__ OUT = static_cast<T *>(p.out);
    T *__restrict__ OUT2 = static_cast<T *>(p.out2);

    const int nx = p.nx, ny = p.ny, nz = p.nz;
    // Selective patch: the list of marked tiles (count, then tile indices in
    // ascending order), or every tile without a list; block b takes entries
    // b, b + grid, ...  The marked tiles cluster in space (along a front), and
    // consecutive entries go to consecutive blocks, i.e. round-robin over the
    // XCDs.  Only marked tiles are visited: with one block per tile of the
    // grid, the blocks that returned at once on unmarked tiles cost about
    // 16 us per stage at 256^3 and 21 us at 384^3 (4-plane tiles, measured).
    // Otherwise one tile per block, XCD-contiguous.
    int item = blockIdx.x;
    const int nitems = SEL ? (p.tlist ? p.tlist[0] : p.ntx * p.nty * p.ntz) : 1;
    if (SEL && item >= nitems) return;
    bool nfbad = false;   // non-finite watch of this thread's outputs
    do {
        const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * BX + tx;
        const int tile = SEL ? (p.tlist ? p.tlist[1 + item] : item) : xcd_logical_tile(blockIdx.x, gridDim.x);
        const int gx0 = (tile % p.ntx) * (BX - 2) - 1, gy0 = ((tile / p.ntx) % p.nty) * (BY - 2) - 1;
        const int gx = gx0 + tx, gy = gy0 + ty;
        const int zb = (tile / (p.ntx * p.nty)) * p.zc, ze = min(zb + p.zc, nz);
        const bool interior = tx >= 1 && tx <= BX - 2 && ty >= 1 && ty <= BY - 2 && gx < nx && gy < ny;
        const size_t plane = (size_t)nx * ny;
        const int kx = WALLS ? p.bc[0] : 0, ky = WALLS ? p.bc[1] : 0, kz = WALLS ? p.bc[2] : 0;   // boundary kinds

        // own column (mapped) and its ghost sign
        float sx0 = 1.f, sy0 = 1.f;
        const uint32_t ocol = (uint32_t)(map_axis(gy, ny, ky, sy0) * nx + map_axis(gx, nx, kx, sx0));

        // ring cells this thread loads (at most 2 of the (BX+4)(BY+4) region)
        constexpr int NREG = LX * LY;
        constexpr int PER = (NREG + NT - 1) / NT;
        uint32_t rcol[PER];
        float rsx[PER], rsy[PER];
#pragma unroll
        for (int r = 0; r < PER; ++r) {
            const int idx = min(tid + r * NT, NREG - 1);
            rsx[r] = rsy[r] = 1.f;
            const int lx = idx % LX, ly = idx / LX;
            rcol[r] = (uint32_t)(map_axis(gy0 - 2 + ly, ny, ky, rsy[r]) * nx + map_axis(gx0 - 2 + lx, nx, kx, rsx[r]));
        }
        auto zoff = [&](int z, float &s) -> size_t {
            s = 1.f;
            return (size_t)map_axis(z, nz, kz, s) * plane;
        };
        auto slot = [](int m) { return ((m % L::NR) + L::NR) % L::NR; };
        // Every load of the march is unconditional, on clamped cells and
        // planes, so that the compiler counts the loads in flight and waits
        // for the words it needs: loads under a branch were waited for at the
        // branch's end, one memory latency each and up to four a plane.  Plane
        // loads keep the raw words; the FP32 increment and the ghost sign are
        // applied when the plane is stored.
        struct Raw {
            Cell<T, NV> q[PER], d[PER];
            float s;
        };
        auto load_plane = [&](int z, Raw &buf) {
            const size_t off = zoff(z, buf.s);
#pragma unroll
            for (int r = 0; r < PER; ++r) {
                buf.q[r] = load_cell<T, NV>(Q, off + rcol[r]);
                if constexpr (HAS_D) buf.d[r] = load_cell<T, NV>(D, off + rcol[r]);
            }
        };
        auto store_plane = [&](int z, const Raw &buf) {
            const int sl = slot(z);
#pragma unroll
            for (int r = 0; r < PER; ++r) {
                const int idx = tid + r * NT;
                if (idx < NREG) {
                    Cell<T, NV> c = buf.q[r];
                    if constexpr (HAS_D) {
#pragma unroll
                        for (int v = 0; v < NV; ++v) c.v[v] += buf.d[r].v[v];
                    }
                    if constexpr (WALLS) apply_bc_sign<T, NV>(c, rsx[r], rsy[r], buf.s);
#pragma unroll
                    for (int v = 0; v < NS; ++v) ring[sl][v][idx / LX][idx % LX] = c.v[v];
                }
            }
        };

        // prologue: planes zb-3 .. zb+1, all requested before the first is stored
        {
            Raw b0[5];
#pragma unroll
            for (int k = 0; k < 5; ++k) load_plane(zb - 3 + k, b0[k]);
#pragma unroll
            for (int k = 0; k < 5; ++k) store_plane(zb - 3 + k, b0[k]);
        }
        __syncthreads();

        const T K = T(p.K), irho = T(p.invrho), sL = T(p.s);
        T zp_prev[NS], Fz_prev[NS], dxy_prev[NS];
#pragma unroll
        for (int v = 0; v < NS; ++v) { zp_prev[v] = T(0); Fz_prev[v] = T(0); dxy_prev[v] = T(0); }
        const int lx = tx + 2, ly = ty + 2;

        // Plane m+3 is requested in iteration m-1, right after the plane before
        // it went to LDS, and stored in iteration m.
        uint8_t fl_next = 0xff;
        Raw nxt;
        {
            float s;
            if constexpr (SEL) fl_next = p.flags[zoff(zb - 1, s) + ocol];
            load_plane(min(zb + 2, ze + 2), nxt);
        }
        for (int m = zb - 1; m <= ze; ++m) {
            // the flags of plane m+1 and the epilogue operands of plane m-1
            const int set = (m - zb) & 1;
            const uint8_t fl = fl_next;
            if constexpr (SEL) {
                float s;
                fl_next = p.flags[zoff(min(m + 1, ze), s) + ocol];
            }
            const bool fin = m >= zb + 1 && interior;
            const size_t cell = (size_t)max(m - 1, zb) * plane + ocol;
            Cell<T, NV> e0, e1, e2;
            if constexpr (HAS_D) e0 = load_cell<T, NV>(D, cell);
            if constexpr (LAST) {
                e1 = load_cell<T, NV>(LO, cell);
                e2 = load_cell<T, NV>(Q, cell);
            }
            const int sm2 = slot(m - 2), s0 = slot(m - 1), s1 = slot(m), s2 = slot(m + 1), sp2 = slot(m + 2);
            T fpx[NS], fmx[NS], fpy[NS], fmy[NS], fmz[NS], fpz[NS];
#pragma unroll
            for (int v = 0; v < NS; ++v) {
                const T(*P0)[LX] = ring[s0][v];
                const T(*P1)[LX] = ring[s1][v];
                const T(*P2)[LX] = ring[s2][v];
                const T(*M2)[LX] = ring[sm2][v];
                const T(*Q2)[LX] = ring[sp2][v];
                // stencil slot q -> LDS (slot order of cweno_weights)
                auto get = [&](int q) -> T {
                    switch (q) {
                    case 0: return P1[ly][lx];
                    case 1: return P1[ly][lx - 2];
                    case 2: return P1[ly][lx - 1];
                    case 3: return P1[ly][lx + 1];
                    case 4: return P1[ly][lx + 2];
                    case 5: return P1[ly - 2][lx];
                    case 6: return P1[ly - 1][lx];
                    case 7: return P1[ly + 1][lx];
                    case 8: return P1[ly + 2][lx];
                    case 9: return M2[ly][lx];
                    case 10: return P0[ly][lx];
                    case 11: return P2[ly][lx];
                    case 12: return Q2[ly][lx];
                    case 13: return P1[ly + 1][lx + 1];   // xy: ++ +- -+ --
                    case 14: return P1[ly - 1][lx + 1];
                    case 15: return P1[ly + 1][lx - 1];
                    case 16: return P1[ly - 1][lx - 1];
                    case 17: return P2[ly + 1][lx];       // yz (y,z): ++ +- -+ --
                    case 18: return P0[ly + 1][lx];
                    case 19: return P2[ly - 1][lx];
                    case 20: return P0[ly - 1][lx];
                    case 21: return P2[ly][lx + 1];       // zx (z,x): ++ +- -+ --
                    case 22: return P2[ly][lx - 1];
                    case 23: return P0[ly][lx + 1];
                    case 24: return P0[ly][lx - 1];
                    case 25: return P2[ly + 1][lx + 1];   // corners (x,y,z): +++ -++ +-+ ++- --+ -+- +-- ---
                    case 26: return P2[ly + 1][lx - 1];
                    case 27: return P2[ly - 1][lx + 1];
                    case 28: return P0[ly + 1][lx + 1];
                    case 29: return P2[ly - 1][lx - 1];
                    case 30: return P0[ly + 1][lx - 1];
                    case 31: return P0[ly - 1][lx + 1];
                    default: return P0[ly - 1][lx - 1];
                    }
                };

                T m3[3], p3[3];
                cweno_faces<ACX_ACOUSTIC4, T>(get, p, !SEL || ((fl >> v) & 1), m3, p3);
                fmx[v] = m3[0]; fpx[v] = p3[0];
                fmy[v] = m3[1]; fpy[v] = p3[1];
                s_fy[set][v][0][ty][tx] = m3[1];
                s_fy[set][v][1][ty][tx] = p3[1];
                fmz[v] = m3[2]; fpz[v] = p3[2];
                asm volatile("" ::: "memory");   // one component's stencil live at a time
            }
            // over plane m-3, last read before the barrier of iteration m-1
            if (m + 3 <= ze + 2) store_plane(m + 3, nxt);
            load_plane(min(m + 4, ze + 2), nxt);
            __syncthreads();   // y states and plane m+3 visible; every read of plane m-2 is done

            T dxy[NS];
            {
                T Fx[NS], Fy[NS], Fym[NS], Lf[NS], Rf[NS];
#pragma unroll
                for (int v = 0; v < NS; ++v) { Lf[v] = fpx[v]; Rf[v] = __shfl_down(fmx[v], 1, 32); }
                face_flux(0, Lf, Rf, K, irho, sL, Fx);
                // rows without a neighbour are no outputs
                const int up = min(ty + 1, BY - 1), dn = max(ty - 1, 0);
#pragma unroll
                for (int v = 0; v < NS; ++v) Rf[v] = s_fy[set][v][0][up][tx];
                face_flux(1, fpy, Rf, K, irho, sL, Fy);
#pragma unroll
                for (int v = 0; v < NS; ++v) Lf[v] = s_fy[set][v][1][dn][tx];
                face_flux(1, Lf, fmy, K, irho, sL, Fym);
#pragma unroll
                for (int v = 0; v < NS; ++v) dxy[v] = (Fx[v] - __shfl_up(Fx[v], 1, 32)) + (Fy[v] - Fym[v]);
            }

            if (m >= zb) {
                T Fz[NS], Lf[NS], Rf[NS];
#pragma unroll
                for (int v = 0; v < NS; ++v) { Lf[v] = zp_prev[v]; Rf[v] = fmz[v]; }
                face_flux(2, Lf, Rf, K, irho, sL, Fz);
                if (fin) {
                    Cell<T, NV> r;
                    const T ih = T(p.inv_h);
#pragma unroll
                    for (int v = 0; v < 4; ++v) r.v[v] = -ih * (dxy_prev[v] + (Fz[v] - Fz_prev[v]));
                    Cell<T, NV> o;
#pragma unroll
                    for (int v = 0; v < NV; ++v) o.v[v] = (HAS_D ? T(p.b) * e0.v[v] : T(0)) + T(p.c) * r.v[v];
                    if constexpr (LAST) {
                        Cell<T, NV> nh, nl;
#pragma unroll
                        for (int v = 0; v < NV; ++v) {
                            float t = e1.v[v] + o.v[v];
                            float sm, er;
                            two_sum(e2.v[v], t, sm, er);
                            nh.v[v] = sm;
                            nl.v[v] = er;
                        }
                        store_cell<T, NV>(OUT2, cell, nl);
                        o = nh;
                    }
                    if (p.nf) finite_acc<T, NV>(nfbad, o);
                    store_cell<T, NV>(OUT, cell, o);
                }
#pragma unroll
                for (int v = 0; v < NS; ++v) Fz_prev[v] = Fz[v];
            }
#pragma unroll
            for (int v = 0; v < NS; ++v) { zp_prev[v] = fpz[v]; dxy_prev[v] = dxy[v]; }
        }
        if constexpr (SEL) {
            __syncthreads();   // the next tile's prologue rewrites the ring
            item += gridDim.x;
        }
    } while (SEL && item < nitems);
    watch_flush(p.nf, nfbad);
}

// FP64 stage kernel, bound by FP64 issue (cweno_faces: about 265 of the 300
// FP64 instructions per cell and component).  A thread reconstructs at most
// two of the components: an ACOUSTIC4 block is 32 x 12 columns times two halves
// (waves 0-5 p and u, waves 6-11 v and w), a WAVE2 block 32 x 16 columns on
// the one component.  What decided the shape, measured on the 256^3 ACOUSTIC4
// step (8.24 ms with cweno_weights + cweno_combine, four components per
// thread on 32 x 16 columns): the new arithmetic in the old kernel 5.38 ms (256
// VGPRs, 2 waves per SIMD, 24 spilled); two components per thread on 32 x 16
// columns 8.07 ms (128 VGPRs for 4 waves per SIMD, 35 spilled: the scratch
// traffic leaves the L1); on 32 x 12 columns 4.64 ms (3 waves per SIMD, 150 to
// 167 VGPRs, no spills), although the smaller tile recomputes more of its ring
// (outputs are 78 % of the reconstructed columns instead of 82 %).  The WAVE2
// RHS at 70 x 45 x 61 with walls: 31.8 -> 22.0 us.
//
// The LDS ring holds the four planes m-1 .. m+2 of iteration m (each thread
// keeps its own columns' m-1 and m-2 in registers) and takes plane m+3, which
// was requested an iteration before, into a fifth slot; with two sets of the
// exchanged states one barrier a plane is enough.  Against a 4-plane ring and a
// second barrier, us per step: ACOUSTIC4 256^3 4408 -> 4400, 64^3 151.7 ->
// 149.5; WAVE2 70 x 45 x 61 67.6 -> 64.5, 150 x 131 x 90 160 -> 154, 256^3 1338
// -> 1352.  x-neighbour
// face states move by lane shuffles inside a 32-lane row; y-neighbour states
// and, across the two halves of the block, the coupled states (p with v at
// y faces, p with w at z faces; p with u at x faces are in one thread) go
// through LDS.
template <int SYS>
struct Cw64 {
    static constexpr int NS = SYS == ACX_ACOUSTIC4 ? 4 : 1;   // reconstructed components
    static constexpr int NC = SYS == ACX_ACOUSTIC4 ? 2 : 1;   // of them per thread
    static constexpr int NV = SYS == ACX_ACOUSTIC4 ? 4 : 2;   // components in memory
    static constexpr int BX = 32, BY = SYS == ACX_ACOUSTIC4 ? 12 : 16, NCOL = BX * BY;
    static constexpr int NT = NCOL * (NS / NC);
    static constexpr int WPE = SYS == ACX_ACOUSTIC4 ? 3 : 4;  // waves per SIMD
    static constexpr int LX = BX + 4, LY = BY + 4, NREG = LX * LY;
    static constexpr int CS = NREG + 4;                       // doubles per component of a slot
    static constexpr int NR = 5;
    static constexpr int SLOT = NS * CS;
    static constexpr int EX = NS * 2 * NCOL;                  // -y and +y face states
    static constexpr int EZ = SYS == ACX_ACOUSTIC4 ? 2 * NCOL : 0;   // p and w sums at the lower z face
    static constexpr size_t bytes = (size_t)(NR * SLOT + 2 * (EX + EZ)) * sizeof(double);
    static constexpr int NLD = NREG * NV / 2;                 // 16-byte loads of one plane
    static constexpr int PER = (NLD + NT - 1) / NT;
};

template <int SYS, int EPI, bool WALLS>
__global__ void __launch_bounds__(Cw64<SYS>::NT) __attribute__((amdgpu_waves_per_eu(Cw64<SYS>::WPE)))
k_cweno64(CwArgs p)
{
    using L = Cw64<SYS>;
    constexpr int NC = L::NC, NV = L::NV, BX = L::BX, BY = L::BY, LX = L::LX, NCOL = L::NCOL, PER = L::PER;
    constexpr bool AC = SYS == ACX_ACOUSTIC4;
    extern __shared__ __align__(16) unsigned char smem[];
    double *const ring = reinterpret_cast<double *>(smem);
    double *const s_ex = ring + L::NR * L::SLOT;   // two sets of the exchanged states

    const double *__restrict__ Q = static_cast<const double *>(p.q);
    const double *__restrict__ U0 = static_cast<const double *>(p.u0);
    double *__restrict__ OUT = static_cast<double *>(p.out);
    const int nx = p.nx, ny = p.ny, nz = p.nz;
    const size_t plane = (size_t)nx * ny;
    const int kx = WALLS ? p.bc[0] : 0, ky = WALLS ? p.bc[1] : 0, kz = WALLS ? p.bc[2] : 0;

    const int tid = threadIdx.x, colid = tid % NCOL, tx = colid % BX, ty = colid / BX;
    const int half = AC ? __builtin_amdgcn_readfirstlane(tid / NCOL) : 0, v0 = half * NC;
    const int tile = xcd_logical_tile(blockIdx.x, gridDim.x);
    const int gx0 = (tile % p.ntx) * (BX - 2) - 1, gy0 = ((tile / p.ntx) % p.nty) * (BY - 2) - 1;
    const int gx = gx0 + tx, gy = gy0 + ty;
    const int zb = (tile / (p.ntx * p.nty)) * p.zc, ze = min(zb + p.zc, nz);
    const bool interior = tx >= 1 && tx <= BX - 2 && ty >= 1 && ty <= BY - 2 && gx < nx && gy < ny;
    float sx0 = 1.f, sy0 = 1.f;
    const uint32_t ocol = (uint32_t)(map_axis(gy, ny, ky, sy0) * nx + map_axis(gx, nx, kx, sx0));

    // this thread's 16-byte pieces (component pairs) of a plane's region
    uint32_t rcol[PER];
    float rs[PER][2];        // ghost signs of the pair from the x and y axes
    int rdst[PER];           // ring index of its first component
#pragma unroll
    for (int r = 0; r < PER; ++r) {
        const int idx = tid + r * L::NT, cell = idx / (NV / 2), part = idx % (NV / 2);
        rcol[r] = 0;
        rdst[r] = -1;
        rs[r][0] = rs[r][1] = 1.f;
        if (idx < L::NLD) {
            const int lx = cell % LX, ly = cell / LX;
            float sx = 1.f, sy = 1.f;
            const int c = map_axis(gy0 - 2 + ly, ny, ky, sy) * nx + map_axis(gx0 - 2 + lx, nx, kx, sx);
            rcol[r] = (uint32_t)c * (NV / 2) + part;
            rdst[r] = (AC ? 2 * part * L::CS : 0) + cell;
            if constexpr (WALLS) {
                if (AC) {
                    rs[r][0] = part == 0 ? 1.f : sy;   // p, v
                    rs[r][1] = part == 0 ? sx : 1.f;   // u, w
                } else {
                    rs[r][0] = sx * sy;
                }
            }
        }
    }
    auto load_plane = [&](int z, acx_dbl2 (&buf)[PER], float &sz) {
        sz = 1.f;
        const acx_dbl2 *P = reinterpret_cast<const acx_dbl2 *>(Q) + (size_t)map_axis(z, nz, kz, sz) * plane * (NV / 2);
#pragma unroll
        for (int r = 0; r < PER; ++r)
            if (rdst[r] >= 0) buf[r] = P[rcol[r]];
    };
    auto store_plane = [&](int slot, const acx_dbl2 (&buf)[PER], float sz) {
        double *d = ring + slot * L::SLOT;
#pragma unroll
        for (int r = 0; r < PER; ++r)
            if (rdst[r] >= 0) {
                double a = buf[r].x, b = buf[r].y;
                if constexpr (WALLS) {
                    a *= rs[r][0];
                    b *= rs[r][1];
                    if (!AC) a *= sz;
                    else if (rdst[r] >= 2 * L::CS) b *= sz;   // w
                }
                d[rdst[r]] = a;
                if constexpr (AC) d[rdst[r] + L::CS] = b;
            }
    };
    const int cen = (ty + 2) * LX + tx + 2 + v0 * L::CS;   // own column, first own component

    // prologue: planes zb-3 .. zb+2 in flight at once; zb-3 only feeds the
    // column values of iteration zb-1, so its slot is the one of zb+2
    double um1[NC], um2[NC];
    acx_dbl2 nxt[PER];
    float nsz;
    {
        acx_dbl2 b[5][PER];
        float sz[5];
#pragma unroll
        for (int k = 0; k < 5; ++k) load_plane(zb - 3 + k, b[k], sz[k]);
        load_plane(zb + 2, nxt, nsz);
#pragma unroll
        for (int k = 0; k < 5; ++k) store_plane((k + 4) % L::NR, b[k], sz[k]);
        __syncthreads();
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            um2[k] = ring[4 * L::SLOT + cen + k * L::CS];
            um1[k] = ring[cen + k * L::CS];
        }
        __syncthreads();
    }

    const double K = p.K, irho = p.invrho, sL = p.s;
    double zp_prev[NC], Fz_prev[NC], dxy_prev[NC];   // of plane m-1: +z state, flux below, in-plane divergence
#pragma unroll
    for (int k = 0; k < NC; ++k) zp_prev[k] = Fz_prev[k] = dxy_prev[k] = 0.0;
    double vcen = 0.0, vcen_prev = 0.0;
    bool nfbad = false;
    int slot = 0;   // of plane m-1
    auto after = [](int s, int k) { return s + k < L::NR ? s + k : s + k - L::NR; };
    for (int m = zb - 1; m <= ze; ++m) {
        double *const s_y = s_ex + ((m - zb) & 1) * (L::EX + L::EZ);   // [component][-y, +y][column]
        double *const s_z = s_y + L::EX;                               // [p, w][column]
        if constexpr (!AC) {
            float s = 1.f;
            vcen = Q[((size_t)map_axis(m, nz, kz, s) * plane + ocol) * NV + 1];
        }
        const double *R0 = ring + slot * L::SLOT + cen, *R1 = ring + after(slot, 1) * L::SLOT + cen;
        const double *R2 = ring + after(slot, 2) * L::SLOT + cen, *R3 = ring + after(slot, 3) * L::SLOT + cen;
        double fmx[NC], fpx[NC], F[NC];   // F: twice the flux at the face between planes m-1 and m
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            const int o = k * L::CS;
            const double u0 = R1[o];
            // stencil slot q (order of cweno_weights)
            auto get = [&](int q) -> double {
                switch (q) {
                case 0: return u0;
                case 1: return R1[o - 2];
                case 2: return R1[o - 1];
                case 3: return R1[o + 1];
                case 4: return R1[o + 2];
                case 5: return R1[o - 2 * LX];
                case 6: return R1[o - LX];
                case 7: return R1[o + LX];
                case 8: return R1[o + 2 * LX];
                case 9: return um2[k];
                case 10: return um1[k];
                case 11: return R2[o];
                case 12: return R3[o];
                case 13: return R1[o + LX + 1];   // xy: ++ +- -+ --
                case 14: return R1[o - LX + 1];
                case 15: return R1[o + LX - 1];
                case 16: return R1[o - LX - 1];
                case 17: return R2[o + LX];       // yz (y,z): ++ +- -+ --
                case 18: return R0[o + LX];
                case 19: return R2[o - LX];
                case 20: return R0[o - LX];
                case 21: return R2[o + 1];        // zx (z,x): ++ +- -+ --
                case 22: return R2[o - 1];
                case 23: return R0[o + 1];
                case 24: return R0[o - 1];
                case 25: return R2[o + LX + 1];   // corners (x,y,z): +++ -++ +-+ ++- --+ -+- +-- ---
                case 26: return R2[o + LX - 1];
                case 27: return R2[o - LX + 1];
                case 28: return R0[o + LX + 1];
                case 29: return R2[o - LX - 1];
                case 30: return R0[o + LX - 1];
                case 31: return R0[o - LX + 1];
                default: return R0[o - LX - 1];
                }
            };
            double fm[3], fp[3];
            cweno_faces<SYS, double>(get, p, true, fm, fp);
            fmx[k] = fm[0]; fpx[k] = fp[0];
            F[k] = AC ? -sL * (fm[2] - zp_prev[k]) : fm[2] + zp_prev[k];
            if constexpr (AC) {
                if (k == half) s_z[half * NCOL + colid] = fm[2] + zp_prev[k];   // p or w
            }
            zp_prev[k] = fp[2];
            s_y[((v0 + k) * 2 + 0) * NCOL + colid] = fm[1];
            s_y[((v0 + k) * 2 + 1) * NCOL + colid] = fp[1];
            um2[k] = um1[k];
            um1[k] = u0;
            asm volatile("" ::: "memory");   // one component's stencil live at a time
        }

        // plane m+3, over plane m-2 (last read before the barrier of iteration
        // m-1; this iteration's barrier makes it visible)
        if (m + 3 <= ze + 2) store_plane(after(slot, 4), nxt, nsz);
        if (m + 4 <= ze + 2) load_plane(m + 4, nxt, nsz);
        // the base state of plane m-1, requested where the registers of the
        // stencils are free again and ahead of the exchange: waited for at its use,
        // right after its load, it cost a memory latency a plane (combining stage
        // at 256^3 1219 -> 1153 us)
        acx_dbl2 u = {0.0, 0.0};
        const size_t cell = (size_t)max(m - 1, zb) * plane + ocol;
        if constexpr (EPI == EPI_COMB) u = *reinterpret_cast<const acx_dbl2 *>(U0 + cell * NV + v0);

        // x: twice the flux at the +x face, minus the one at the -x face
        double d[NC];
        {
            double G[NC];
#pragma unroll
            for (int k = 0; k < NC; ++k) {
                const double R = __shfl_down(fmx[k], 1, 32);
                if constexpr (AC) {
                    G[k] = -sL * (R - fpx[k]);
                    fmx[k] = R + fpx[k];
                } else {
                    G[k] = R + fpx[k];
                }
            }
            if constexpr (AC) {
                if (half == 0) {
                    G[0] += K * fmx[1];
                    G[1] += irho * fmx[0];
                }
            }
#pragma unroll
            for (int k = 0; k < NC; ++k) d[k] = G[k] - __shfl_up(G[k], 1, 32);
        }
        __syncthreads();   // exchanged states and plane m+3 visible; every read of plane m-1 is done

        // y: both faces from the neighbours' states
        {
            const int up = ty + 1 < BY ? colid + BX : colid, dn = ty > 0 ? colid - BX : colid;
#pragma unroll
            for (int k = 0; k < NC; ++k) {
                const double *e = s_y + (v0 + k) * 2 * NCOL;
                const double R = e[up], Lm = e[NCOL + dn], lo = e[colid], hi = e[NCOL + colid];
                if constexpr (AC) d[k] -= sL * ((R - hi) - (lo - Lm));
                else d[k] += (R + hi) - (lo + Lm);
            }
            if constexpr (AC) {
                // p takes K (v_L + v_R), v takes (p_L + p_R) / rho0: component 0 of either half
                const double *e = s_y + (half ? 0 : 2) * 2 * NCOL;
                d[0] += (half ? irho : K) * ((e[up] + e[NCOL + colid]) - (e[colid] + e[NCOL + dn]));
            }
        }
        // z: the coupled part
        if constexpr (AC) {
            const double o = s_z[(1 - half) * NCOL + colid];
            if (half == 0) F[0] += K * o;
            else F[1] += irho * o;
        }
        if (m >= zb + 1 && interior) {
            double *oc = OUT + cell * NV;
            acx_dbl2 r, q;
            if constexpr (AC) {
                const double ih = -0.5 * p.inv_h;
                r.x = ih * (dxy_prev[0] + (F[0] - Fz_prev[0]));
                r.y = ih * (dxy_prev[1] + (F[1] - Fz_prev[1]));
                q.x = um2[0];   // the column's plane m-1
                q.y = um2[1];
            } else {
                r.x = vcen_prev;
                r.y = 0.5 * p.c2 * (dxy_prev[0] + (F[0] - Fz_prev[0]));
                q.x = um2[0];
                q.y = vcen_prev;
            }
            acx_dbl2 o;
            if constexpr (EPI == EPI_RHS) {
                o = r;
            } else if constexpr (EPI == EPI_AXPY) {
                o = q + p.c * r;
            } else {
                o = p.a * u + p.b * q + p.c * r;
            }
            nfbad |= !__builtin_isfinite(o.x) || !__builtin_isfinite(o.y);
            *reinterpret_cast<acx_dbl2 *>(oc + v0) = o;
        }
#pragma unroll
        for (int k = 0; k < NC; ++k) {
            dxy_prev[k] = d[k];
            Fz_prev[k] = F[k];
        }
        vcen_prev = vcen;
        slot = after(slot, 1);
    }
    watch_flush(p.nf, nfbad);
}

// ---------------------------------------------------------------------------

constexpr int CW_BX = CwLds::BX, CW_BY = CwLds::BY;

// One block per CWENO tile: a tile is marked when a cell of it, or a face
// neighbour of one (a cell of the one-cell ring outside the tile in exactly one
// coordinate, periodic wrap), is flagged; their outputs use the flagged
// reconstruction.  Every entry is written (0 or 1), one store per tile.  Bound by
// the latency of the byte loads, so their chain is short: mask and list of 256^3
// 68 -> 33 us, of 384^3 133 -> 91, against a block per eight tiles along z.
__global__ void __launch_bounds__(256) k_tile_mark(const uint8_t *__restrict__ flags, int nx, int ny, int nz, int zc,
                                                   int ntx, int nty, uint8_t *__restrict__ mask)
{
    static_assert(CW_BX - 2 + 2 <= 32 && CW_BY - 2 + 2 <= 16, "one thread column per box column, two row passes");
    const int col = blockIdx.x % (ntx * nty), z0 = (blockIdx.x / (ntx * nty)) * zc;
    const int x0 = (col % ntx) * (CW_BX - 2), y0 = (col / ntx) * (CW_BY - 2);
    const int bx = min(CW_BX - 2, nx - x0) + 2, by = min(CW_BY - 2, ny - y0) + 2, bz = min(zc, nz - z0) + 2;
    const int lx = threadIdx.x & 31;
    int x = x0 - 1 + lx;
    x = x < 0 ? x + nx : (x >= nx ? x - nx : x);
    const int ex = (lx == 0 || lx == bx - 1);
    int any = 0;
    if (lx < bx) {
        for (int ly = threadIdx.x >> 5; ly < by; ly += 8) {
            int y = y0 - 1 + ly;
            y = y < 0 ? y + ny : (y >= ny ? y - ny : y);
            const int exy = ex + (ly == 0 || ly == by - 1);
            if (exy > 1) continue;
            for (int lz = exy; lz < bz - exy; ++lz) {   // outside in x or y: not also in z
                int z = z0 - 1 + lz;
                z = z < 0 ? z + nz : (z >= nz ? z - nz : z);
                any |= flags[((size_t)z * ny + y) * nx + x];
            }
        }
    }
    any = __syncthreads_or(any);
    if (threadIdx.x == 0) mask[blockIdx.x] = any ? 1 : 0;
}

// The marked tiles as a list: list[0] = their number, list[1 ..] their
// indices in ascending order.  One block walks the mask in chunks of 1024
// entries; a chunk's marked entries are placed by a wavefront ballot and the
// counts of the wavefronts before it.
constexpr int TL_NT = 1024;

__global__ void __launch_bounds__(TL_NT) k_tile_list(const uint8_t *__restrict__ mask, int tiles, int *__restrict__ list)
{
    __shared__ int wcount[TL_NT / 64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int base = 0;
    for (int c0 = 0; c0 < tiles; c0 += TL_NT) {
        const int t = c0 + (int)threadIdx.x;
        const bool on = t < tiles && mask[t] != 0;
        const unsigned long long b = __ballot(on);
        if (lane == 0) wcount[w] = __popcll(b);
        __syncthreads();
        int before = base, total = 0;
#pragma unroll
        for (int k = 0; k < TL_NT / 64; ++k) {
            before += k < w ? wcount[k] : 0;
            total += wcount[k];
        }
        if (on) list[1 + before + __popcll(b & ((1ull << lane) - 1ull))] = t;
        base += total;
        __syncthreads();   // wcount is rewritten by the next chunk
    }
    if (threadIdx.x == 0) list[0] = base;
}

size_t cweno_sel_tiles(const CwArgs &a)
{
    const size_t ntx = (a.nx + CW_BX - 3) / (CW_BX - 2), nty = (a.ny + CW_BY - 3) / (CW_BY - 2);
    return ntx * nty * ((a.nz + a.zc - 1) / a.zc);
}

int launch_cweno_tilemask(const CwArgs &a, const uint8_t *flags, uint8_t *mask, hipStream_t s)
{
    const int ntx = (a.nx + CW_BX - 3) / (CW_BX - 2), nty = (a.ny + CW_BY - 3) / (CW_BY - 2);
    const int ntz = (a.nz + a.zc - 1) / a.zc;
    const size_t tiles = cweno_sel_tiles(a);
    if (tiles > (size_t)INT32_MAX - 1) return set_error(ACX_EUNSUPPORTED, "tile mask: %zu patch tiles", tiles);
    hipLaunchKernelGGL(k_tile_mark, dim3((unsigned)tiles), dim3(256), 0, s, flags, a.nx, a.ny, a.nz, a.zc, ntx, nty, mask);
    int rc = hip_check(hipGetLastError(), "tile mask launch");
    if (rc) return rc;
    hipLaunchKernelGGL(k_tile_list, dim3(1), dim3(TL_NT), 0, s, mask, (int)tiles,
                       reinterpret_cast<int *>(mask + sel_list_offset(tiles)));
    return hip_check(hipGetLastError(), "tile list launch");
}

template <bool SEL, bool WALLS, int STAGE>
static int launch_cw32_w(const CwArgs &a, hipStream_t s)
{
    constexpr int BX = CW_BX, BY = CW_BY;
    CwArgs b = a;
    b.ntx = (a.nx + BX - 3) / (BX - 2);
    b.nty = (a.ny + BY - 3) / (BY - 2);
    if (b.zc <= 0) {
        // round model with a start of 4 planes (the recomputed ring planes and
        // the prologue)
        static int per_cu = 0;
        if (!per_cu) {
            int n = 0;
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                    &n, reinterpret_cast<const void *>(&k_cweno<SEL, WALLS, STAGE>), BX * BY,
                    CwLds::bytes) != hipSuccess || n <= 0)
                n = 1;
            per_cu = n;
        }
        b.zc = auto_zc(b.ntx, b.nty, a.nz, device_cus() * per_cu, 4);
    }
    b.ntz = (a.nz + b.zc - 1) / b.zc;
    size_t blocks = (size_t)b.ntx * b.nty * b.ntz;
    if (SEL && b.tlist) {
        // the marked tiles of the list, at most one round of resident blocks
        static int per_cu_sel = 0;
        if (!per_cu_sel) {
            int n = 0;
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(
                    &n, reinterpret_cast<const void *>(&k_cweno<SEL, WALLS, STAGE>), BX * BY,
                    CwLds::bytes) != hipSuccess || n <= 0)
                n = 1;
            per_cu_sel = n;
        }
        blocks = std::min(blocks, (size_t)device_cus() * per_cu_sel);
    }
    constexpr size_t lds = CwLds::bytes;
    static bool attr_set = false;
    if (!attr_set) {
        int rc = hip_check(hipFuncSetAttribute(reinterpret_cast<const void *>(&k_cweno<SEL, WALLS, STAGE>),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds),
                           "k_cweno LDS attribute");
        if (rc) return rc;
        attr_set = true;
    }
    dim3 blk(BX, BY, 1);
    dim3 grd((unsigned)blocks, 1, 1);
    hipLaunchKernelGGL((k_cweno<SEL, WALLS, STAGE>), grd, blk, lds, s, b);
    return hip_check(hipGetLastError(), "k_cweno launch");
}

template <int SYS, int EPI, bool WALLS>
static int launch_cw64(const CwArgs &a, hipStream_t s)
{
    using L = Cw64<SYS>;
    const void *fn = reinterpret_cast<const void *>(&k_cweno64<SYS, EPI, WALLS>);
    static bool attr_set = false;
    if (!attr_set) {
        int rc = hip_check(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)L::bytes),
                           "k_cweno64 LDS attribute");
        if (rc) return rc;
        attr_set = true;
    }
    CwArgs b = a;
    b.ntx = (a.nx + L::BX - 3) / (L::BX - 2);
    b.nty = (a.ny + L::BY - 3) / (L::BY - 2);
    // Two WAVE2 blocks fit a CU and take 1.5 times as long as one: us per RHS
    // against a model in which they take no longer (or where only one counts),
    // 70 x 45 x 61 12.7 against 15.7 (12.6), 128^3 49.5, 49.4 (57.5).
    if (b.zc <= 0) b.zc = auto_zc(b.ntx, b.nty, a.nz, device_cus(), 4, nullptr, SYS == ACX_WAVE2 ? 1.5 : 0.0);
    b.ntz = (a.nz + b.zc - 1) / b.zc;
    const size_t blocks = (size_t)b.ntx * b.nty * b.ntz;
    hipLaunchKernelGGL((k_cweno64<SYS, EPI, WALLS>), dim3((unsigned)blocks), dim3(L::NT), L::bytes, s, b);
    return hip_check(hipGetLastError(), "k_cweno64 launch");
}

template <int SYS, int EPI>
static int launch_cw64_e(const CwArgs &a, hipStream_t s)
{
    if (a.bc[0] != ACX_PERIODIC || a.bc[1] != ACX_PERIODIC || a.bc[2] != ACX_PERIODIC)
        return launch_cw64<SYS, EPI, true>(a, s);
    return launch_cw64<SYS, EPI, false>(a, s);
}

template <bool SEL>
static int launch_cw32(const CwArgs &a, hipStream_t s)
{
    const bool walls = a.bc[0] != ACX_PERIODIC || a.bc[1] != ACX_PERIODIC || a.bc[2] != ACX_PERIODIC;
    if (a.final_stage)
        return walls ? launch_cw32_w<SEL, true, F32_LAST>(a, s) : launch_cw32_w<SEL, false, F32_LAST>(a, s);
    if (a.d) return walls ? launch_cw32_w<SEL, true, F32_MID>(a, s) : launch_cw32_w<SEL, false, F32_MID>(a, s);
    return walls ? launch_cw32_w<SEL, true, F32_FIRST>(a, s) : launch_cw32_w<SEL, false, F32_FIRST>(a, s);
}

int launch_cweno(const CwArgs &a, int sys, int epi, bool fp32, bool selective, hipStream_t s)
{
    if (fp32) {
        if (epi != EPI_F32C || sys != ACX_ACOUSTIC4)
            return set_error(ACX_EUNSUPPORTED, "fp32 cweno kernel: compensated ACOUSTIC4 stage only");
        return selective ? launch_cw32<true>(a, s) : launch_cw32<false>(a, s);
    }
    if (selective) return set_error(ACX_EUNSUPPORTED, "fp64 cweno kernel: selective mode not built");
    if (sys == ACX_ACOUSTIC4) {
        switch (epi) {
        case EPI_RHS: return launch_cw64_e<ACX_ACOUSTIC4, EPI_RHS>(a, s);
        case EPI_AXPY: return launch_cw64_e<ACX_ACOUSTIC4, EPI_AXPY>(a, s);
        case EPI_COMB: return launch_cw64_e<ACX_ACOUSTIC4, EPI_COMB>(a, s);
        }
    } else {
        switch (epi) {
        case EPI_RHS: return launch_cw64_e<ACX_WAVE2, EPI_RHS>(a, s);
        case EPI_AXPY: return launch_cw64_e<ACX_WAVE2, EPI_AXPY>(a, s);
        case EPI_COMB: return launch_cw64_e<ACX_WAVE2, EPI_COMB>(a, s);
        }
    }
    return set_error(ACX_EUNSUPPORTED, "cweno kernel: unsupported epilogue");
}

} // namespace acx
