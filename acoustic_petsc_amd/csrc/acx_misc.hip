// acx_misc.hip -- FP64 reductions, the CTCS leapfrog sibling and host-side
// synthetic fields.
#include <math.h>
#include <mutex>
#include <stdlib.h>
#include <string.h>
#include <vector>
#include "acx_device.h"
#include "acx_internal.h"

namespace acx {

// ---- deterministic FP64 reductions ---------------------------------------
// Each block reduces a grid-stride slice to (sum, max) with wavefront
// shuffles and leaves them in host-mapped memory; the host adds up the
// partials in a fixed order once the stream has been waited for.  (The last
// block to finish doing it on the device, with the fences that takes in every
// block, made the kernel twice as long; a second launch costs 10 us.)
// Bound by memory: four loads in flight per thread, nontemporal (9 % faster on
// a state larger than the caches, the same on smaller ones), 4 blocks per CU.
// A call on the 537 MB state of 256^3 ACOUSTIC4: all components 210 -> 96
// us, one component 231 -> 98 us (8-byte loads at the cell's stride; before,
// every value with a 64-bit remainder each), energy 140 -> 96 us.
constexpr int RED_THREADS = 256;
constexpr int RED_BLOCKS = 1024;   // most partials of one reduction
constexpr int RED_UNROLL = 4;

// max that keeps a NaN (fmax drops it): a NaN anywhere makes the result NaN,
// as PETSc's VecNorm(NORM_INFINITY) reports it
__host__ __device__ __forceinline__ double nmax(double a, double b) { return (a > b || a != a) ? a : b; }

__device__ __forceinline__ void wave_reduce(double &s, double &m)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        s += __shfl_down(s, off, 64);
        m = nmax(m, __shfl_down(m, off, 64));
    }
}

__device__ __forceinline__ void block_reduce(double &s, double &m)
{
    __shared__ double ss[RED_THREADS / 64], sm[RED_THREADS / 64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    wave_reduce(s, m);
    if (lane == 0) { ss[wv] = s; sm[wv] = m; }
    __syncthreads();
    if (wv == 0) {
        s = lane < RED_THREADS / 64 ? ss[lane] : 0.0;
        m = lane < RED_THREADS / 64 ? sm[lane] : 0.0;
        wave_reduce(s, m);
    }
}

// ---- vector copy ------------------------------------------------------------
// Y = X with nontemporal 16-byte loads and stores, one pair per thread: a
// block covers CP_THREADS * CP_UNROLL pairs.  Measured on MI355X (read +
// write rate, three alternations on one box): a 256^3 FP64 ACOUSTIC4 state
// 6.29 -> 6.52 TB/s and a 384^3 one 6.10 -> 6.43 TB/s against four pairs per
// thread (each thread's loads issued before its first store).  k_copy1 is
// the scalar form for pointers off 16-byte alignment and for the odd last
// element.
constexpr int CP_THREADS = 256, CP_UNROLL = 1;

__global__ void __launch_bounds__(CP_THREADS) k_copy2(const acx_dbl2 *__restrict__ X, acx_dbl2 *__restrict__ Y, size_t n2)
{
    const size_t base = (size_t)blockIdx.x * (CP_THREADS * CP_UNROLL) + threadIdx.x;
    acx_dbl2 v[CP_UNROLL];
#pragma unroll
    for (int u = 0; u < CP_UNROLL; ++u) {
        const size_t i = base + (size_t)u * CP_THREADS;
        if (i < n2) v[u] = __builtin_nontemporal_load(X + i);
    }
#pragma unroll
    for (int u = 0; u < CP_UNROLL; ++u) {
        const size_t i = base + (size_t)u * CP_THREADS;
        if (i < n2) __builtin_nontemporal_store(v[u], Y + i);
    }
}

__global__ void __launch_bounds__(CP_THREADS) k_copy1(const double *__restrict__ X, double *__restrict__ Y, size_t n)
{
    const size_t base = (size_t)blockIdx.x * (CP_THREADS * CP_UNROLL) + threadIdx.x;
    double v[CP_UNROLL];
#pragma unroll
    for (int u = 0; u < CP_UNROLL; ++u) {
        const size_t i = base + (size_t)u * CP_THREADS;
        if (i < n) v[u] = X[i];
    }
#pragma unroll
    for (int u = 0; u < CP_UNROLL; ++u) {
        const size_t i = base + (size_t)u * CP_THREADS;
        if (i < n) Y[i] = v[u];
    }
}

// Blocks for n items, RED_UNROLL per thread and sweep.
static int red_blocks(size_t n)
{
    const size_t per = (size_t)RED_THREADS * RED_UNROLL, b = (n + per - 1) / per;
    return b < 1 ? 1 : b > RED_BLOCKS ? RED_BLOCKS : (int)b;
}

// f(i) over i = 0 .. n-1, RED_UNROLL loads of a thread in flight: get(i)
// loads item i, use(item) accumulates it (items in ascending order per thread).
template <typename Get, typename Use>
__device__ __forceinline__ void red_sweep(size_t n, Get get, Use use)
{
    constexpr size_t span = (size_t)RED_THREADS * RED_UNROLL;
    size_t base = blockIdx.x * span + threadIdx.x;
    const size_t step = gridDim.x * span;
    for (; base + (RED_UNROLL - 1) * RED_THREADS < n; base += step) {
        decltype(get(base)) v[RED_UNROLL];
#pragma unroll
        for (int u = 0; u < RED_UNROLL; ++u) v[u] = get(base + (size_t)u * RED_THREADS);
#pragma unroll
        for (int u = 0; u < RED_UNROLL; ++u) use(v[u]);
    }
    for (; base < n; base += RED_THREADS) use(get(base));   // the last, partial sweep
}

// Sum of squares and largest magnitude: of n2 pairs of values (PAIRS: the
// array is 16-byte aligned and every component counts), or of the n values
// X[0], X[stride], ...
template <bool PAIRS>
__global__ void __launch_bounds__(RED_THREADS)
k_norms(const double *__restrict__ X, size_t n, int stride, double *__restrict__ part)
{
    double s = 0.0, m = 0.0;
    if constexpr (PAIRS) {
        const acx_dbl2 *X2 = reinterpret_cast<const acx_dbl2 *>(X);
        double t = 0.0, k = 0.0;
        red_sweep(n / 2, [&](size_t i) { return __builtin_nontemporal_load(X2 + i); }, [&](acx_dbl2 v) {
            s = fma(v.x, v.x, s);
            t = fma(v.y, v.y, t);
            m = nmax(m, fabs(v.x));
            k = nmax(k, fabs(v.y));
        });
        if ((n & 1) && blockIdx.x == 0 && threadIdx.x == 0) {
            const double v = X[n - 1];
            s = fma(v, v, s);
            m = nmax(m, fabs(v));
        }
        s += t;
        m = nmax(m, k);
    } else {
        red_sweep(n, [&](size_t i) { return __builtin_nontemporal_load(X + i * stride); }, [&](double v) {
            s = fma(v, v, s);
            m = nmax(m, fabs(v));
        });
    }
    block_reduce(s, m);
    if (threadIdx.x == 0) { part[2 * blockIdx.x] = s; part[2 * blockIdx.x + 1] = m; }
}

__global__ void __launch_bounds__(RED_THREADS)
k_diff(const float *__restrict__ HI, const float *__restrict__ LO, const double *__restrict__ B, size_t n,
       double *__restrict__ part)
{
    struct Item { float hi, lo; double b; };
    double s = 0.0, m = 0.0, sb = 0.0, mb = 0.0;
    red_sweep(n, [&](size_t i) { return Item{HI[i], LO ? LO[i] : 0.f, B[i]}; }, [&](const Item &v) {
        const double d = ((double)v.hi + (double)v.lo) - v.b;
        s += d * d;
        m = nmax(m, fabs(d));
        sb += v.b * v.b;
    });
    block_reduce(s, m);
    __syncthreads();
    block_reduce(sb, mb);
    if (threadIdx.x == 0) { part[3 * blockIdx.x] = s; part[3 * blockIdx.x + 1] = m; part[3 * blockIdx.x + 2] = sb; }
}

// Twice the acoustic energy density summed over the cells, as 2 ncell pairs of
// values: (p, u) where the pair index is even, (v, w) where it is odd; a
// thread's pairs are all of one kind.
__global__ void __launch_bounds__(RED_THREADS)
k_energy(const double *__restrict__ U, size_t ncell, double invK, double rho0, double *__restrict__ part)
{
    static_assert(RED_THREADS % 2 == 0, "pair parity per thread");
    const acx_dbl2 *X2 = reinterpret_cast<const acx_dbl2 *>(U);
    const double wx = threadIdx.x & 1 ? rho0 : invK;
    double s = 0.0, t = 0.0, m = 0.0;
    red_sweep(2 * ncell, [&](size_t i) { return __builtin_nontemporal_load(X2 + i); }, [&](acx_dbl2 v) {
        s = fma(v.x, v.x, s);
        t = fma(v.y, v.y, t);
    });
    s = wx * s + rho0 * t;
    block_reduce(s, m);
    if (threadIdx.x == 0) { part[2 * blockIdx.x] = s; part[2 * blockIdx.x + 1] = m; }
}

// The partials of one call (up to three per block) in host-mapped memory.
// Each device keeps RED_SLOTS of them, made on first use and lent to one call
// at a time, so calls on different streams and threads never share one; a
// call that finds none free makes its own.  A call on a 24^3 state, with the
// second launch, the pool allocation and the copy gone: 67 -> 21 us.
constexpr int RED_SLOTS = 16;
constexpr size_t RED_PART = 3 * (size_t)RED_BLOCKS;

struct RedPool {
    double *host = nullptr, *dev = nullptr;
    unsigned used = 0;
};
static RedPool g_red[64];
static std::mutex g_red_mu;

struct RedScratch {
    int device = -1, slot = -1;
    double *host = nullptr, *part = nullptr;   // host and device address of the partials
};

static int red_make(double **host, double **dev, size_t slots)
{
    // an allocation is allowed here while another thread captures a stream
    hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    int rc = hip_check(hipHostMalloc((void **)host, slots * RED_PART * sizeof(double),
                                     hipHostMallocMapped | hipHostMallocCoherent), "reduce scratch");
    if (!rc && (rc = hip_check(hipHostGetDevicePointer((void **)dev, *host, 0), "reduce scratch"))) {
        (void)hipHostFree(*host);
        *host = nullptr;
    }
    (void)hipThreadExchangeStreamCaptureMode(&mode);
    return rc;
}

static int red_take(RedScratch &r, hipStream_t s)
{
    // a reduction waits for its stream, which a capture does not allow
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cap) == hipSuccess && cap != hipStreamCaptureStatusNone)
        return hip_check(hipErrorStreamCaptureUnsupported, "reduce");
    int rc = hip_check(hipGetDevice(&r.device), "reduce scratch: device");
    if (rc) return rc;
    if (r.device >= 0 && r.device < 64) {
        std::lock_guard<std::mutex> lk(g_red_mu);
        RedPool &p = g_red[r.device];
        if (!p.host && (rc = red_make(&p.host, &p.dev, RED_SLOTS))) return rc;
        for (int k = 0; k < RED_SLOTS; ++k)
            if (!(p.used >> k & 1u)) {
                p.used |= 1u << k;
                r.slot = k;
                r.host = p.host + k * RED_PART;
                r.part = p.dev + k * RED_PART;
                return ACX_OK;
            }
    }
    return red_make(&r.host, &r.part, 1);
}

// The launch's error, the wait and the sums over the blocks (out: sum, max,
// third column); the scratch goes back unless the wait failed (its kernel
// might still run).
static int red_finish(RedScratch &r, int nblk, int cols, double (&out)[3], hipStream_t s, const char *what)
{
    const int rc = hip_check(hipGetLastError(), what);
    const int rs = hip_check(hipStreamSynchronize(s), "reduce sync");
    if (rs) return rc ? rc : rs;
    out[0] = out[1] = out[2] = 0.0;
    if (!rc)
        for (int b = 0; b < nblk; ++b) {
            const double *p = r.host + (size_t)cols * b;
            out[0] += p[0];
            out[1] = nmax(out[1], p[1]);
            if (cols > 2) out[2] += p[2];
        }
    if (r.slot >= 0) {
        std::lock_guard<std::mutex> lk(g_red_mu);
        g_red[r.device].used &= ~(1u << r.slot);
    } else {
        (void)hipHostFree(r.host);
    }
    return rc;
}

// ---- CTCS leapfrog (3d/ctcs/point_source/wave.c:138-215) -----------------

// The source's share of one update at its cell (wave.c:234-240), formed once
// per launch on the host: every kernel form adds the same value.
static double ctcs_source_step(const acx_ctcs &c, int it)
{
    const double t = it * c.dt, f0 = c.f0, t0 = 4.0 / f0;
    const double s = -2.0 * (t - t0) * f0 * f0 * exp(-1.0 * f0 * f0 * (t - t0) * (t - t0));
    return s / (c.dx * c.dy * c.dz) * c.dt * c.dt;
}

template <int ST>
__global__ void __launch_bounds__(256)
k_ctcs(const double *__restrict__ Pold, const double *__restrict__ P, double *__restrict__ Pnew,
       const double *__restrict__ C, acx_ctcs c, double src, double *__restrict__ rcv)
{
    const int nx = c.n[0], ny = c.n[1], nz = c.n[2];
    const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y, k = blockIdx.z;
    if (i >= nx) return;
    // periodic wrap of offsets within 2 cells (axes have 1 or at least 5
    // cells); an axis of 1 cell (2D / 1D programs) maps every offset to 0
    auto W = [](int a, int n) { return n == 1 ? 0 : (a < 0 ? a + n : (a >= n ? a - n : a)); };
    auto at = [&](int a, int b, int e) { return P[((size_t)W(e, nz) * ny + W(b, ny)) * nx + W(a, nx)]; };
    const double invdx2 = 1.0 / (c.dx * c.dx), invdy2 = 1.0 / (c.dy * c.dy), invdz2 = 1.0 / (c.dz * c.dz);
    const double p0 = at(i, j, k);
    double pxx, pyy, pzz;
    if (ST == 1) {
        pxx = (at(i + 1, j, k) - 2.0 * p0 + at(i - 1, j, k)) * invdx2;
        pyy = (at(i, j + 1, k) - 2.0 * p0 + at(i, j - 1, k)) * invdy2;
        pzz = (at(i, j, k + 1) - 2.0 * p0 + at(i, j, k - 1)) * invdz2;
    } else {
        pxx = (-1.0 / 12 * at(i + 2, j, k) + 4.0 / 3.0 * at(i + 1, j, k) - 5.0 / 2.0 * p0 + 4.0 / 3.0 * at(i - 1, j, k) -
               1.0 / 12.0 * at(i - 2, j, k)) * invdx2;
        pyy = (-1.0 / 12 * at(i, j + 2, k) + 4.0 / 3.0 * at(i, j + 1, k) - 5.0 / 2.0 * p0 + 4.0 / 3.0 * at(i, j - 1, k) -
               1.0 / 12.0 * at(i, j - 2, k)) * invdy2;
        pzz = (-1.0 / 12 * at(i, j, k + 2) + 4.0 / 3.0 * at(i, j, k + 1) - 5.0 / 2.0 * p0 + 4.0 / 3.0 * at(i, j, k - 1) -
               1.0 / 12.0 * at(i, j, k - 2)) * invdz2;
    }
    const size_t o = ((size_t)k * ny + j) * nx + i;
    const double cc = C[o], dt = c.dt;
    double pn = 2.0 * p0 - Pold[o] + cc * cc * dt * dt * (pxx + pyy + pzz);
    if (i == c.src[0] && j == c.src[1] && k == c.src[2]) pn += src;
    if (rcv && i == c.rcv[0] && j == c.rcv[1] && k == c.rcv[2]) rcv[0] = p0;
    Pnew[o] = pn;
}

// The same update as a 2.5D z-march for 3D grids (every axis >= 5 cells): a
// block owns a 32 x 8 column tile and a chunk of zc planes; each thread
// keeps its column's planes z-ST .. z+ST in registers (the z part of the
// Laplacian) and plane z sits in LDS with an ST-cell x/y halo (double
// buffered, one barrier per plane), so P is read about once per update
// instead of through 13 scattered loads.  Arithmetic as in k_ctcs, term by
// term.  zc: planes per block (32, fewer for small grids, see the launcher).
constexpr int CT_BX = 32, CT_BY = 8;

template <int ST>
__global__ void __launch_bounds__(CT_BX *CT_BY)
k_ctcs_z(const double *__restrict__ Pold, const double *__restrict__ P, double *__restrict__ Pnew,
         const double *__restrict__ C, acx_ctcs c, double src, int zc, double *__restrict__ rcv)
{
    constexpr int LX = CT_BX + 2 * ST, LY = CT_BY + 2 * ST, NH = 2 * ST * (CT_BX + CT_BY);
    static_assert(NH <= CT_BX * CT_BY, "every halo cell of a plane needs a thread of its own");
    __shared__ double pl[2][LY][LX];
    const int nx = c.n[0], ny = c.n[1], nz = c.n[2];
    const int ntx = (nx + CT_BX - 1) / CT_BX, nty = (ny + CT_BY - 1) / CT_BY;
    const int b = blockIdx.x;
    const int x0 = (b % ntx) * CT_BX, y0 = ((b / ntx) % nty) * CT_BY, zb = (b / (ntx * nty)) * zc;
    const int ze = min(zb + zc, nz);
    const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * CT_BX + tx;
    const int i = x0 + tx, j = y0 + ty;
    const bool active = i < nx && j < ny;
    auto M = [](int a, int n) { a %= n; return a < 0 ? a + n : a; };   // set-up only
    auto Wz = [nz](int a) { return a < 0 ? a + nz : (a >= nz ? a - nz : a); };   // |offset| <= ST + 1 < nz
    const size_t plane = (size_t)nx * ny;
    // columns past the grid edge hold the periodic image, so the last tile's
    // LDS row also serves as the wrapped x/y neighbours of the edge cells
    const size_t col = (size_t)M(j, ny) * nx + M(i, nx);
    int hx = -1, hy = -1;
    size_t hcol = 0;
    if (tid < NH) {
        int t = tid;
        if (t < 2 * ST * CT_BY) {
            const int row = t / (2 * ST), k = t % (2 * ST);
            hy = row + ST;
            hx = k < ST ? k : CT_BX + k;
        } else {
            t -= 2 * ST * CT_BY;
            const int cx = t % CT_BX, k = t / CT_BX;
            hx = cx + ST;
            hy = k < ST ? k : CT_BY + k;
        }
        hcol = (size_t)M(y0 + hy - ST, ny) * nx + M(x0 + hx - ST, nx);
    }
    const double invdx2 = 1.0 / (c.dx * c.dx), invdy2 = 1.0 / (c.dy * c.dy), invdz2 = 1.0 / (c.dz * c.dz);
    const double dt = c.dt;
    double q[2 * ST + 1];
#pragma unroll
    for (int d = -ST; d <= ST; ++d) q[d + ST] = P[(size_t)Wz(zb + d) * plane + col];
    int buf = 0;
    for (int z = zb; z < ze; ++z) {
        const double nxt = P[(size_t)Wz(z + ST + 1) * plane + col];   // enters the queue at the end
        const size_t o = (size_t)z * plane + col;
        const double po = Pold[o], cc = C[o];
        pl[buf][ty + ST][tx + ST] = q[ST];
        if (hx >= 0) pl[buf][hy][hx] = P[(size_t)z * plane + hcol];
        __syncthreads();
        if (active) {
            const double p0 = q[ST];
            const double *row = &pl[buf][ty + ST][tx + ST];
            double pxx, pyy, pzz;
            if (ST == 1) {
                pxx = (row[1] - 2.0 * p0 + row[-1]) * invdx2;
                pyy = (pl[buf][ty + ST + 1][tx + ST] - 2.0 * p0 + pl[buf][ty + ST - 1][tx + ST]) * invdy2;
                pzz = (q[2] - 2.0 * p0 + q[0]) * invdz2;
            } else {
                pxx = (-1.0 / 12 * row[2] + 4.0 / 3.0 * row[1] - 5.0 / 2.0 * p0 + 4.0 / 3.0 * row[-1] -
                       1.0 / 12.0 * row[-2]) * invdx2;
                pyy = (-1.0 / 12 * pl[buf][ty + ST + 2][tx + ST] + 4.0 / 3.0 * pl[buf][ty + ST + 1][tx + ST] -
                       5.0 / 2.0 * p0 + 4.0 / 3.0 * pl[buf][ty + ST - 1][tx + ST] -
                       1.0 / 12.0 * pl[buf][ty + ST - 2][tx + ST]) * invdy2;
                pzz = (-1.0 / 12 * q[2 * ST] + 4.0 / 3.0 * q[ST + 1] - 5.0 / 2.0 * p0 + 4.0 / 3.0 * q[ST - 1] -
                       1.0 / 12.0 * q[0]) * invdz2;
            }
            double pn = 2.0 * p0 - po + cc * cc * dt * dt * (pxx + pyy + pzz);
            if (i == c.src[0] && j == c.src[1] && z == c.src[2]) pn += src;
            if (rcv && i == c.rcv[0] && j == c.rcv[1] && z == c.rcv[2]) rcv[0] = p0;
            Pnew[o] = pn;
        }
#pragma unroll
        for (int d = 0; d < 2 * ST; ++d) q[d] = q[d + 1];
        q[2 * ST] = nxt;
        buf ^= 1;
    }
}

// The same update on an LDS-DMA march (3D grids with an even x extent and
// 16-byte aligned arrays): a block of 32 x 16 threads owns a 32 x 16 column
// tile; each plane of P with a 2-cell x/y halo (36 x 20 cells) and the
// tile's Pold and C go straight from memory into one slot of a 5-slot LDS
// ring with global_load_lds_dwordx4 (16 bytes = two x-neighbours per lane).
// At iteration z the slots hold planes z-1 .. z+3: plane z feeds the x/y
// stencils and the update, z+1 and z+2 have landed (z+2 enters the column's
// z-queue of planes z-2 .. z+2 in registers), z+3 and the plane z+4 issued in
// this iteration are in flight.  Loads complete in issue order, so
// s_waitcnt vmcnt(nj) (nj = this wavefront's loads of one plane) means plane
// z+2 has landed in this wavefront's part; one s_barrier then publishes all
// parts and frees the slot of plane z-1 for plane z+4.  The loads are issued
// from inline assembly so that the compiler does not guard every LDS read
// with a wait for all of them.  69.8 KB of LDS per block: two blocks per
// CU.  The arithmetic is k_ctcs_z's term by term.
struct CtDma {
    static constexpr int BX = 32, BY = 16, R = 2;                 // tile, halo loaded (covers ST 1 and 2)
    static constexpr int RW = BX + 2 * R, RH = BY + 2 * R;        // 36 x 20 cells of P
    static constexpr int NP = RW / 2 * RH;                        // 360 entries (cell pairs) of P
    static constexpr int NI = BX / 2 * BY;                        // 256 entries of Pold, and of C
    static constexpr int NENT = NP + 2 * NI;                      // 872
    static constexpr int SLOT = NENT * 16;                        // 13952 bytes
    static constexpr int NSLOT = 5;
    static constexpr int NWAVE = BX * BY / 64;                    // 8
    static constexpr int NCHUNK = (NENT + 63) / 64;               // 14 wavefront loads per plane
    static constexpr int MAXJ = (NCHUNK + NWAVE - 1) / NWAVE;     // 2
};

template <int ST>
__global__ void __launch_bounds__(CtDma::BX *CtDma::BY) __attribute__((amdgpu_waves_per_eu(4)))
k_ctcs_dma(const double *__restrict__ Pold, const double *__restrict__ P, double *__restrict__ Pnew,
           const double *__restrict__ C, acx_ctcs c, double src, int zc, double *__restrict__ rcv)
{
    using D = CtDma;
    __shared__ __attribute__((aligned(16))) unsigned char ring[D::NSLOT * D::SLOT];
    const int nx = c.n[0], ny = c.n[1], nz = c.n[2];
    const int ntx = (nx + D::BX - 1) / D::BX, nty = (ny + D::BY - 1) / D::BY;
    const int b = xcd_logical_tile(blockIdx.x, gridDim.x);
    const int x0 = (b % ntx) * D::BX, y0 = ((b / ntx) % nty) * D::BY, zb = (b / (ntx * nty)) * zc;
    const int ze = min(zb + zc, nz);
    const int tx = threadIdx.x, ty = threadIdx.y, tid = ty * D::BX + tx;
    const int wave = tid >> 6, lane = tid & 63;
    const int i = x0 + tx, j = y0 + ty;
    const bool active = i < nx && j < ny;
    const size_t plane = (size_t)nx * ny;
    auto M = [](int a, int n) { a %= n; return a < 0 ? a + n : a; };

    // this lane's entries: chunk q = wave + 8 k covers entries 64 q .. 64 q + 63
    const int nj = wave + D::NWAVE * (D::MAXJ - 1) < D::NCHUNK ? D::MAXJ : D::MAXJ - 1;
    const double *eptr[D::MAXJ];   // P, Pold or C at the entry's cell of plane 0
    bool eok[D::MAXJ];
#pragma unroll
    for (int k = 0; k < D::MAXJ; ++k) {
        const int e = (wave + D::NWAVE * k) * 64 + lane;
        eok[k] = k < nj && e < D::NENT;
        int gx, gy;
        const double *base;
        if (e < D::NP) {
            const int r = e / (D::RW / 2), cp = e - r * (D::RW / 2);
            gx = M(x0 - D::R + 2 * cp, nx);
            gy = M(y0 - D::R + r, ny);
            base = P;
        } else {
            const int e2 = (e - D::NP) % D::NI, r = e2 / (D::BX / 2), cp = e2 - r * (D::BX / 2);
            gx = M(x0 + 2 * cp, nx);
            gy = M(y0 + r, ny);
            base = e < D::NP + D::NI ? Pold : C;
        }
        eptr[k] = base + (eok[k] ? (size_t)gy * nx + gx : 0);
    }
    auto slot_of = [&](int z) { return (z - zb + 2) % D::NSLOT; };
    auto issue = [&](int z, int slot) {
        const size_t zo = (size_t)M(z, nz) * plane;
        unsigned char *dst = ring + slot * D::SLOT;
#pragma unroll
        for (int k = 0; k < D::MAXJ; ++k) {
            if (k < nj) {
                const unsigned lds = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)(
                    (__attribute__((address_space(3))) unsigned char *)(dst + (wave + D::NWAVE * k) * 1024)));
                const double *g = eptr[k] + zo;
                if (eok[k])
                    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
                                 :: "s"(lds), "v"(g) : "memory", "m0");
            }
        }
    };
    // vmcnt (gfx9 encoding, expcnt 7, lgkmcnt 15): all loads, or all but the
    // nj of the most recent plane
    auto wait_planes = [&](bool keep_last) {
        if (!keep_last) __builtin_amdgcn_s_waitcnt(0x0F70);
        else if (nj == 2) __builtin_amdgcn_s_waitcnt(0x0F72);
        else __builtin_amdgcn_s_waitcnt(0x0F71);
    };
    // P at region row r, column cc of a slot; Pold / C of the tile cell (ty, tx)
    auto pv = [&](int slot, int r, int cc) {
        return *reinterpret_cast<const double *>(ring + slot * D::SLOT + (r * D::RW + cc) * 8);
    };
    auto tile_v = [&](int slot, int part) {
        return *reinterpret_cast<const double *>(ring + slot * D::SLOT + D::NP * 16 + part * D::NI * 16 +
                                                 (ty * D::BX + tx) * 8);
    };

    // prologue: planes zb-2 .. zb+2 into slots 0 .. 4, the column queue, then zb+3
    for (int d = 0; d < D::NSLOT; ++d) issue(zb - 2 + d, d);
    wait_planes(false);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    double q[5];
#pragma unroll
    for (int d = 0; d < 5; ++d) q[d] = pv(d, ty + D::R, tx + D::R);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (zb + 3 <= ze + 1) issue(zb + 3, slot_of(zb + 3));

    const double invdx2 = 1.0 / (c.dx * c.dx), invdy2 = 1.0 / (c.dy * c.dy), invdz2 = 1.0 / (c.dz * c.dz);
    const double dt = c.dt;
    const size_t col = (size_t)M(j, ny) * nx + M(i, nx);
    for (int z = zb; z < ze; ++z) {
        if (z > zb) {
            // plane z+2 landed: only plane z+3's loads may be outstanding
            wait_planes(z + 3 <= ze + 1);
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
#pragma unroll
            for (int d = 0; d < 4; ++d) q[d] = q[d + 1];
            q[4] = pv(slot_of(z + 2), ty + D::R, tx + D::R);
        }
        // every wavefront is past iteration z-1: its slot takes plane z+4
        if (z + 4 <= ze + 1) issue(z + 4, slot_of(z + 4));
        const int s0 = slot_of(z);
        if (active) {
            const double p0 = q[2];
            const double po = tile_v(s0, 0), cc = tile_v(s0, 1);
            const int r0 = ty + D::R, c0 = tx + D::R;
            double pxx, pyy, pzz;
            if (ST == 1) {
                pxx = (pv(s0, r0, c0 + 1) - 2.0 * p0 + pv(s0, r0, c0 - 1)) * invdx2;
                pyy = (pv(s0, r0 + 1, c0) - 2.0 * p0 + pv(s0, r0 - 1, c0)) * invdy2;
                pzz = (q[3] - 2.0 * p0 + q[1]) * invdz2;
            } else {
                pxx = (-1.0 / 12 * pv(s0, r0, c0 + 2) + 4.0 / 3.0 * pv(s0, r0, c0 + 1) - 5.0 / 2.0 * p0 +
                       4.0 / 3.0 * pv(s0, r0, c0 - 1) - 1.0 / 12.0 * pv(s0, r0, c0 - 2)) * invdx2;
                pyy = (-1.0 / 12 * pv(s0, r0 + 2, c0) + 4.0 / 3.0 * pv(s0, r0 + 1, c0) - 5.0 / 2.0 * p0 +
                       4.0 / 3.0 * pv(s0, r0 - 1, c0) - 1.0 / 12.0 * pv(s0, r0 - 2, c0)) * invdy2;
                pzz = (-1.0 / 12 * q[4] + 4.0 / 3.0 * q[3] - 5.0 / 2.0 * p0 + 4.0 / 3.0 * q[1] -
                       1.0 / 12.0 * q[0]) * invdz2;
            }
            double pn = 2.0 * p0 - po + cc * cc * dt * dt * (pxx + pyy + pzz);
            if (i == c.src[0] && j == c.src[1] && z == c.src[2]) pn += src;
            if (rcv && i == c.rcv[0] && j == c.rcv[1] && z == c.rcv[2]) rcv[0] = p0;
            Pnew[(size_t)z * plane + col] = pn;
        }
    }
    // every load issued has been waited for by the last iteration (vmcnt 0)
}

// The same update for 3D grids that live in the caches between steps (even x
// extent, 16-byte aligned arrays): one thread per pair of x-neighbours, 13
// 16-byte loads all in flight at once instead of a march along z.
// Arithmetic as in k_ctcs, term by term.  At the sizes of ctcs_route the march
// is bound by the latency of its planes, not by bytes.
constexpr int CD_THREADS = 256;

template <int ST>
__global__ void __launch_bounds__(CD_THREADS)
k_ctcs_pair(const double *__restrict__ Pold, const double *__restrict__ P, double *__restrict__ Pnew,
            const double *__restrict__ C, acx_ctcs c, double src, int bpp, double *__restrict__ rcv)
{
    const int np = c.n[0] / 2, ny = c.n[1], nz = c.n[2];
    const int b = xcd_logical_tile(blockIdx.x, gridDim.x), k = b / bpp;
    const unsigned e = (unsigned)(b - k * bpp) * CD_THREADS + threadIdx.x;   // pair of the plane
    if (e >= (unsigned)np * (unsigned)ny) return;
    const int j = (int)(e / (unsigned)np), i2 = (int)(e - (unsigned)j * (unsigned)np);
    auto W = [](int a, int n) { return a < 0 ? a + n : (a >= n ? a - n : a); };
    const acx_dbl2 *P2 = reinterpret_cast<const acx_dbl2 *>(P);
    auto at = [&](int a, int bb, int d) {
        return P2[((size_t)W(k + d, nz) * ny + W(j + bb, ny)) * np + W(i2 + a, np)];
    };
    const size_t o = ((size_t)k * ny + j) * np + i2;
    const acx_dbl2 p0 = P2[o], xm = at(-1, 0, 0), xp = at(1, 0, 0);
    const acx_dbl2 ym1 = at(0, -1, 0), yp1 = at(0, 1, 0), zm1 = at(0, 0, -1), zp1 = at(0, 0, 1);
    acx_dbl2 ym2 = p0, yp2 = p0, zm2 = p0, zp2 = p0;
    if (ST == 2) {
        ym2 = at(0, -2, 0);
        yp2 = at(0, 2, 0);
        zm2 = at(0, 0, -2);
        zp2 = at(0, 0, 2);
    }
    const acx_dbl2 po = reinterpret_cast<const acx_dbl2 *>(Pold)[o], cc = reinterpret_cast<const acx_dbl2 *>(C)[o];
    const double x[6] = {xm.x, xm.y, p0.x, p0.y, xp.x, xp.y};
    const double invdx2 = 1.0 / (c.dx * c.dx), invdy2 = 1.0 / (c.dy * c.dy), invdz2 = 1.0 / (c.dz * c.dz);
    const double dt = c.dt;
    acx_dbl2 r;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const double q = x[2 + h];
        double pxx, pyy, pzz;
        if (ST == 1) {
            pxx = (x[3 + h] - 2.0 * q + x[1 + h]) * invdx2;
            pyy = (yp1[h] - 2.0 * q + ym1[h]) * invdy2;
            pzz = (zp1[h] - 2.0 * q + zm1[h]) * invdz2;
        } else {
            pxx = (-1.0 / 12 * x[4 + h] + 4.0 / 3.0 * x[3 + h] - 5.0 / 2.0 * q + 4.0 / 3.0 * x[1 + h] -
                   1.0 / 12.0 * x[h]) * invdx2;
            pyy = (-1.0 / 12 * yp2[h] + 4.0 / 3.0 * yp1[h] - 5.0 / 2.0 * q + 4.0 / 3.0 * ym1[h] - 1.0 / 12.0 * ym2[h]) *
                  invdy2;
            pzz = (-1.0 / 12 * zp2[h] + 4.0 / 3.0 * zp1[h] - 5.0 / 2.0 * q + 4.0 / 3.0 * zm1[h] - 1.0 / 12.0 * zm2[h]) *
                  invdz2;
        }
        double pn = 2.0 * q - po[h] + cc[h] * cc[h] * dt * dt * (pxx + pyy + pzz);
        const int i = 2 * i2 + h;
        if (i == c.src[0] && j == c.src[1] && k == c.src[2]) pn += src;
        if (rcv && i == c.rcv[0] && j == c.rcv[1] && k == c.rcv[2]) rcv[0] = q;
        r[h] = pn;
    }
    reinterpret_cast<acx_dbl2 *>(Pnew)[o] = r;
}

static int check_ctcs(const acx_ctcs *c, const double *POLD, const double *P, const double *PNEW, const double *C)
{
    if (!c || !POLD || !P || !PNEW || !C || PNEW == P) return set_error(ACX_EINVAL, "ctcs: bad arguments");
    for (int d = 0; d < 3; ++d)
        if (c->n[d] < 5 && c->n[d] != 1) return set_error(ACX_EINVAL, "ctcs: at least 5 cells per axis (or 1)");
    if (c->stencil != 1 && c->stencil != 2) return set_error(ACX_EINVAL, "stencil width can be either 1 or 2");
    return ACX_OK;
}

// One leapfrog update; rcv (device, may be null) receives P at the receiver.
static int launch_ctcs(const acx_ctcs *c, const double *POLD, const double *P, double *PNEW, const double *C, int it,
                       double *rcv, hipStream_t s)
{
    const double src = ctcs_source_step(*c, it);
    const int route = ctcs_route(c->n[0], c->n[1], c->n[2], (uintptr_t)POLD | (uintptr_t)P | (uintptr_t)C, (uintptr_t)PNEW);
    if (route == CTCS_PAIRS) {
        const size_t bpp = ((size_t)c->n[0] / 2 * c->n[1] + CD_THREADS - 1) / CD_THREADS;
        dim3 blk(CD_THREADS), grd((unsigned)(bpp * c->n[2]));
        if (c->stencil == 1) hipLaunchKernelGGL(k_ctcs_pair<1>, grd, blk, 0, s, POLD, P, PNEW, C, *c, src, (int)bpp, rcv);
        else hipLaunchKernelGGL(k_ctcs_pair<2>, grd, blk, 0, s, POLD, P, PNEW, C, *c, src, (int)bpp, rcv);
    } else if (route == CTCS_DMA) {
        // 3D, LDS-DMA march: z-chunk from the round model, two blocks per CU
        // (measured at 256^3: 144 -> 152 G cell-updates/s, bit-identical to
        // the register-queue march below)
        const int ntx = (c->n[0] + CtDma::BX - 1) / CtDma::BX, nty = (c->n[1] + CtDma::BY - 1) / CtDma::BY;
        const int zc = auto_zc(ntx, nty, c->n[2], device_cus() * 2, 4);
        const size_t nb = (size_t)ntx * nty * ((c->n[2] + zc - 1) / zc);
        dim3 blk(CtDma::BX, CtDma::BY), grd((unsigned)nb);
        if (c->stencil == 1) hipLaunchKernelGGL(k_ctcs_dma<1>, grd, blk, 0, s, POLD, P, PNEW, C, *c, src, zc, rcv);
        else hipLaunchKernelGGL(k_ctcs_dma<2>, grd, blk, 0, s, POLD, P, PNEW, C, *c, src, zc, rcv);
    } else if (route == CTCS_MARCH) {
        // 3D: z-march; 32 planes per block, halved (down to 4) below 1024 blocks
        const size_t cols = (size_t)((c->n[0] + CT_BX - 1) / CT_BX) * ((c->n[1] + CT_BY - 1) / CT_BY);
        int zc = 32;
        while (zc > 4 && cols * ((c->n[2] + zc - 1) / zc) < 1024) zc /= 2;
        const size_t nb = cols * ((c->n[2] + zc - 1) / zc);
        dim3 blk(CT_BX, CT_BY), grd((unsigned)nb);
        if (c->stencil == 1) hipLaunchKernelGGL(k_ctcs_z<1>, grd, blk, 0, s, POLD, P, PNEW, C, *c, src, zc, rcv);
        else hipLaunchKernelGGL(k_ctcs_z<2>, grd, blk, 0, s, POLD, P, PNEW, C, *c, src, zc, rcv);
    } else {
        // 2D / 1D programs (axes of one cell): one thread per cell
        dim3 blk(256), grd((c->n[0] + 255) / 256, c->n[1], c->n[2]);
        if (c->stencil == 1) hipLaunchKernelGGL(k_ctcs<1>, grd, blk, 0, s, POLD, P, PNEW, C, *c, src, rcv);
        else hipLaunchKernelGGL(k_ctcs<2>, grd, blk, 0, s, POLD, P, PNEW, C, *c, src, rcv);
    }
    return hip_check(hipGetLastError(), "ctcs launch");
}

// ---- host fields ---------------------------------------------------------

static inline uint64_t splitmix64(uint64_t &s)
{
    uint64_t z = (s += 0x9e3779b97f4a7c15ULL);
    z = (z ^ (z >> 30)) * 0xbf58476d1ce4e5b9ULL;
    z = (z ^ (z >> 27)) * 0x94d049bb133111ebULL;
    return z ^ (z >> 31);
}
static inline double unif(uint64_t &s) { return (splitmix64(s) >> 11) * (1.0 / 9007199254740992.0); }

// 1D cell averages of exp(-(x-c)^2/(2 sigma^2)) on the periodic unit interval
static void gauss_1d(int n, double h, double c, double sigma, std::vector<double> &out)
{
    out.assign(n, 0.0);
    const double k = sigma * sqrt(M_PI / 2.0) / h, r = 1.0 / (sigma * sqrt(2.0));
    for (int i = 0; i < n; ++i) {
        const double a = i * h, b = (i + 1) * h;
        double acc = 0.0;
        for (int img = -1; img <= 1; ++img) acc += erf((b - c + img) * r) - erf((a - c + img) * r);
        out[i] = k * acc;
    }
}

} // namespace acx

using namespace acx;

extern "C" {

int acx_norms_f64(const double *X, size_t ncells, int nvar, int comp, double *out, void *stream)
{
    if (!X || !out || nvar < 1 || comp >= nvar) return set_error(ACX_EINVAL, "norms: bad arguments");
    hipStream_t s = (hipStream_t)stream;
    RedScratch sc;
    int rc = red_take(sc, s);
    if (rc) return rc;
    const size_t n = comp < 0 ? ncells * nvar : ncells;
    const bool pairs = comp < 0 && ((uintptr_t)X & 15) == 0;
    const int nblk = red_blocks(pairs ? n / 2 : n);
    if (pairs)
        hipLaunchKernelGGL(k_norms<true>, dim3(nblk), dim3(RED_THREADS), 0, s, X, n, 1, sc.part);
    else
        hipLaunchKernelGGL(k_norms<false>, dim3(nblk), dim3(RED_THREADS), 0, s, comp < 0 ? X : X + comp, n,
                           comp < 0 ? 1 : nvar, sc.part);
    double r[3];
    if ((rc = red_finish(sc, nblk, 2, r, s, "norms launch"))) return rc;
    out[0] = r[0];
    out[1] = r[1];
    return ACX_OK;
}

int acx_vec_copy_f64(const double *X, double *Y, size_t n, void *stream)
{
    if (n == 0) return ACX_OK;
    if (!X || !Y) return set_error(ACX_EINVAL, "vec copy: null pointer");
    if ((X < Y + n) && (Y < X + n) && X != Y) return set_error(ACX_EINVAL, "vec copy: overlapping arrays");
    if (X == Y) return ACX_OK;
    hipStream_t s = (hipStream_t)stream;
    const size_t per_block = (size_t)CP_THREADS * CP_UNROLL;
    const bool aligned = (((uintptr_t)X | (uintptr_t)Y) & 15) == 0;
    const size_t nv = aligned ? n / 2 : n;                 // elements of the main launch
    const size_t blocks = (nv + per_block - 1) / per_block;
    if (blocks > 0x7fffffffULL) return set_error(ACX_EINVAL, "vec copy: %zu elements is too many", n);
    if (blocks) {
        if (aligned)
            hipLaunchKernelGGL(k_copy2, dim3((unsigned)blocks), dim3(CP_THREADS), 0, s, (const acx_dbl2 *)X,
                               (acx_dbl2 *)Y, nv);
        else
            hipLaunchKernelGGL(k_copy1, dim3((unsigned)blocks), dim3(CP_THREADS), 0, s, X, Y, nv);
    }
    if (aligned && (n & 1)) hipLaunchKernelGGL(k_copy1, dim3(1), dim3(CP_THREADS), 0, s, X + n - 1, Y + n - 1, (size_t)1);
    return hip_check(hipGetLastError(), "vec copy");
}

int acx_diff_f32c_f64(const float *HI, const float *LO, const double *B, size_t n, double *out, void *stream)
{
    if (!HI || !B || !out) return set_error(ACX_EINVAL, "diff: bad arguments");
    hipStream_t s = (hipStream_t)stream;
    RedScratch sc;
    int rc = red_take(sc, s);
    if (rc) return rc;
    const int nblk = red_blocks(n);
    hipLaunchKernelGGL(k_diff, dim3(nblk), dim3(RED_THREADS), 0, s, HI, LO, B, n, sc.part);
    double r[3];
    if ((rc = red_finish(sc, nblk, 3, r, s, "diff launch"))) return rc;
    out[0] = r[2] > 0 ? sqrt(r[0] / r[2]) : sqrt(r[0]);
    out[1] = r[1];
    return ACX_OK;
}

int acx_energy_f64(const acx_grid *g, const double *U, double *out, void *stream)
{
    if (!g || !U || !out || g->system != ACX_ACOUSTIC4) return set_error(ACX_EINVAL, "energy: ACOUSTIC4 state required");
    hipStream_t s = (hipStream_t)stream;
    RedScratch sc;
    int rc = red_take(sc, s);
    if (rc) return rc;
    const size_t nc = (size_t)g->n[0] * g->n[1] * g->n[2];
    const double K = g->rho0 * g->c0 * g->c0;
    const int nblk = red_blocks(2 * nc);
    hipLaunchKernelGGL(k_energy, dim3(nblk), dim3(RED_THREADS), 0, s, U, nc, 1.0 / K, g->rho0, sc.part);
    double r[3];
    if ((rc = red_finish(sc, nblk, 2, r, s, "energy launch"))) return rc;
    out[0] = 0.5 * r[0] * g->h * g->h * (g->n[2] == 1 ? 1.0 : g->h);   // cell area on a 2D grid
    return ACX_OK;
}

int acx_ctcs_update_f64(const acx_ctcs *c, const double *POLD, const double *P, double *PNEW, const double *C,
                        int it, double *rcv_out, void *stream)
{
    int rc = check_ctcs(c, POLD, P, PNEW, C);
    if (rc) return rc;
    hipStream_t s = (hipStream_t)stream;
    // the receiver sample goes through a one-value buffer of this call (none
    // when the caller does not ask for it)
    double *rcv = nullptr;
    if (rcv_out) {
        const int ra = hip_check(hipMallocAsync((void **)&rcv, sizeof(double), s), "ctcs receiver buffer");
        if (ra) return ra;
    }
    rc = launch_ctcs(c, POLD, P, PNEW, C, it, rcv, s);
    if (rcv_out) {
        if (!rc) rc = hip_check(hipMemcpyAsync(rcv_out, rcv, sizeof(double), hipMemcpyDeviceToHost, s), "ctcs rcv copy");
        const int rf = hip_check(hipFreeAsync(rcv, s), "ctcs receiver buffer free");
        if (!rc) rc = rf;
        if (!rc) rc = hip_check(hipStreamSynchronize(s), "ctcs sync");
    }
    return rc;
}

int acx_ctcs_steps_f64(const acx_ctcs *c, double *POLD, double *P, double *PNEW, const double *C, int it, int nt,
                       double *trace, void *stream)
{
    if (nt < 0) return set_error(ACX_EINVAL, "ctcs: nt must be >= 0");
    int rc = check_ctcs(c, POLD, P, PNEW, C);
    if (!rc && (POLD == P || POLD == PNEW)) rc = set_error(ACX_EINVAL, "ctcs: the three time levels must be distinct");
    for (int k = 0; k < nt && !rc; ++k) {
        rc = launch_ctcs(c, POLD, P, PNEW, C, it + k, trace ? trace + k : nullptr, (hipStream_t)stream);
        double *t = POLD;
        POLD = P;
        P = PNEW;
        PNEW = t;
    }
    return rc;
}

int acx_field_gaussians(const acx_grid *g, uint64_t seed, int npulse, double amin, double amax, double smin,
                        double smax, double *U)
{
    if (!g || !U || npulse < 0) return set_error(ACX_EINVAL, "field: bad arguments");
    const int nx = g->n[0], ny = g->n[1], nz = g->n[2], nv = g->system == ACX_ACOUSTIC4 ? 4 : 2;
    const size_t nc = (size_t)nx * ny * nz;
    memset(U, 0, nc * nv * sizeof(double));
    uint64_t st = seed;
    std::vector<double> fx, fy, fz;
    for (int q = 0; q < npulse; ++q) {
        const double A = amin + (amax - amin) * unif(st);
        const double sg = smin + (smax - smin) * unif(st);
        const double cx = unif(st), cy = unif(st), cz = unif(st);
        gauss_1d(nx, 1.0 / nx, cx, sg, fx);
        gauss_1d(ny, 1.0 / ny, cy, sg, fy);
        gauss_1d(nz, 1.0 / nz, cz, sg, fz);
        for (int k = 0; k < nz; ++k)
            for (int j = 0; j < ny; ++j) {
                const double a = A * fz[k] * fy[j];
                double *row = U + ((size_t)k * ny + j) * nx * nv;
                for (int i = 0; i < nx; ++i) row[(size_t)i * nv] += a * fx[i];
            }
    }
    return ACX_OK;
}

int acx_field_plane_wave(const acx_grid *g, const int k[3], double A, double t, double *U)
{
    if (!g || !U || g->system != ACX_ACOUSTIC4) return set_error(ACX_EINVAL, "plane wave: ACOUSTIC4 grid required");
    const int nx = g->n[0], ny = g->n[1], nz = g->n[2];
    const double kk = sqrt((double)k[0] * k[0] + (double)k[1] * k[1] + (double)k[2] * k[2]);
    if (kk == 0) return set_error(ACX_EINVAL, "plane wave: k = 0");
    const double w = 2.0 * M_PI * kk * g->c0;
    // cell averages: point value at the centre times prod sinc(pi k_d h_d)
    auto sinc = [](double x) { return x == 0 ? 1.0 : sin(x) / x; };
    const double damp = sinc(M_PI * k[0] / nx) * sinc(M_PI * k[1] / ny) * sinc(M_PI * k[2] / nz);
    const double ap = A * cos(w * t) * damp, au = -(A / (g->rho0 * g->c0)) * sin(w * t) * damp;
    for (int c = 0; c < nz; ++c)
        for (int b = 0; b < ny; ++b)
            for (int a = 0; a < nx; ++a) {
                const double th = 2.0 * M_PI * (k[0] * (a + 0.5) / nx + k[1] * (b + 0.5) / ny + k[2] * (c + 0.5) / nz);
                double *o = U + (((size_t)c * ny + b) * nx + a) * 4;
                const double sn = sin(th), cs = cos(th);
                o[0] = ap * sn;
                o[1] = au * (k[0] / kk) * cs;
                o[2] = au * (k[1] / kk) * cs;
                o[3] = au * (k[2] / kk) * cs;
            }
    return ACX_OK;
}

} // extern "C"
