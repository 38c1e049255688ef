// acx_ensemble.hip -- persistent-kernel stepping of a batch of independent
// acoustic problems (include/acx_ensemble.h).
//
// The schedule of a configuration is made on the host
// (acx_ensemble_plan.h); the kernel runs its workgroup's list with the same
// tile code as the per-grid linear kernel (acx_linear_core.h).  (A queue per
// XCD drawn from with atomics cost more than the tiles' differences in speed:
// at the end of a stage every workgroup finds eight queues empty, 4000 atomics
// on one line, about 40 us.)
#include <algorithm>
#include <exception>
#include <stdlib.h>
#include <string.h>
#include <type_traits>
#include <vector>
#include "acx_ensemble_plan.h"
#include "acx_linear_core.h"
#include "../../include/acx_ensemble.h"

namespace acx {

constexpr int ENS_MAXP = 256;

constexpr int ENS_NCONFIG = 8;
static const EnsConfig kConfigs[ENS_NCONFIG] = {{8, 16}, {8, 32}, {8, 64}, {12, 16}, {12, 32}, {12, 64},
                                                {8, 128}, {12, 128}};

// WIDE: the march with 64-bit offsets inside a plane (ens_wide).
template <int BY, int STAGE, bool WIDE>
__global__ void __launch_bounds__(ENS_BX *BY) __attribute__((amdgpu_waves_per_eu(STAGE == F32_LAST ? BY / 4 : 4)))
k_ensemble(const EnsProblem *__restrict__ probs, const EnsItem *__restrict__ items, const int *__restrict__ first,
           LinArgs base)
{
    __shared__ typename Tile32<ACX_ACOUSTIC4, BY>::template Shared<STAGE> lds;
    const int end = first[blockIdx.x + 1];
    for (int k = first[blockIdx.x]; k < end; ++k) {
        const EnsItem it = items[k];
        const EnsProblem pr = probs[it.prob];
        const int local = it.tile;
        LinArgs a = base;
        a.nx = pr.n[0];
        a.ny = pr.n[1];
        a.nz = pr.n[2];
        a.ntx = pr.ntx;
        a.nty = pr.nty;
        a.ntz = pr.ntz;
        const size_t o = pr.off * 4;
        a.q = static_cast<const float *>(base.q) + o;
        a.d = base.d ? static_cast<const float *>(base.d) + o : nullptr;
        a.lo = static_cast<const float *>(base.lo) + o;
        a.out = static_cast<float *>(base.out) + o;
        a.out2 = base.out2 ? static_cast<float *>(base.out2) + o : nullptr;
        const int x0 = (local % pr.ntx) * ENS_BX, y0 = ((local / pr.ntx) % pr.nty) * BY;
        a.zc = pr.zc;
        const int zb = (local / (pr.ntx * pr.nty)) * a.zc;
        linear_tile32<ACX_ACOUSTIC4, BY, STAGE, WIDE, true>(a, x0, y0, zb, lds);
        __syncthreads();   // LDS is reused by the next item
    }
}

} // namespace acx

using namespace acx;

// A configuration's problems and its two schedules (stages 1-3, last stage).
struct EnsTables {
    size_t at;                         // offset in d_tables
    const EnsProblem *probs;           // device pointers, null until written
    const EnsItem *items[2];
    const int *first[2];
    int grid[2];                       // workgroups each schedule is made for
};

struct acx_ensemble {
    int nprob;
    double h;
    std::vector<size_t> off;            // first cell of every problem
    std::vector<int> dims;
    bool wide;                         // a problem's planes need the march with 64-bit offsets
    size_t ncell;
    unsigned char *d_tables;           // problems and schedules of every configuration, each in a place of its own
    EnsTables tables[ENS_NCONFIG];     // written on a configuration's first use, never again: launches in flight read them
    float *hi[2], *lo[2], *d0, *d1;
    int cur;                           // index of the current (hi, lo)
    int config;
    int fit[2][2];                     // workgroups that fit at once per rows-per-tile variant (8, 12) and schedule
    hipGraphExec_t graph;
    double graph_dt;
    int graph_config, graph_cur;
    hipStream_t graph_stream;
};

static std::vector<EnsProblem> ens_problems(const acx_ensemble *e, const EnsConfig &c)
{
    return ens_problems(e->dims, e->off, c);
}

static size_t ens_count(const std::vector<EnsProblem> &probs)
{
    size_t n = 0;
    for (const EnsProblem &q : probs) n += (size_t)q.ntx * q.nty * q.ntz;
    return n;
}

// Bytes of a configuration's tables.
static size_t ens_table_bytes(const acx_ensemble *e, const EnsConfig &c)
{
    const int(&fit)[2] = e->fit[c.by == 8 ? 0 : 1];
    const size_t items = ens_count(ens_problems(e, c));
    return sizeof(EnsProblem) * e->nprob + 2 * sizeof(EnsItem) * items + sizeof(int) * (fit[0] + 1 + fit[1] + 1);
}

// Makes and uploads a configuration's tables unless they are there.
static int ens_layout(acx_ensemble *e, int config)
try {
    EnsTables &t = e->tables[config];
    if (t.probs) return ACX_OK;
    const EnsConfig &c = kConfigs[config];
    const EnsPlan plan = ens_plan(ens_problems(e, c), e->fit[c.by == 8 ? 0 : 1]);
    std::vector<unsigned char> h;
    auto put = [&](const auto &v) {   // its offset
        const size_t o = h.size();
        const unsigned char *b = reinterpret_cast<const unsigned char *>(v.data());
        h.insert(h.end(), b, b + v.size() * sizeof(v[0]));
        return o;
    };
    const EnsSchedule(&q)[2] = plan.schedule;
    const size_t at_probs = put(plan.probs);
    const size_t at_items[2] = {put(q[0].items), put(q[1].items)};
    const size_t at_first[2] = {put(q[0].first), put(q[1].first)};
    unsigned char *d = e->d_tables + t.at;
    if (int rc = hip_check(hipMemcpy(d, h.data(), h.size(), hipMemcpyHostToDevice), "ensemble tables")) return rc;
    for (int k = 0; k < 2; ++k) {
        t.items[k] = reinterpret_cast<const EnsItem *>(d + at_items[k]);
        t.first[k] = reinterpret_cast<const int *>(d + at_first[k]);
        t.grid[k] = q[k].blocks();
    }
    t.probs = reinterpret_cast<const EnsProblem *>(d + at_probs);
    return ACX_OK;
} catch (const std::exception &x) {
    return set_error(ACX_EHIP, "ensemble schedule: %s", x.what());
}

// Configuration until tuned: by the work of the busiest workgroup in the
// last, longest stage, and three quarters of the longest item for what the
// workgroups differ in speed (a plane of a 12-row tile takes about 1.3 times
// as long as one of 8 rows).  us per step, this choice and the best of the
// eight: 48 problems of 64 .. 160 cells an edge 3444 and 3383, 12 of 64 .. 128
// 451, 5 330; with the atomic queue and its fixed default 3709, 615, 380.
static int ens_default_config(const acx_ensemble *e)
try {
    int best = 0;
    double best_t = -1.0;
    for (int c = 0; c < ENS_NCONFIG; ++c) {
        const bool r8 = kConfigs[c].by == 8;
        const std::vector<EnsProblem> probs = ens_problems(e, kConfigs[c]);
        int longest = 0;
        for (const EnsProblem &q : probs) longest = std::max(longest, q.zc);
        const EnsSchedule last = ens_schedule(probs, e->fit[r8 ? 0 : 1][ens_schedule_of(F32_LAST)]);
        const double t = (last.most + 0.75 * (longest + 10)) * (r8 ? 1.0 : 1.3);
        if (best_t < 0 || t < best_t) {
            best_t = t;
            best = c;
        }
    }
    return best;
} catch (const std::exception &) {
    return 1;   // 8 rows, 32 planes
}

template <int BY, int STAGE>
static int ens_launch(const acx_ensemble *e, const LinArgs &a, hipStream_t s)
{
    constexpr int k = ens_schedule_of(STAGE);
    const EnsTables &t = e->tables[e->config];
    if (e->wide)
        hipLaunchKernelGGL((k_ensemble<BY, STAGE, true>), dim3(t.grid[k]), dim3(ENS_BX, BY), 0, s, t.probs, t.items[k],
                           t.first[k], a);
    else
        hipLaunchKernelGGL((k_ensemble<BY, STAGE, false>), dim3(t.grid[k]), dim3(ENS_BX, BY), 0, s, t.probs, t.items[k],
                           t.first[k], a);
    return hip_check(hipGetLastError(), "ensemble launch");
}

template <int BY>
static int ens_launch(const acx_ensemble *e, const LinArgs &a, hipStream_t s)
{
    return a.final_stage ? ens_launch<BY, F32_LAST>(e, a, s)
           : a.d         ? ens_launch<BY, F32_MID>(e, a, s)
                         : ens_launch<BY, F32_FIRST>(e, a, s);
}

static int ens_stage(acx_ensemble *e, const float *D, float *OUT, float *OUT2, double b, double c, int final_stage,
                     hipStream_t s)
{
    LinArgs a;
    memset(&a, 0, sizeof(a));
    a.q = e->hi[e->cur];
    a.d = D;
    a.lo = e->lo[e->cur];
    a.out = OUT;
    a.out2 = OUT2;
    a.b = b;
    a.c = c;
    a.final_stage = final_stage;
    a.K = 1.0;
    a.invrho = 1.0;
    a.s = 1.0;
    a.inv48h = 1.0 / (48.0 * e->h);
    a.K_s = a.invrho_s = 1.0;
    a.nf = final_stage ? nonfinite_word_current() : nullptr;   // the step's output is watched
    // bc = periodic (0) from memset
    return kConfigs[e->config].by == 8 ? ens_launch<8>(e, a, s) : ens_launch<12>(e, a, s);
}

static int ens_step(acx_ensemble *e, double dt, hipStream_t s)
{
    const int nxt = 1 - e->cur;
    int rc;
    // same increment sequence as acx_ssp_rks3_step_f32c
    if ((rc = ens_stage(e, nullptr, e->d0, nullptr, 0.0, dt / 2, 0, s))) return rc;
    if ((rc = ens_stage(e, e->d0, e->d1, nullptr, 1.0, dt / 2, 0, s))) return rc;
    if ((rc = ens_stage(e, e->d1, e->d0, nullptr, 1.0 / 3.0, dt / 6, 0, s))) return rc;
    if ((rc = ens_stage(e, e->d0, e->hi[nxt], e->lo[nxt], 1.0, dt / 2, 1, s))) return rc;
    e->cur = nxt;
    return ACX_OK;
}

static int ens_make(acx_ensemble *e, int nprob, const int32_t *n, double h)
{
    e->nprob = nprob;
    e->h = h;
    e->dims.assign(n, n + 3 * nprob);
    e->wide = ens_wide(e->dims);
    e->ncell = 0;
    for (int p = 0; p < nprob; ++p) {
        e->off.push_back(e->ncell);
        e->ncell += (size_t)n[3 * p] * n[3 * p + 1] * n[3 * p + 2];
    }
    (void)nonfinite_word();   // the watch word exists before any capture
    e->graph = nullptr;
    e->graph_stream = nullptr;
    const size_t bytes = e->ncell * 4 * sizeof(float);
    int rc = ACX_OK;
    for (int k = 0; k < 2 && !rc; ++k) {
        rc = hip_check(hipMalloc(&e->hi[k], bytes), "ensemble alloc");
        rc = rc ? rc : hip_check(hipMalloc(&e->lo[k], bytes), "ensemble alloc");
    }
    rc = rc ? rc : hip_check(hipMalloc(&e->d0, bytes), "ensemble alloc");
    rc = rc ? rc : hip_check(hipMalloc(&e->d1, bytes), "ensemble alloc");
    if (!rc) {
        hipMemset(e->hi[0], 0, bytes);
        hipMemset(e->lo[0], 0, bytes);
        e->cur = 0;
        // persistent grids: the blocks that fit at once
        auto fit = [](const void *kernel, int by) {
            int n = 0;
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, ENS_BX * by, 0) != hipSuccess || n < 1) n = 1;
            return n * device_cus();
        };
        auto fits = [&](auto wide) {
            constexpr bool W = decltype(wide)::value;
            e->fit[0][0] = fit(reinterpret_cast<const void *>(&k_ensemble<8, F32_MID, W>), 8);
            e->fit[0][1] = fit(reinterpret_cast<const void *>(&k_ensemble<8, F32_LAST, W>), 8);
            e->fit[1][0] = fit(reinterpret_cast<const void *>(&k_ensemble<12, F32_MID, W>), 12);
            e->fit[1][1] = fit(reinterpret_cast<const void *>(&k_ensemble<12, F32_LAST, W>), 12);
        };
        if (e->wide) fits(std::true_type{});
        else fits(std::false_type{});
        size_t at = 0;
        for (int c = 0; c < ENS_NCONFIG; ++c) {
            e->tables[c].at = at;
            at += (ens_table_bytes(e, kConfigs[c]) + 255) / 256 * 256;
        }
        rc = hip_check(hipMalloc(&e->d_tables, at), "ensemble alloc");
        e->config = ens_default_config(e);
        rc = rc ? rc : ens_layout(e, e->config);
    }
    return rc;
}

extern "C" {

int acx_ensemble_num_configs(void) { return ENS_NCONFIG; }

int acx_ensemble_create(int nprob, const int32_t *n, double h, acx_ensemble **out)
{
    if (nprob < 1 || nprob > ENS_MAXP || !n || !out || !(h > 0)) return set_error(ACX_EINVAL, "ensemble: bad arguments");
    for (int i = 0; i < 3 * nprob; ++i)
        if (n[i] < 4) return set_error(ACX_EINVAL, "ensemble: at least 4 cells per axis");
    acx_ensemble *e = nullptr;
    int rc;
    try {
        e = new acx_ensemble();
        rc = ens_make(e, nprob, n, h);
    } catch (const std::exception &x) {
        rc = set_error(ACX_EHIP, "ensemble: %s", x.what());
    }
    if (rc) {
        acx_ensemble_destroy(e);
        return rc;
    }
    *out = e;
    return ACX_OK;
}

int acx_ensemble_destroy(acx_ensemble *e)
{
    if (!e) return ACX_OK;
    if (e->graph) hipGraphExecDestroy(e->graph);
    hipFree(e->d_tables);
    for (int k = 0; k < 2; ++k) {
        hipFree(e->hi[k]);
        hipFree(e->lo[k]);
    }
    hipFree(e->d0);
    hipFree(e->d1);
    delete e;
    return ACX_OK;
}

int acx_ensemble_offsets(const acx_ensemble *e, size_t *offsets)
{
    if (!e || !offsets) return set_error(ACX_EINVAL, "ensemble: bad arguments");
    for (int p = 0; p < e->nprob; ++p) offsets[p] = e->off[p];
    offsets[e->nprob] = e->ncell;
    return ACX_OK;
}

int acx_ensemble_state(acx_ensemble *e, float **hi, float **lo)
{
    if (!e || !hi || !lo) return set_error(ACX_EINVAL, "ensemble: bad arguments");
    *hi = e->hi[e->cur];
    *lo = e->lo[e->cur];
    return ACX_OK;
}

int acx_ensemble_copy_in(acx_ensemble *e, const float *hi, const float *lo, void *stream)
{
    if (!e || !hi || !lo) return set_error(ACX_EINVAL, "ensemble: bad arguments");
    const size_t bytes = e->ncell * 4 * sizeof(float);
    hipStream_t s = (hipStream_t)stream;
    int rc = hip_check(hipMemcpyAsync(e->hi[e->cur], hi, bytes, hipMemcpyDeviceToDevice, s), "ensemble copy in");
    return rc ? rc : hip_check(hipMemcpyAsync(e->lo[e->cur], lo, bytes, hipMemcpyDeviceToDevice, s), "ensemble copy in");
}

int acx_ensemble_copy_out(const acx_ensemble *e, float *hi, float *lo, void *stream)
{
    if (!e || !hi || !lo) return set_error(ACX_EINVAL, "ensemble: bad arguments");
    const size_t bytes = e->ncell * 4 * sizeof(float);
    hipStream_t s = (hipStream_t)stream;
    int rc = hip_check(hipMemcpyAsync(hi, e->hi[e->cur], bytes, hipMemcpyDeviceToDevice, s), "ensemble copy out");
    return rc ? rc : hip_check(hipMemcpyAsync(lo, e->lo[e->cur], bytes, hipMemcpyDeviceToDevice, s), "ensemble copy out");
}

int acx_ensemble_set_config(acx_ensemble *e, int config)
{
    if (!e || config < 0 || config >= ENS_NCONFIG) return set_error(ACX_EINVAL, "ensemble: config out of range");
    const int rc = ens_layout(e, config);
    if (!rc) e->config = config;
    return rc;
}

int acx_ensemble_get_config(const acx_ensemble *e) { return e ? e->config : -1; }

int acx_ensemble_step(acx_ensemble *e, double dt, void *stream)
{
    if (!e) return set_error(ACX_EINVAL, "ensemble: null");
    if (nonfinite_raised()) return set_error(ACX_ENONFINITE, "ensemble step: a kernel on this device wrote a NaN or Inf");
    return ens_step(e, dt, (hipStream_t)stream);
}

int acx_ensemble_graph_steps(acx_ensemble *e, double dt, int nsteps, void *stream)
{
    if (!e || nsteps < 0 || nsteps % 2) return set_error(ACX_EINVAL, "ensemble: nsteps must be even");
    if (nonfinite_raised()) return set_error(ACX_ENONFINITE, "ensemble steps: a kernel on this device wrote a NaN or Inf");
    hipStream_t s = (hipStream_t)stream;
    int rc;
    if (!e->graph || e->graph_dt != dt || e->graph_config != e->config || e->graph_cur != e->cur) {
        if (e->graph) {
            hipGraphExecDestroy(e->graph);
            e->graph = nullptr;
        }
        hipStream_t cs;
        if ((rc = hip_check(hipStreamCreate(&cs), "ensemble capture stream"))) return rc;
        const int cur0 = e->cur;
        hipGraph_t g;
        rc = hip_check(hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal), "begin capture");
        if (!rc) rc = ens_step(e, dt, cs);
        if (!rc) rc = ens_step(e, dt, cs);
        int rc2 = hip_check(hipStreamEndCapture(cs, &g), "end capture");
        rc = rc ? rc : rc2;
        e->cur = cur0;   // capture did not run anything
        if (!rc) {
            rc = hip_check(hipGraphInstantiate(&e->graph, g, nullptr, nullptr, 0), "graph instantiate");
            hipGraphDestroy(g);
        }
        hipStreamDestroy(cs);
        if (rc) return rc;
        e->graph_dt = dt;
        e->graph_config = e->config;
        e->graph_cur = e->cur;
    }
    for (int k = 0; k < nsteps; k += 2)
        if ((rc = hip_check(hipGraphLaunch(e->graph, s), "graph launch"))) return rc;
    // two steps per replay: the state is back in the same buffer
    return ACX_OK;
}

int acx_ensemble_autotune(acx_ensemble *e, double dt, void *stream, int *best, float *ms_per_step)
{
    if (!e) return set_error(ACX_EINVAL, "ensemble: null");
    hipStream_t s = (hipStream_t)stream;
    const size_t bytes = e->ncell * 4 * sizeof(float);
    float *shi = nullptr, *slo = nullptr;
    int rc = hip_check(hipMalloc(&shi, bytes), "autotune alloc");
    if (!rc) rc = hip_check(hipMalloc(&slo, bytes), "autotune alloc");
    if (!rc) rc = hip_check(hipMemcpyAsync(shi, e->hi[e->cur], bytes, hipMemcpyDeviceToDevice, s), "autotune save");
    if (!rc) rc = hip_check(hipMemcpyAsync(slo, e->lo[e->cur], bytes, hipMemcpyDeviceToDevice, s), "autotune save");
    const int saved_cur = e->cur;
    hipEvent_t a, b;
    hipEventCreate(&a);
    hipEventCreate(&b);
    float bestms = 1e30f;
    int bestc = e->config;
    for (int c = 0; c < ENS_NCONFIG && !rc; ++c) {
        if ((rc = acx_ensemble_set_config(e, c))) break;
        if ((rc = ens_step(e, dt, s))) break;   // warm-up
        hipEventRecord(a, s);
        for (int k = 0; k < 4 && !rc; ++k) rc = ens_step(e, dt, s);
        hipEventRecord(b, s);
        hipEventSynchronize(b);
        float ms = 0.f;
        hipEventElapsedTime(&ms, a, b);
        ms /= 4.f;
        if (ms < bestms) {
            bestms = ms;
            bestc = c;
        }
    }
    hipEventDestroy(a);
    hipEventDestroy(b);
    if (!rc) {
        // restore the state the tuning steps advanced
        e->cur = saved_cur;
        rc = hip_check(hipMemcpyAsync(e->hi[e->cur], shi, bytes, hipMemcpyDeviceToDevice, s), "autotune restore");
        if (!rc) rc = hip_check(hipMemcpyAsync(e->lo[e->cur], slo, bytes, hipMemcpyDeviceToDevice, s), "autotune restore");
        if (!rc) rc = hip_check(hipStreamSynchronize(s), "autotune sync");
        if (!rc) rc = acx_ensemble_set_config(e, bestc);
    }
    hipFree(shi);
    hipFree(slo);
    if (!rc) {
        if (best) *best = bestc;
        if (ms_per_step) *ms_per_step = bestms;
    }
    return rc;
}

} // extern "C"
