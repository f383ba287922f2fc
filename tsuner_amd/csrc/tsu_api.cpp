// tsu_api.cpp -- host runtime behind the libtsuner C ABI (include/tsuner.h).
//
// A tsu_state owns everything one simulation needs on one device: two
// planar SoA state buffers (U^n and the first RK stage), the bed mask as
// bytes, the inflow series, the step-control block and one stream.  Steps are
// enqueued without host synchronisation: dt and the simulation time live on
// the device (GPU/main_TSUNER.cu:147-197 keeps them on the host and blocks on
// a device-to-host copy every step).
#define TSU_BUILDING_LIBRARY 1
#include "../../include/tsuner.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <climits>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "tsu_host.h"
#include "tsu_kernels.h"

using tsu::Ctrl;
using tsu::DevParams;

namespace {

thread_local std::string g_err;

int fail(int code, const std::string& msg)
{
    g_err = msg;
    return code;
}

#define HIPCHK(expr)                                                                        \
    do {                                                                                    \
        hipError_t e_ = (expr);                                                             \
        if (e_ != hipSuccess) return fail(TSU_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)); \
    } while (0)


double bitsd(unsigned long long b)
{
    double v;
    std::memcpy(&v, &b, 8);
    return v;
}

// Host twin of tsu::finalize_dt.
double finalize_host(const DevParams& P, unsigned long long bits)
{
    double m = bitsd(bits);
    if (P.dt_narrow && P.nvol > 4096) m = (double)(float)m;
    return (m < 1e30) ? m : 1e30;
}

int check_scheme(const tsu_scheme* s)
{
    if (s->order != 1 && s->order != 2) return fail(TSU_ERR_UNSUPPORTED, "order must be 1 or 2");
    for (int i = 0; i < 4; i++)
        if (s->bc[i] < TSU_BC_FREE || s->bc[i] > TSU_BC_INFLOW) return fail(TSU_ERR_ARG, "bad boundary type");
    if ((s->bc[0] == TSU_BC_PERIODIC) != (s->bc[1] == TSU_BC_PERIODIC) ||
        (s->bc[2] == TSU_BC_PERIODIC) != (s->bc[3] == TSU_BC_PERIODIC))
        return fail(TSU_ERR_UNSUPPORTED, "periodic boundaries must be paired on an axis");
    if (s->limiter < 0 || s->limiter > 1 || s->bedload_law < 0 || s->bedload_law > 1 || s->friction_law < 0 ||
        s->friction_law > 1)
        return fail(TSU_ERR_ARG, "bad law selector");
    if ((s->bedload != 0 && s->bedload != 1) || (s->suspension != 0 && s->suspension != 1))
        return fail(TSU_ERR_ARG, "bedload and suspension are 0/1 switches");
    return TSU_OK;
}

}  // namespace

namespace tsu {

// Run constants from the reference parameters, evaluated in the reference's
// operation order (Reconstructor.cu:64-77, SedFlux.cuh:56-83).
void make_dev_params(const tsu_sim_params* p, const tsu_scheme* s, DevParams* P)
{
    std::memset(P, 0, sizeof(*P));
    const double G = 9.81;
    P->npx = p->npx;
    P->npy = p->npy;
    P->nvol = (long long)p->npx * p->npy;
    P->dx = p->dx;
    P->dy = p->dy;
    P->inv_dx = 1.0 / p->dx;
    P->inv_dy = 1.0 / p->dy;
    P->cfl_half = p->CFL * 0.5;
    P->FR = p->FR;
    P->epsilon_h = p->epsilon_h;
    P->Q = p->Q;
    P->Opar = p->Opar;
    P->OC = p->OC;
    P->sqrtOC = std::sqrt(p->OC);
    P->HQB = p->HQB;
    P->fiveDS = 5 * p->DS;
    const double nu = 1.002e-6;
    const double sd = p->R - 1.0;
    P->vs = std::sqrt((13.95 * nu / p->DS) * (13.95 * nu / p->DS) + 1.09 * sd * G * p->DS) - 13.95 * nu / p->DS;
    const double Rp = (p->DS * std::sqrt(sd * G * p->DS)) / nu;
    P->ka = (Rp > 2.36) ? 1.0 * std::pow(Rp, 0.6) : 0.586 * std::pow(Rp, 1.23);
    P->sqrtFR = std::sqrt(p->FR);
    P->cbk = 1.64 + 0.4 * std::pow(p->DS / p->Dsg, 1.64);
    P->vs1p = P->vs * (1 - p->porosity);
    P->inv_vs = 1.0 / P->vs;
    P->grass_k = s->grass_ag / (1.0 - p->porosity);
    P->manning_n = s->manning_n;
    P->bedload = s->bedload;
    P->suspension = s->suspension;
    P->limiter = s->limiter;
    P->bedload_law = s->bedload_law;
    P->friction_law = s->friction_law;
    P->order = s->order;
    P->dt_narrow = s->dt_narrow;
    P->extrema = s->extrema;
    // bedload square roots: |u|^2 > OC (1 - 2^-40) / Opar and O > OC there
    const double tiny = std::ldexp(1.0, -700);
    P->bed_sqrt_unscaled = (P->OC > tiny && P->Opar > 0.0 && std::isfinite(P->Opar) &&
                            P->OC * (1.0 - std::ldexp(1.0, -40)) / P->Opar > tiny) ? 1 : 0;
    for (int i = 0; i < 4; i++) P->bc[i] = s->bc[i];
    P->ring = 2LL * p->npx + 2LL * p->npy;
}

int validate_scheme(const tsu_scheme* s) { return check_scheme(s); }

int set_error(int code, const std::string& msg) { return fail(code, msg); }

namespace {
// A buffer for transfers of count values.  False where the host converts: few
// values, whose launch and wait would cost more than they save (a download of
// 100^2 cells 33 us on the host and 41 on the device, of 256^2 217 and 166),
// and a device without room.
bool reserve(Staging* g, long long nv, long long count)
{
    if (nv <= 16384) return false;
    const long long want = std::min(count, 4LL << 20);
    if (g->cap >= want) return true;
    free_staging(g);
    if (hipMalloc((void**)&g->buf, (size_t)want * sizeof(double)) != hipSuccess) {
        (void)hipGetLastError();
        g->buf = nullptr;
        return false;
    }
    g->cap = want;
    return true;
}

// plane of the low parts of plane f, or -1
constexpr int kLoPlane[5] = {5, -1, -1, 6, 7};
}  // namespace

void free_staging(Staging* g)
{
    (void)hipFree(g->buf);
    *g = Staging{};
}

int upload_planes(Staging* g, const double* host, void* state, int precision, long long nv, hipStream_t s)
{
    const long long count = 5 * nv;
    if (precision == TSU_FP64) {
        HIPCHK(hipMemcpyAsync(state, host, (size_t)count * sizeof(double), hipMemcpyHostToDevice, s));
    } else if (reserve(g, nv, count)) {
        for (long long o = 0; o < count; o += g->cap) {
            const long long n = std::min(g->cap, count - o);
            HIPCHK(hipMemcpyAsync(g->buf, host + o, (size_t)n * sizeof(double), hipMemcpyHostToDevice, s));
            HIPCHK(launch_narrow(g->buf, (float*)state, nv, o, n, s));
        }
    } else {
        std::vector<float> v((size_t)(8 * nv));
        for (int f = 0; f < 5; f++) {
            const double* from = host + f * nv;
            float* hi = v.data() + f * nv;
            for (long long i = 0; i < nv; i++) hi[i] = (float)from[i];
            if (kLoPlane[f] < 0) continue;
            float* lo = v.data() + kLoPlane[f] * nv;
            for (long long i = 0; i < nv; i++) lo[i] = (float)(from[i] - (double)hi[i]);
        }
        HIPCHK(hipMemcpyAsync(state, v.data(), v.size() * sizeof(float), hipMemcpyHostToDevice, s));
        HIPCHK(hipStreamSynchronize(s));                    // v ends here
    }
    return TSU_OK;
}

int download_planes(Staging* g, const void* state, double* host, int precision, long long nv, int first, int planes,
                    hipStream_t s)
{
    const long long count = planes * nv, at = first * nv;
    if (precision == TSU_FP64) {
        HIPCHK(hipMemcpyAsync(host, (const double*)state + at, (size_t)count * sizeof(double), hipMemcpyDeviceToHost,
                              s));
    } else if (reserve(g, nv, count)) {
        for (long long o = 0; o < count; o += g->cap) {
            const long long n = std::min(g->cap, count - o);
            HIPCHK(launch_widen((const float*)state, g->buf, nv, at + o, n, s));
            HIPCHK(hipMemcpyAsync(host + o, g->buf, (size_t)n * sizeof(double), hipMemcpyDeviceToHost, s));
        }
    } else {
        // from the first plane to the last low part, in one copy
        const int last = planes == 5 ? 7 : std::max(first, kLoPlane[first]);
        std::vector<float> v((size_t)((last - first + 1) * nv));
        HIPCHK(hipMemcpyAsync(v.data(), (const float*)state + at, v.size() * sizeof(float), hipMemcpyDeviceToHost, s));
        HIPCHK(hipStreamSynchronize(s));
        for (int f = 0; f < planes; f++) {
            const float* hi = v.data() + f * nv;
            const float* lo = kLoPlane[first + f] < 0 ? nullptr : v.data() + (kLoPlane[first + f] - first) * nv;
            double* to = host + f * nv;
            for (long long i = 0; i < nv; i++) to[i] = lo ? (double)hi[i] + (double)lo[i] : (double)hi[i];
        }
        return TSU_OK;
    }
    HIPCHK(hipStreamSynchronize(s));
    return TSU_OK;
}

// The tile height with the least estimated cost of a stage.
//
// Alone on the GPU: a tile of r rows costs its wave r + 0.6 rows (the
// prologue's faces and edge, partly under the launch's start); k waves that
// share a SIMD take from 1.4 (FP64) or 1.7 (FP32) rows' time per row for one
// to w for w, the kernel's waves per SIMD (a wave alone leaves issue slots
// idle: 256^2 in FP32 takes 23.8 us a step with up to two one-row waves per
// SIMD, 29.5 with one of two rows).
// Tiles that fit the chip at once last as long as the SIMD with most waves;
// more run in rounds, the last one partly filled, and with more rounds the
// tiles' uneven costs (still, dry) blur them into a steady rate.  The 0.4 is
// the wait for the slowest wave.
//
// Beside other runs on the GPU (two to three simulations on streams of their
// own) idle slots are filled by the others and what counts is the work,
// r + 0.87 rows per tile, until a run's own latency shows: the hypotenuse of
// the work and half of the time alone.
//
// The product of both is least for the height chosen: a grid steps alone or
// beside other runs, half an ensemble beside the other half.  The constants are
// fits to sweeps of the height over 40 grids of 256^2 .. 2048^2 cells in both
// precisions, with and without sediment, alone and beside two others: over these
// the chosen heights are 0.4 % from the best alone and 4 % beside others, on
// average.  Over ensembles of 0.08 to 8 million cells in two halves, both
// schemes and precisions, with and without sediment, at rest and in motion, they
// are 2 % from the best on average and 11 % at most (by the time alone 6 % and
// 28 %: 8 members of 2.2 million cells in FP32, two-stage, 147 us a step for 122
// with 6 rows).  Against powers of two from 32 down to 2 (at least 8192 tiles,
// then at least 2048), us a step alone: 700^2 FP64 143 -> 117 (5 rows for 4),
// 4096^2 2399 -> 2336 (24 for 32).
int choose_tile_rows(const std::vector<std::pair<int, int>>& grids, bool sed, int precision, int device)
{
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess || cus < 1) cus = 256;
    const int waves = stage_waves_per_simd(sed, precision);
    const double simds = 4.0 * cus, slots = simds * waves, lone = precision == TSU_FP64 ? 1.4 : 1.7;
    auto together = [&](double k) { return waves > 1 ? lone + (waves - lone) * (k - 1.0) / (waves - 1.0) : k; };
    int best = 1;
    double best_cost = INFINITY;
    for (int r = 1; r <= 32; r++) {
        double n = 0.0;
        for (const auto& g : grids)
            n += (double)((g.first + kStripOut - 1) / kStripOut) * (double)((g.second + (long long)r - 1) / r);
        double rounds;
        if (n <= slots) {
            rounds = together(std::ceil(n / simds));
        } else {
            const double full = std::floor(n / slots), rest = n - full * slots;
            const double hard = full * waves + (rest > 0 ? together(std::ceil(rest / simds)) : 0.0);
            const double steady = n / simds + 0.1 * waves, blur = std::min(1.0, 0.5 * (full - 1.0));
            rounds = hard + (steady - hard) * blur;
        }
        const double alone = (r + 0.6) * (rounds + 0.4);
        const double cost = alone * std::hypot(n / simds * (r + 0.87), 0.5 * alone);
        if (cost < best_cost) {
            best = r;
            best_cost = cost;
        }
    }
    return best;
}

}  // namespace tsu

struct tsu_state {
    std::recursive_mutex calls;
    int device = 0;
    int precision = TSU_FP64;
    bool sed = true;
    bool uploaded = false;
    tsu_sim_params p{};
    tsu_scheme s{};
    DevParams P{};
    size_t esize = 8;
    long long nvol = 0;
    void* A = nullptr;
    void* B = nullptr;
    uint8_t* fix = nullptr;
    Ctrl* ctrl = nullptr;
    tsu::DtSlots* dts = nullptr;
    tsu::StepReport* report = nullptr;
    tsu::Staging staging;
    double* ext = nullptr;
    double* CC = nullptr;
    double* tCC = nullptr;
    unsigned long timeCC = 0;
    double* mass_buf = nullptr;
    int mass_nb = 0;
    DevParams* dP = nullptr;   // device copy of P read by the stage kernels
    hipStream_t stream = nullptr;
    int tile_rows = 0, nstrips = 0, nchunks = 0, ntiles = 0;
    bool split = false;        // stage_split_kernel (tile_rows 1)
    bool rows_given = false;   // tile_rows by the caller, not by default
    int graph_chunk = 0;
    hipGraphExec_t gexec = nullptr;
    hipGraph_t graph = nullptr;
    bool capturing = false;
    // stage-kernel event timing
    bool timing = false;
    std::vector<hipEvent_t> ev;        // start/end pairs, reused
    std::vector<int> ev_stage;         // stage index of each pair
    size_t ev_used = 0;                // pairs recorded since the last read
    double stage_ms[2] = {0.0, 0.0};
    long long launches[2] = {0, 0};
};

namespace {

struct DeviceGuard {
    int prev = -1;
    explicit DeviceGuard(int dev)
    {
        if (hipGetDevice(&prev) != hipSuccess) prev = -1;
        (void)hipSetDevice(dev);
    }
    ~DeviceGuard()
    {
        if (prev >= 0) (void)hipSetDevice(prev);
    }
};

// FP64: h, qx, qy, H, hc.  FP32: the same five planes plus the low-order
// parts of h, H and hc (compensated accumulation).
size_t planes_of(const tsu_state* st) { return st->precision == TSU_FP64 ? 5 : 8; }

// Whether all rows of a grid, each with three waves (stage_split_kernel), run
// at once with at most two waves per SIMD in FP64 and three in FP32.  Above
// that its extra work (a row's edge along y is solved by both its rows, with a
// reconstruction more) costs more than the shorter chain gives, first beside
// other runs.  us a step, alone and with two others of its size beside it (a
// third of their time), against one wave per tile: FP64 with sediment 100^2
// 26.9 -> 16.3 and 12.1 -> 7.4, 160^2 28.5 -> 20.9 and 12.7 -> 10.5, past the
// line 200^2 28.8 -> 26.8 and 14.0 -> 14.6, 320^2 40 -> 48 and 26.8 -> 30.9;
// FP32 100^2 21.1 -> 14.1 and 9.0 -> 6.6, 240 x 256 23.3 -> 18.0 and 10.2 ->
// 10.4, past it 320^2 24.1 -> 27.2 and 12.4 -> 15.8.  Without sediment, and
// single-stage, the kernels hold more waves but there is as little left to gain at
// the line: FP64 100^2 18.9 -> 12.8 and 10.8 -> 8.0, 180 x 200 19.8 -> 18.9 and
// 11.4 -> 10.6, single-stage 13.6 -> 13.4 and 8.2 -> 8.1.
bool split_rows(const tsu_state* st)
{
    int cus = 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, st->device) != hipSuccess || cus < 1)
        cus = 256;
    const long long strips = (st->p.npx + tsu::kStripOut - 1) / tsu::kStripOut;
    return tsu::kSplitWaves * strips * st->p.npy <= 4LL * cus * (st->precision == TSU_FP64 ? 2 : 3);
}

// rows 0: the default for the grid, precision and scheme.
void set_tiling(tsu_state* st, int rows)
{
    st->split = rows == 0 && split_rows(st);
    if (st->split)
        rows = 1;
    else if (rows == 0)
        rows = tsu::choose_tile_rows({{st->p.npx, st->p.npy}}, st->sed, st->precision, st->device);
    st->tile_rows = rows;
    st->nstrips = (st->p.npx + tsu::kStripOut - 1) / tsu::kStripOut;
    st->nchunks = (st->p.npy + rows - 1) / rows;
    st->ntiles = st->nstrips * st->nchunks;
}

void drop_graph(tsu_state* st)
{
    if (st->gexec) (void)hipGraphExecDestroy(st->gexec);
    if (st->graph) (void)hipGraphDestroy(st->graph);
    st->gexec = nullptr;
    st->graph = nullptr;
}

void free_state(tsu_state* st)
{
    if (!st) return;
    DeviceGuard g(st->device);
    drop_graph(st);
    if (st->stream) (void)hipStreamSynchronize(st->stream);
    for (hipEvent_t e : st->ev) (void)hipEventDestroy(e);
    (void)hipFree(st->A);
    (void)hipFree(st->B);
    (void)hipFree(st->fix);
    (void)hipFree(st->ctrl);
    (void)hipFree(st->dts);
    (void)hipFree(st->report);
    tsu::free_staging(&st->staging);
    (void)hipFree(st->ext);
    (void)hipFree(st->CC);
    (void)hipFree(st->tCC);
    (void)hipFree(st->mass_buf);
    (void)hipFree(st->dP);
    if (st->stream) (void)hipStreamDestroy(st->stream);
    delete st;
}

tsu::StageArgs stage_args(const tsu_state* st, int k)
{
    tsu::StageArgs a{};
    const size_t plane = (size_t)st->nvol * st->esize;
    a.Hin = (const char*)st->A + 3 * plane;
    a.fix = st->fix;
    a.ctrl = st->ctrl;
    a.dts = st->dts;
    a.ext = st->s.extrema ? st->ext : nullptr;
    a.tile_rows = st->tile_rows;
    a.nstrips = st->nstrips;
    a.ntiles = st->ntiles;
    a.split = st->split;
    a.npx = st->P.npx;
    a.npy = st->P.npy;
    a.periodic = tsu::periodic_sides(st->P);
    a.P = st->dP;
    a.k = k;
    if (st->s.order == 1) {
        a.in = st->A;
        a.out = st->B;
        a.v0 = st->A;
        a.pingpong = 1;
        a.last = 1;
    } else if (k == 0) {
        a.in = st->A;
        a.out = st->B;
        a.v0 = st->A;
        a.last = 0;
    } else {
        a.in = st->B;
        a.out = st->A;
        a.v0 = st->A;
        a.last = 1;
    }
    return a;
}

int enqueue_step(tsu_state* st)
{
    const bool timed = st->timing && !st->capturing;
    for (int k = 0; k < st->s.order; k++) {
        tsu::StageArgs a = stage_args(st, k);
        if (timed) {
            if (st->ev_used * 2 + 2 > st->ev.size()) {
                for (int i = 0; i < 2; i++) {
                    hipEvent_t e;
                    HIPCHK(hipEventCreate(&e));
                    st->ev.push_back(e);
                }
                st->ev_stage.push_back(0);
            }
            st->ev_stage[st->ev_used] = k;
            HIPCHK(hipEventRecord(st->ev[2 * st->ev_used], st->stream));
        }
        HIPCHK(tsu::launch_stage(a, st->sed, st->precision, st->stream, tsu::fast_bedload(st->P)));
        if (timed) {
            HIPCHK(hipEventRecord(st->ev[2 * st->ev_used + 1], st->stream));
            st->ev_used++;
        }
    }
    if (st->s.order == 1) HIPCHK(tsu::launch_advance(st->ctrl, st->dts, st->P, st->stream));
    return TSU_OK;
}

int read_ctrl(tsu_state* st, Ctrl* c)
{
    HIPCHK(hipMemcpyAsync(c, st->ctrl, sizeof(Ctrl), hipMemcpyDeviceToHost, st->stream));
    HIPCHK(hipStreamSynchronize(st->stream));
    return TSU_OK;
}

// Buffer holding U^n (the single-stage scheme alternates by step parity).
int current_buffer(tsu_state* st, void** buf)
{
    if (st->s.order == 2) {
        *buf = st->A;
        return TSU_OK;
    }
    Ctrl c;
    int rc = read_ctrl(st, &c);
    if (rc) return rc;
    *buf = (c.step & 1) ? st->B : st->A;
    return TSU_OK;
}

}  // namespace

extern "C" {

TSU_API const char* tsu_last_error(void) { return g_err.c_str(); }

TSU_API const char* tsu_version(void) { return "tsuner-amd 0.1 (gfx950)"; }

TSU_API int checkCUDAsupport(int device)
{
    int n = 0;
    if (hipGetDeviceCount(&n) != hipSuccess || n == 0) return 1;
    if (device < 0 || device >= n) return 3;
    hipDeviceProp_t prop;
    if (hipGetDeviceProperties(&prop, device) != hipSuccess) return 2;
    return std::strncmp(prop.gcnArchName, "gfx950", 6) == 0 ? 0 : 2;
}

TSU_API int tsu_device_check(int device) { return checkCUDAsupport(device); }

TSU_API void initializeGPU(void)
{
    (void)tsu::launch_warmup(nullptr);
    (void)hipDeviceSynchronize();
}

TSU_API int tsu_state_create(tsu_state** out, const tsu_sim_params* p, const tsu_scheme* s, int precision,
                             int device)
{
    if (!out || !p || !s) return fail(TSU_ERR_ARG, "null argument");
    *out = nullptr;
    if (p->npx < 1 || p->npy < 1) return fail(TSU_ERR_ARG, "npx and npy must be positive");
    if (!(p->dx > 0) || !(p->dy > 0)) return fail(TSU_ERR_ARG, "dx and dy must be positive");
    if (precision != TSU_FP64 && precision != TSU_FP32) return fail(TSU_ERR_ARG, "precision must be FP64 or FP32");
    int rc = check_scheme(s);
    if (rc) return rc;
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return fail(TSU_ERR_HIP, "no HIP device");
    if (device < 0 || device >= ndev) return fail(TSU_ERR_ARG, "bad device index");

    tsu_state* st = new tsu_state();
    st->device = device;
    st->precision = precision;
    st->p = *p;
    st->p.nvol = p->npx * p->npy;
    st->s = *s;
    st->esize = precision == TSU_FP64 ? 8 : 4;
    st->nvol = (long long)p->npx * p->npy;
    tsu::make_dev_params(&st->p, &st->s, &st->P);
    st->sed = s->bedload || s->suspension;
    set_tiling(st, 0);

    DeviceGuard g(device);
    const size_t state_bytes = planes_of(st) * (size_t)st->nvol * st->esize;
    st->mass_nb = tsu::mass_blocks(st->nvol);
    hipError_t e = hipStreamCreateWithFlags(&st->stream, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipMalloc(&st->A, state_bytes);
    if (e == hipSuccess) e = hipMalloc(&st->B, state_bytes);
    if (e == hipSuccess) e = hipMalloc((void**)&st->fix, (size_t)st->nvol);
    if (e == hipSuccess) e = hipMalloc((void**)&st->ctrl, sizeof(Ctrl));
    if (e == hipSuccess) e = hipMalloc((void**)&st->dts, sizeof(tsu::DtSlots));
    if (e == hipSuccess) e = hipMalloc((void**)&st->report, sizeof(tsu::StepReport));
    if (e == hipSuccess) e = hipMalloc((void**)&st->mass_buf, (2 * (size_t)st->mass_nb + 2) * sizeof(double));
    if (e == hipSuccess) e = hipMalloc((void**)&st->dP, sizeof(DevParams));
    if (e == hipSuccess) e = hipMemcpy(st->dP, &st->P, sizeof(DevParams), hipMemcpyHostToDevice);
    if (e == hipSuccess && s->extrema) e = hipMalloc((void**)&st->ext, 3 * (size_t)st->nvol * sizeof(double));
    if (e == hipSuccess) e = tsu::launch_reset_steps(st->ctrl, st->dts, 1, st->stream);
    if (e != hipSuccess) {
        free_state(st);
        (void)hipGetLastError();
        return fail(TSU_ERR_DEVICE_MEMORY, std::string("device allocation failed: ") + hipGetErrorString(e));
    }
    *out = st;
    return TSU_OK;
}

TSU_API int tsu_state_destroy(tsu_state* st)
{
    free_state(st);
    return TSU_OK;
}

TSU_API int tsu_state_upload(tsu_state* st, const double* V, const int* fixH)
{
    if (!st || !V || !fixH) return fail(TSU_ERR_ARG, "null argument");
    const long long nv = st->nvol;
    std::vector<uint8_t> fx((size_t)nv);
    for (long long i = 0; i < nv; i++) {
        if (fixH[i] != 0 && fixH[i] != 1) return fail(TSU_ERR_ARG, "fixH values must be 0 or 1");
        fx[(size_t)i] = (uint8_t)fixH[i];
    }
    bool hc_zero = true;
    for (long long i = 0; i < nv && hc_zero; i++) hc_zero = V[4 * nv + i] == 0.0;
    tsu::HandleGuard g(st->calls, st->device);
    st->sed = st->s.bedload || st->s.suspension || !hc_zero;
    drop_graph(st);
    if (!st->rows_given) set_tiling(st, 0);
    const size_t bytes = planes_of(st) * (size_t)nv * st->esize;
    if (int rc = tsu::upload_planes(&st->staging, V, st->A, st->precision, nv, st->stream)) return rc;
    HIPCHK(hipMemcpyAsync(st->B, st->A, bytes, hipMemcpyDeviceToDevice, st->stream));
    HIPCHK(hipMemcpyAsync(st->fix, fx.data(), (size_t)nv, hipMemcpyHostToDevice, st->stream));
    if (st->ext) HIPCHK(tsu::launch_fill(st->ext, 3 * nv, -1e30, st->stream));
    HIPCHK(tsu::launch_reset_steps(st->ctrl, st->dts, 1, st->stream));
    HIPCHK(hipStreamSynchronize(st->stream));
    st->uploaded = true;
    return TSU_OK;
}

TSU_API int tsu_state_download(tsu_state* st, double* V)
{
    if (!st || !V) return fail(TSU_ERR_ARG, "null argument");
    tsu::HandleGuard g(st->calls, st->device);
    void* cur;
    int rc = current_buffer(st, &cur);
    if (rc) return rc;
    return tsu::download_planes(&st->staging, cur, V, st->precision, st->nvol, 0, 5, st->stream);
}

TSU_API int tsu_state_set_inflow(tsu_state* st, const double* CC, const double* tCC, unsigned long timeCC)
{
    if (!st || !CC || !tCC) return fail(TSU_ERR_ARG, "null argument");
    if (timeCC < 2) return fail(TSU_ERR_ARG, "the inflow series needs at least two time levels");
    // interpolate_time divides by tCC[1] - tCC[0] and truncates the quotient
    // to an int level index (VolumeSolver.cu:174-176): the times must be
    // finite and increasing
    for (unsigned long k = 0; k < timeCC; k++)
        if (!std::isfinite(tCC[k]) || (k > 0 && !(tCC[k] > tCC[k - 1])))
            return fail(TSU_ERR_ARG, "inflow times must be finite and strictly increasing");
    tsu::HandleGuard g(st->calls, st->device);
    // steps already enqueued may still read the old series and run constants
    HIPCHK(hipStreamSynchronize(st->stream));
    drop_graph(st);
    (void)hipFree(st->CC);
    (void)hipFree(st->tCC);
    st->CC = st->tCC = nullptr;
    const size_t ncc = (size_t)st->P.ring * 4 * timeCC;
    hipError_t e = hipMalloc((void**)&st->CC, ncc * sizeof(double));
    if (e == hipSuccess) e = hipMalloc((void**)&st->tCC, timeCC * sizeof(double));
    if (e != hipSuccess) return fail(TSU_ERR_DEVICE_MEMORY, "inflow series allocation failed");
    HIPCHK(hipMemcpy(st->CC, CC, ncc * sizeof(double), hipMemcpyHostToDevice));
    HIPCHK(hipMemcpy(st->tCC, tCC, timeCC * sizeof(double), hipMemcpyHostToDevice));
    st->timeCC = timeCC;
    st->P.CC = st->CC;
    st->P.tCC = st->tCC;
    st->P.timeCC = (long long)timeCC;
    st->P.tcc0 = tCC[0];
    st->P.dtcc = tCC[1] - tCC[0];
    st->P.tcc_end = tCC[timeCC - 2];
    HIPCHK(hipMemcpy(st->dP, &st->P, sizeof(DevParams), hipMemcpyHostToDevice));
    return TSU_OK;
}

static int check_ready(tsu_state* st)
{
    if (!st) return fail(TSU_ERR_ARG, "null state");
    if (!st->uploaded) return fail(TSU_ERR_ARG, "state not uploaded");
    for (int i = 0; i < 4; i++)
        if (st->s.bc[i] == TSU_BC_INFLOW && !st->CC)
            return fail(TSU_ERR_ARG, "an inflow side needs tsu_state_set_inflow first");
    return TSU_OK;
}

TSU_API int tsu_init_dt(tsu_state* st)
{
    int rc = check_ready(st);
    if (rc) return rc;
    tsu::HandleGuard g(st->calls, st->device);
    Ctrl c;
    rc = read_ctrl(st, &c);
    if (rc) return rc;
    HIPCHK(tsu::launch_arm_dt(st->dts, st->stream));
    void* cur = (st->s.order == 1 && (c.step & 1)) ? st->B : st->A;
    HIPCHK(tsu::launch_init_dt(cur, st->P, st->dts, c.step, st->precision, st->stream));
    HIPCHK(hipStreamSynchronize(st->stream));
    return TSU_OK;
}

TSU_API int tsu_step(tsu_state* st, int nsteps)
{
    int rc = check_ready(st);
    if (rc) return rc;
    if (nsteps < 0) return fail(TSU_ERR_ARG, "negative step count");
    tsu::HandleGuard g(st->calls, st->device);
    int done = 0;
    if (st->graph_chunk > 0 && nsteps >= st->graph_chunk) {
        if (!st->gexec) {
            HIPCHK(hipStreamBeginCapture(st->stream, hipStreamCaptureModeThreadLocal));
            st->capturing = true;
            for (int i = 0; i < st->graph_chunk; i++) {
                rc = enqueue_step(st);
                if (rc) {
                    hipGraph_t gph = nullptr;
                    st->capturing = false;
                    (void)hipStreamEndCapture(st->stream, &gph);
                    if (gph) (void)hipGraphDestroy(gph);
                    return rc;
                }
            }
            st->capturing = false;
            HIPCHK(hipStreamEndCapture(st->stream, &st->graph));
            HIPCHK(hipGraphInstantiate(&st->gexec, st->graph, nullptr, nullptr, 0));
        }
        while (nsteps - done >= st->graph_chunk) {
            HIPCHK(hipGraphLaunch(st->gexec, st->stream));
            done += st->graph_chunk;
        }
    }
    for (; done < nsteps; done++) {
        rc = enqueue_step(st);
        if (rc) return rc;
    }
    return TSU_OK;
}

TSU_API int tsu_synchronize(tsu_state* st)
{
    if (!st) return fail(TSU_ERR_ARG, "null state");
    DeviceGuard g(st->device);   // no call is kept waiting
    HIPCHK(hipStreamSynchronize(st->stream));
    return TSU_OK;
}

TSU_API int tsu_get_time(tsu_state* st, double* t, double* dt, long long* steps)
{
    if (!st) return fail(TSU_ERR_ARG, "null state");
    tsu::HandleGuard g(st->calls, st->device);
    tsu::StepReport r;
    HIPCHK(tsu::launch_report(st->ctrl, st->dts, st->report, st->stream));
    HIPCHK(hipMemcpyAsync(&r, st->report, sizeof(r), hipMemcpyDeviceToHost, st->stream));
    HIPCHK(hipStreamSynchronize(st->stream));
    if (t) *t = r.t;
    if (dt) *dt = finalize_host(st->P, r.dt_bits);
    if (steps) *steps = r.step;
    return TSU_OK;
}

TSU_API int tsu_set_time(tsu_state* st, double t, double dt)
{
    if (!st) return fail(TSU_ERR_ARG, "null state");
    tsu::HandleGuard g(st->calls, st->device);
    HIPCHK(tsu::launch_set_time(st->ctrl, st->dts, t, dt, st->stream));
    HIPCHK(hipStreamSynchronize(st->stream));
    return TSU_OK;
}

TSU_API int tsu_set_stop_time(tsu_state* st, double stop_time)
{
    if (!st) return fail(TSU_ERR_ARG, "null state");
    tsu::HandleGuard g(st->calls, st->device);
    static_assert(offsetof(Ctrl, stop_time) == 8, "ctrl layout");
    HIPCHK(hipMemcpyAsync((char*)st->ctrl + offsetof(Ctrl, stop_time), &stop_time, sizeof(double),
                          hipMemcpyHostToDevice, st->stream));
    HIPCHK(hipStreamSynchronize(st->stream));
    return TSU_OK;
}

TSU_API int tsu_set_clamp(tsu_state* st, int on)
{
    if (!st) return fail(TSU_ERR_ARG, "null state");
    tsu::HandleGuard g(st->calls, st->device);
    const long long v = on ? 1 : 0;
    HIPCHK(hipMemcpyAsync((char*)st->ctrl + offsetof(Ctrl, clamp), &v, sizeof(long long), hipMemcpyHostToDevice,
                          st->stream));
    HIPCHK(hipStreamSynchronize(st->stream));
    return TSU_OK;
}

TSU_API int tsu_mass(tsu_state* st, double out[2])
{
    if (!st || !out) return fail(TSU_ERR_ARG, "null argument");
    tsu::HandleGuard g(st->calls, st->device);
    void* cur;
    int rc = current_buffer(st, &cur);
    if (rc) return rc;
    double* res = st->mass_buf + 2 * st->mass_nb;
    HIPCHK(tsu::launch_mass(cur, st->nvol, st->precision, st->mass_buf, st->mass_nb, res, st->stream));
    HIPCHK(hipMemcpyAsync(out, res, 2 * sizeof(double), hipMemcpyDeviceToHost, st->stream));
    HIPCHK(hipStreamSynchronize(st->stream));
    return TSU_OK;
}

TSU_API int tsu_get_extrema(tsu_state* st, double* hmax, double* bmax, double* eta_max)
{
    if (!st) return fail(TSU_ERR_ARG, "null state");
    if (!st->ext) return fail(TSU_ERR_ARG, "extrema are not enabled in the scheme");
    tsu::HandleGuard g(st->calls, st->device);
    const size_t b = (size_t)st->nvol * sizeof(double);
    if (hmax) HIPCHK(hipMemcpyAsync(hmax, st->ext, b, hipMemcpyDeviceToHost, st->stream));
    if (bmax) HIPCHK(hipMemcpyAsync(bmax, st->ext + st->nvol, b, hipMemcpyDeviceToHost, st->stream));
    if (eta_max) HIPCHK(hipMemcpyAsync(eta_max, st->ext + 2 * st->nvol, b, hipMemcpyDeviceToHost, st->stream));
    HIPCHK(hipStreamSynchronize(st->stream));
    return TSU_OK;
}

TSU_API int tsu_set_tile_rows(tsu_state* st, int rows)
{
    if (!st) return fail(TSU_ERR_ARG, "null state");
    if (rows < 0 || rows > 4096) return fail(TSU_ERR_ARG, "tile rows out of range");
    tsu::HandleGuard g(st->calls, st->device);
    drop_graph(st);
    st->rows_given = rows != 0;
    set_tiling(st, rows);
    return TSU_OK;
}

TSU_API int tsu_get_tile_rows(tsu_state* st) { return st ? st->tile_rows : -1; }

TSU_API int tsu_set_graph_chunk(tsu_state* st, int chunk)
{
    if (!st) return fail(TSU_ERR_ARG, "null state");
    if (chunk < 0) return fail(TSU_ERR_ARG, "negative graph chunk");
    if (st->s.order == 1 && (chunk & 1)) return fail(TSU_ERR_ARG, "single-stage graphs need an even chunk");
    tsu::HandleGuard g(st->calls, st->device);
    drop_graph(st);
    st->graph_chunk = chunk;
    return TSU_OK;
}

TSU_API int tsu_set_timing(tsu_state* st, int on)
{
    if (!st) return fail(TSU_ERR_ARG, "null state");
    tsu::HandleGuard g(st->calls, st->device);
    st->timing = on != 0;
    return TSU_OK;
}

TSU_API int tsu_get_timing(tsu_state* st, double stage_ms[2], long long launches[2], int reset)
{
    if (!st) return fail(TSU_ERR_ARG, "null state");
    tsu::HandleGuard g(st->calls, st->device);
    HIPCHK(hipStreamSynchronize(st->stream));
    for (size_t i = 0; i < st->ev_used; i++) {
        float ms = 0.0f;
        HIPCHK(hipEventElapsedTime(&ms, st->ev[2 * i], st->ev[2 * i + 1]));
        st->stage_ms[st->ev_stage[i]] += ms;
        st->launches[st->ev_stage[i]]++;
    }
    st->ev_used = 0;
    for (int k = 0; k < 2; k++) {
        if (stage_ms) stage_ms[k] = st->stage_ms[k];
        if (launches) launches[k] = st->launches[k];
        if (reset) {
            st->stage_ms[k] = 0.0;
            st->launches[k] = 0;
        }
    }
    return TSU_OK;
}

TSU_API void* tsu_stream(tsu_state* st) { return st ? (void*)st->stream : nullptr; }

TSU_API void* tsu_device_state(tsu_state* st) { return st ? st->A : nullptr; }

TSU_API int tsu_bandwidth_probe(int device, long long bytes, int reps, double* gbs)
{
    if (bytes < 16 || reps < 1 || !gbs) return fail(TSU_ERR_ARG, "bad argument");
    bytes &= ~15LL;
    DeviceGuard g(device);
    void *a = nullptr, *b = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    hipError_t e = hipMalloc(&a, (size_t)bytes);
    if (e == hipSuccess) e = hipMalloc(&b, (size_t)bytes);
    if (e == hipSuccess) e = hipMemset(a, 0, (size_t)bytes);
    if (e == hipSuccess) e = hipEventCreate(&e0);
    if (e == hipSuccess) e = hipEventCreate(&e1);
    if (e == hipSuccess) e = tsu::launch_copy(a, b, bytes, nullptr);   // warm-up
    if (e == hipSuccess) e = hipEventRecord(e0, nullptr);
    for (int i = 0; i < reps && e == hipSuccess; i++) e = tsu::launch_copy(a, b, bytes, nullptr);
    if (e == hipSuccess) e = hipEventRecord(e1, nullptr);
    if (e == hipSuccess) e = hipEventSynchronize(e1);
    float ms = 0.0f;
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, e0, e1);
    if (e0) (void)hipEventDestroy(e0);
    if (e1) (void)hipEventDestroy(e1);
    (void)hipFree(a);
    (void)hipFree(b);
    if (e != hipSuccess) return fail(TSU_ERR_HIP, std::string("bandwidth probe: ") + hipGetErrorString(e));
    *gbs = 2.0 * (double)bytes * reps / (ms * 1e-3) / 1e9;
    return TSU_OK;
}

namespace {

// Shared host side of the edge known-answer entries: pairs = false solves
// every edge alone (edge_flux), true solves edges 2k and 2k + 1 together
// (edge_flux_pair, n even).
int kat_edges(const tsu_sim_params* p, const tsu_scheme* s, int n, const double* left, const double* right,
              const int* normal, const int* fixed, double* Dm, double* Dp, int device, bool pairs)
{
    if (!p || !s || n < 0 || (n > 0 && (!left || !right || !normal || !fixed || !Dm || !Dp)))
        return fail(TSU_ERR_ARG, "bad argument");
    if (pairs && n % 2 != 0) return fail(TSU_ERR_ARG, "edge pairs need an even number of edges");
    if (n == 0) return TSU_OK;
    DevParams P;
    tsu::make_dev_params(p, s, &P);
    std::vector<int> kind((size_t)n);
    for (int i = 0; i < n; i++) {
        int nx = normal[2 * i], ny = normal[2 * i + 1];
        if (nx == 1 && ny == 0) kind[i] = tsu::N_PX;
        else if (nx == -1 && ny == 0) kind[i] = tsu::N_MX;
        else if (nx == 0 && ny == 1) kind[i] = tsu::N_PY;
        else if (nx == 0 && ny == -1) kind[i] = tsu::N_MY;
        else return fail(TSU_ERR_ARG, "normals must be axis-aligned unit vectors");
    }
    DeviceGuard g(device);
    double *dl = nullptr, *dr = nullptr, *dm = nullptr, *dp = nullptr;
    int *dk = nullptr, *df = nullptr;
    const size_t b5 = 5 * (size_t)n * sizeof(double), bi = (size_t)n * sizeof(int);
    hipError_t e = hipMalloc((void**)&dl, b5);
    if (e == hipSuccess) e = hipMalloc((void**)&dr, b5);
    if (e == hipSuccess) e = hipMalloc((void**)&dm, b5);
    if (e == hipSuccess) e = hipMalloc((void**)&dp, b5);
    if (e == hipSuccess) e = hipMalloc((void**)&dk, bi);
    if (e == hipSuccess) e = hipMalloc((void**)&df, bi);
    if (e == hipSuccess) e = hipMemcpy(dl, left, b5, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dr, right, b5, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(dk, kind.data(), bi, hipMemcpyHostToDevice);
    if (e == hipSuccess) e = hipMemcpy(df, fixed, bi, hipMemcpyHostToDevice);
    if (e == hipSuccess)
        e = pairs ? tsu::launch_kat_edge_pairs(P, n / 2, dl, dr, dk, df, dm, dp, nullptr)
                  : tsu::launch_kat_edge(P, n, dl, dr, dk, df, dm, dp, nullptr);
    if (e == hipSuccess) e = hipMemcpy(Dm, dm, b5, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(Dp, dp, b5, hipMemcpyDeviceToHost);
    (void)hipFree(dl);
    (void)hipFree(dr);
    (void)hipFree(dm);
    (void)hipFree(dp);
    (void)hipFree(dk);
    (void)hipFree(df);
    if (e != hipSuccess) return fail(TSU_ERR_HIP, std::string("kat edge: ") + hipGetErrorString(e));
    return TSU_OK;
}

}  // namespace

TSU_API int tsu_kat_edge_flux(const tsu_sim_params* p, const tsu_scheme* s, int n, const double* left,
                              const double* right, const int* normal, const int* fixed, double* Dm, double* Dp,
                              int device)
{
    return kat_edges(p, s, n, left, right, normal, fixed, Dm, Dp, device, false);
}

TSU_API int tsu_kat_edge_flux_pairs(const tsu_sim_params* p, const tsu_scheme* s, int n, const double* left,
                                    const double* right, const int* normal, const int* fixed, double* Dm,
                                    double* Dp, int device)
{
    return kat_edges(p, s, n, left, right, normal, fixed, Dm, Dp, device, true);
}

TSU_API int tsu_kat_point(const tsu_sim_params* p, const tsu_scheme* s, int what, int n, const double* a,
                          const double* b, const double* c, const double* d, double* o1, double* o2, double* o3,
                          double* o4, int device)
{
    if (!p || !s || n < 0 || what < 0 || what > 7) return fail(TSU_ERR_ARG, "bad argument");
    if (n == 0) return TSU_OK;
    DevParams P;
    tsu::make_dev_params(p, s, &P);
    DeviceGuard g(device);
    const size_t bytes = (size_t)n * sizeof(double);
    const double* in[4] = {a, b, c, d};
    double* outs[4] = {o1, o2, o3, o4};
    double* din[4] = {nullptr, nullptr, nullptr, nullptr};
    double* dout[4] = {nullptr, nullptr, nullptr, nullptr};
    hipError_t e = hipSuccess;
    for (int i = 0; i < 4 && e == hipSuccess; i++) {
        e = hipMalloc((void**)&din[i], bytes);
        if (e == hipSuccess && in[i]) e = hipMemcpy(din[i], in[i], bytes, hipMemcpyHostToDevice);
        if (e == hipSuccess && !in[i]) e = hipMemset(din[i], 0, bytes);
        if (e == hipSuccess) e = hipMalloc((void**)&dout[i], bytes);
    }
    if (e == hipSuccess)
        e = tsu::launch_kat_point(what, s->limiter, n, din[0], din[1], din[2], din[3], dout[0], dout[1], dout[2],
                                  dout[3], P, nullptr);
    for (int i = 0; i < 4 && e == hipSuccess; i++)
        if (outs[i]) e = hipMemcpy(outs[i], dout[i], bytes, hipMemcpyDeviceToHost);
    for (int i = 0; i < 4; i++) {
        (void)hipFree(din[i]);
        (void)hipFree(dout[i]);
    }
    if (e != hipSuccess) return fail(TSU_ERR_HIP, std::string("kat point: ") + hipGetErrorString(e));
    return TSU_OK;
}

}  // extern "C"
