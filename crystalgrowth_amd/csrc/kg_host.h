// kg_host.h -- host-side helpers shared by the C ABI sources: error state,
// HIP status checks, and the StepArgs a kernel launch needs.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <string>
#include <utility>
#include <vector>

#include "../../include/kobayashi_gpu.h"
#include "kg_internal.h"

namespace kg {
struct AdjointWork;
void free_adjoint(AdjointWork *w);

// Copies pieces of device memory to host memory, after what is on the stream,
// and waits for them (kg_copy.hip).
struct HostPiece {
    void *host;
    const void *dev;
    size_t bytes;
};
hipError_t copy_to_host(hipStream_t s, const HostPiece *pieces, int count);
inline hipError_t copy_to_host(hipStream_t s, void *host, const void *dev, size_t bytes)
{
    const HostPiece p{host, dev, bytes};
    return copy_to_host(s, &p, 1);
}
// Its pinned buffers live while any handle does.
void stages_retain();
void stages_release();
}  // namespace kg

// A solver handle (kg_handle): one grid's device fields and parameters.
struct kg_solver_s {
    int nx = 0, ny = 0, precision = KG_F32;
    kg_params params{};
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    void *phi[2] = {nullptr, nullptr};
    void *T[2] = {nullptr, nullptr};
    void *theta = nullptr;
    void *theta_alt = nullptr;  // other theta buffer of launches of several steps (null: none)
    void *temps = nullptr;  // 6 fields, two-pass kernel only
    double *partials = nullptr;
    kg::ReduceOut *red = nullptr;
    kg::DiskEntry *disks = nullptr;  // nuclei of a reset that are too many for partials
    size_t disks_cap = 0;
    void *image = nullptr;  // colours of the last ramp, up to IMAGE_KEEP bytes
    size_t image_cap = 0;
    int cur = 0;
    uint64_t steps = 0;
    int kernel = KG_KERNEL_FUSED;
    kg::AdjointWork *adj = nullptr;  // adjoint buffers, allocated on first use
    // tile status of the fused kernel: 2 x tiles words (one set per buffer
    // index); stat_valid false = unknown, cleared before the next fused step
    uint32_t *stat = nullptr;
    int stat_tiles = 0, tiles_x = 0, tiles_y = 0;
    bool stat_ok = false, stat_valid = false;
    // chunks the fused step works on (kg_api.hip, skip_cycle): the list in
    // use (n < 0: all), and SKIP_AGE pinned host buffers of liveness flags,
    // each with the event of the kernel that writes it, the tag that request
    // writes and whether it is still to be read
    kg::LiveList live{-1, 0, nullptr, {}};
    std::vector<uint16_t> live_order;
    int nchunks = 0;
    uint8_t *live_host[kg::SKIP_AGE] = {};
    hipEvent_t live_ev[kg::SKIP_AGE] = {};
    uint32_t live_tag[kg::SKIP_AGE] = {};
    bool live_pending[kg::SKIP_AGE] = {};
    uint32_t next_tag = 0;
    // lists longer than LIVE_MAX: two device copies used in turn, each
    // filled from a pinned staging buffer by an asynchronous copy whose
    // event guards the staging buffer's next use
    uint16_t *live_dev[2] = {};
    uint16_t *live_stage[2] = {};
    hipEvent_t live_copy_ev[2] = {};
    int live_dev_next = 0;
    uint64_t live_stale = 0;       // answers found not yet written (full launches instead)
    uint64_t listed_launches = 0;  // step launches that covered only listed chunks
    // bound on |theta| of angles not written by the step (resets write 0,
    // kg_set_fields what it is given; infinite after kg_device_fields)
    double theta_given = 0.0;

    size_t cells() const { return (size_t)nx * (size_t)ny; }
    size_t esize() const { return precision == KG_F64 ? sizeof(double) : sizeof(float); }
    size_t field_bytes() const { return cells() * esize(); }
};

// A batch handle (kg_batch): every member's fields in one allocation per field.
struct kg_batch_s {
    int count = 0, precision = KG_F32;
    std::vector<int> nx, ny;
    std::vector<kg_params> params;
    std::vector<size_t> off;   // element offset of each member in the field buffers
    size_t total = 0;          // elements per field buffer
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    void *phi[2] = {nullptr, nullptr};
    void *T[2] = {nullptr, nullptr};
    void *theta = nullptr;
    void *members = nullptr;   // StepArgs<R>[count]
    int4 *tiles = nullptr;
    int ntiles = 0;
    uint32_t *step_base = nullptr;
    double *partials = nullptr;
    kg::ReduceOut *red = nullptr;
    kg::DiskEntry *disks = nullptr;  // nuclei of a reset that are too many for partials
    size_t disks_cap = 0;
    uint64_t steps = 0;        // steps since the last reset of all members
    uint64_t base_host = 0;    // value of *step_base
    uint32_t base_tmp = 0;     // host source of step_base uploads
    int mode = KG_BATCH_LAUNCH, graph_steps = 0;
    hipGraph_t graph = nullptr;
    hipGraphExec_t exec = nullptr;
    kg::AdjointWork *adj = nullptr;  // batched adjoint buffers, allocated on first use
    // tile status of the step kernel: two sets (buffer 0, buffer 1) of one
    // word per tile of every member; stat_valid false = unknown
    uint32_t *stat = nullptr;
    int stat_tiles = 0;
    bool stat_valid = false;
    std::vector<double> theta_given;  // per member, as kg_solver_s::theta_given
    // launches of several steps (shape 0: none; kg_step.hip, k_batch_multi):
    // tile table, member offsets, and the other theta buffer (launch mode); the
    // member tables without tile status for the steps they leave over, and
    // whether these hold the members' current parameters
    int multi_shape = 0, nmulti = 0;
    int4 *multi_tiles = nullptr;
    size_t *multi_off = nullptr;
    void *theta_alt = nullptr;
    void *members_plain = nullptr;
    std::vector<char> plain_host;  // source of its uploads
    bool plain_valid = false;
    // chunk lists (launch mode, batches of at least SKIP_MIN_CHUNKS chunks;
    // kg_batch.hip, batch_skip_cycle): the chunks in the order the tile
    // table deals them (member, chunk column, chunk row), the pinned flags
    // of the request in flight, and the tile table of the listed chunks on
    // the device with its pinned staging copy; ntiles_listed < 0: the full
    // table
    int cw = 0, ch = 0;        // chunk shape (tiles) of the tile table and the lists
    std::vector<int4> chunk_list;
    int4 *chunks_dev = nullptr;
    int nchunks = 0;
    uint8_t *live_flags = nullptr;
    hipEvent_t live_ev = nullptr;
    bool live_pending = false;
    uint32_t live_tag = 0, next_tag = 0;
    int4 *tiles_listed = nullptr, *tiles_stage = nullptr;
    size_t listed_cap = 0;
    int ntiles_listed = -1;
    bool listed_all = false;   // the list holds every chunk (for its order and busy chunks)
    // the same lists kept on the device in KG_BATCH_GRAPH mode (kg_step.hip,
    // k_batch_compact): two flag buffers, the listed length, lists made
    uint8_t *dflags2 = nullptr;
    int *dcount = nullptr;
    uint32_t *dperiods = nullptr;
    uint64_t listed_launches = 0, live_stale = 0;

    size_t esize() const { return precision == KG_F64 ? sizeof(double) : sizeof(float); }
    size_t cells(int m) const { return (size_t)nx[m] * (size_t)ny[m]; }
    int cur() const { return (int)(steps & 1u); }
    char *field(void *base, int m) const { return static_cast<char *>(base) + off[m] * esize(); }
};

namespace kg {

int fail(int code, const std::string &msg);
int hip_fail(hipError_t e, const char *what);

#define KG_HIP(call)                               \
    do {                                           \
        hipError_t e_ = (call);                    \
        if (e_ != hipSuccess)                      \
            return ::kg::hip_fail(e_, #call);      \
    } while (0)

// Scalar parameters combined in R, in the reference's association order
// (see StepArgs); pointers and step counter filled in by the caller.
template <typename R>
StepArgs<R> make_args(const kg_params &p, int nx, int ny)
{
    StepArgs<R> a{};
    a.nx = nx;
    a.ny = ny;
    a.boundary = p.boundary;
    const R dx = (R)p.dx, dy = (R)p.dy, dt = (R)p.dt, tau = (R)p.tau;
    a.inv_dx = (R)1 / dx;
    a.inv_dy = (R)1 / dy;
    a.inv_3dx2 = (R)1 / ((R)3 * dx * dx);
    a.dt = dt;
    a.dt_tau = dt / tau;
    a.eps_bar = (R)p.eps_bar;
    a.delta = (R)p.delta;
    a.aniso = (R)p.aniso;
    a.theta0 = (R)p.theta0;
    a.neg_ebar_j_delta = -(R)p.eps_bar * (R)p.aniso * (R)p.delta;
    a.alpha_pi = (R)p.alpha / (sizeof(R) == 4 ? (R)3.14159274f : (R)3.14159265358979323846);
    a.gamma = (R)p.gamma;
    a.teq = (R)p.teq;
    a.K = (R)p.K;
    a.noise_a = (R)p.noise_a;
    a.instance = p.instance;
    a.key0 = (uint32_t)p.seed;
    a.key1 = (uint32_t)(p.seed >> 32);
    return a;
}

// StepArgs::stream_out for a launch over `cells` cells of `esize` bytes:
// whether its per-step working set -- phi and T read and written, theta --
// exceeds MI355X's 256 MiB last-level (Infinity) cache, so that its outputs
// cannot be served from cache to the next step anyway.
#ifndef KG_STREAM_OUT_BYTES
#define KG_STREAM_OUT_BYTES (256ull << 20)
#endif
inline int stream_outputs(size_t cells, size_t esize)
{
    return (unsigned long long)cells * esize * 5ull > (unsigned long long)KG_STREAM_OUT_BYTES ? 1 : 0;
}

// |theta| the step itself writes stays below 2 pi + pi/2 < 8.
constexpr double STEP_THETA_BOUND = 8.0;

// StepArgs::wide_angles for parameters p and a bound on the stored |theta|:
// whether |aniso (theta - theta0)| may leave the reduced sin/cos range (with
// a margin for float rounding; NaN or infinite bounds count as wide).
inline int wide_angles(const kg_params &p, double theta_given)
{
    const double b = theta_given > STEP_THETA_BOUND ? theta_given : STEP_THETA_BOUND;
    const double m = std::fabs(p.aniso) * (b + std::fabs(p.theta0));
    return m <= 0.99e4 ? 0 : 1;
}

// Largest |v| of n values of the given precision (NaN -> infinity), which are at
// `host` and, once the stream's copies have run, at `dev`; waits for the stream.
// Few values are scanned on the host, 1.3 ns each (5.3 ms for 2048 x 2048): k_max_abs
// and the copy of its partial maxima, through the reduction scratch `partials`,
// take 14 us at least (and 25 us for 2048 x 2048 FP32 values).  kg_set_fields, us,
// host / device: 96^2 cells FP32 33 / 46, FP64 34 / 48; 128^2 39 / 48, 42 / 53; 250^2
// 109 / 62, 122 / 79.
constexpr size_t HOST_SCAN = 24576;
inline int max_abs(const void *host, const void *dev, size_t n, int precision, double *partials,
                   hipStream_t s, double *out)
{
    double m = 0.0;
    if (n <= HOST_SCAN) {
        for (size_t i = 0; i < n; ++i) {
            const double x = precision == KG_F64 ? static_cast<const double *>(host)[i]
                                                 : (double)static_cast<const float *>(host)[i];
            const double a = std::fabs(x);
            if (!(a <= m))
                m = a == a ? a : HUGE_VAL;
        }
        KG_HIP(hipStreamSynchronize(s));
        *out = m;
        return KG_OK;
    }
    double part[MAX_ABS_BLOCKS];
    KG_HIP(precision == KG_F64
               ? launch_max_abs<double>(static_cast<const double *>(dev), n, partials, s)
               : launch_max_abs<float>(static_cast<const float *>(dev), n, partials, s));
    KG_HIP(copy_to_host(s, part, partials, sizeof(part)));
    for (double x : part)
        m = x > m ? x : m;
    *out = m;
    return KG_OK;
}

// n elements of each field 0 but for phi = 1 on the disks.  A few disks of the
// grid at phi travel with the launch; a list goes to the device in the reduction
// scratch, or, if it is longer, in the buffer `dev` of `cap` entries, grown as
// needed up to DISK_CHUNK (longer lists go in turns).
constexpr size_t DISK_CHUNK = 65536;
template <typename R>
int reset_fields(R *phi, R *T, R *theta, size_t n, const std::vector<DiskEntry> &disks, double r2,
                 double *scratch, DiskEntry *&dev, size_t &cap, hipStream_t s)
{
    FewDisks few{};
    bool all = disks.size() <= (size_t)FewDisks::MAX;
    for (const DiskEntry &d : disks) {
        all = all && d.off == 0;
        if (!all)
            break;
        few.cx[few.n] = d.cx;
        few.cy[few.n++] = d.cy;
    }
    if (!all)
        few.n = 0;
    const int nx = disks.empty() ? 0 : disks[0].nx, ny = disks.empty() ? 0 : disks[0].ny;
    KG_HIP(launch_reset<R>(phi, T, theta, n, nx, ny, few, r2, s));
    if (all)
        return KG_OK;
    const size_t want = disks.size() < DISK_CHUNK ? disks.size() : DISK_CHUNK;
    const bool fits = want * sizeof(DiskEntry) <= reduce_partials_size() * sizeof(double);
    if (!fits && want > cap) {
        if (dev)
            KG_HIP(hipFree(dev));
        dev = nullptr;
        cap = 0;
        KG_HIP(hipMalloc(&dev, want * sizeof(DiskEntry)));
        cap = want;
    }
    DiskEntry *list = fits ? reinterpret_cast<DiskEntry *>(scratch) : dev;
    for (size_t at = 0; at < disks.size(); at += want) {
        const size_t m = disks.size() - at < want ? disks.size() - at : want;
        KG_HIP(hipMemcpyAsync(list, disks.data() + at, m * sizeof(DiskEntry), hipMemcpyHostToDevice,
                              s));
        KG_HIP(launch_disks<R>(phi, list, (int)m, r2, s));
    }
    return KG_OK;
}

// MULTI_STEPS steps of a handle that has theta_alt, in one launch; a: its
// arguments for a single step.
template <typename R>
hipError_t step_multi(kg_solver_s &h, StepArgs<R> a)
{
    a.step = (uint32_t)h.steps;
    a.theta_in = static_cast<const R *>(h.theta);
    a.theta = static_cast<R *>(h.theta_alt);
    const hipError_t e = launch_step_multi<R>(a, 0, h.stream);
    if (e == hipSuccess) {
        std::swap(h.theta, h.theta_alt);
        h.cur ^= 1;
        h.steps += MULTI_STEPS;
    }
    return e;
}

// MULTI_STEPS steps of every member of a batch that has multi_shape, from step
// count `step`; stride as in launch_step_multi.
template <typename R>
hipError_t batch_multi(const kg_batch_s &b, const MultiIO<R> &io, uint32_t step, size_t stride)
{
    return launch_batch_multi<R>(b.multi_shape, static_cast<const StepArgs<R> *>(b.members),
                                 b.multi_off, b.multi_tiles, b.nmulti, io, step, stride, b.stream);
}

// Centres of `count` Philox-drawn nuclei (kg_reset_seeds).
void seed_centres(int nx, int ny, int count, int margin, uint64_t seed, int *cxy);

}  // namespace kg
